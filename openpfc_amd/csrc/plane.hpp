// plane.hpp -- host interface of the plane kernels (plane_kernels.hpp): which
// extents they take, their line plans and their launch.
#pragma once

#include "fft_kernels.hpp"

namespace pfc_amd {

// PL_FWD  fields blockIdx.y = 0: psi, 1: N(psi), 2: lam -> dst[blockIdx.y]
// PL_INV  src -> psi_out * scale
// PL_BND  src -> psi in registers -> blockIdx.y = 0: psi, 1: N(psi) -> dst
// PL_TUNG src (mean field) -> N(psi_in, mean field) -> dst[0]; optional mf_out
// PL_ADJ  src, src2 -> a, b in real space; psi_out = a + 3 (m + psi_in)^2 b (double)
enum PlaneMode { PL_FWD = 0, PL_INV = 1, PL_BND = 2, PL_TUNG = 3, PL_ADJ = 4 };

template <typename T> struct PlaneArgs {
  Nonlin<T> nl;
  TungNl<T> tnl;
  const T *mnl; // batched plans: per-field (3m, 3m^2) pairs, or null
  const T *psi_in;
  const T *lam_in;
  T *psi_out;
  T *mf_out;
  const cplx<T> *src, *src2;
  cplx<T> *dst[3];
  const cplx<T> *tw_x; // nx/2-point line twiddles
  const cplx<T> *tw_y; // ny-point line twiddles
  const cplx<double> *wn; // exp(-2 pi i k/nx), k = 0..nx/2, in double
  int nx, ny, nz; // nz: planes per field
  int pitch;      // row pitch of the spectra in memory (complex elements)
  int nfields;    // PL_FWD, PL_BND: fields made (grid y)
  T scale;        // PL_INV
  T mean;         // PL_ADJ
};

// Line plans per length: columns (ny) and rows (nx/2).  Lines of 64 points and
// more run 8 threads at least where the registers allow it, so that a wave
// holds at most 8 lines and each strided access moves 8 neighbouring values.
// Single precision keeps the radices of the row and column kernels' defaults,
// the fewest passes (and roundings) a length takes: a second pass for 12 points
// put a 1024x12x96 run 1.27 times as far from the 64-bit result.  It has the
// registers for them (rows of 128 as 16x8: 13.5 us at 256x64x64 against 17.4 as
// 8x4x4), while 16 doubles with the operands of the C2R merge spill at the 128
// registers that a block of 16 waves leaves.
template <typename T, int N> struct PlanePlan;
template <> struct PlanePlan<double, 8> { using P = FftPlan<8, 4, RadixList<4, 2>>; };
template <> struct PlanePlan<float, 8> { using P = FftPlan<8, 8, RadixList<8>>; };
template <> struct PlanePlan<double, 12> { using P = FftPlan<12, 6, RadixList<6, 2>>; };
template <> struct PlanePlan<float, 12> { using P = FftPlan<12, 12, RadixList<12>>; };
template <> struct PlanePlan<double, 16> { using P = FftPlan<16, 4, RadixList<4, 4>>; };
template <> struct PlanePlan<float, 16> { using P = FftPlan<16, 16, RadixList<16>>; };
template <typename T> struct PlanePlan<T, 24> { using P = FftPlan<24, 12, RadixList<12, 2>>; };
template <typename T> struct PlanePlan<T, 32> { using P = FftPlan<32, 8, RadixList<8, 4>>; };
template <typename T> struct PlanePlan<T, 48> { using P = FftPlan<48, 12, RadixList<12, 4>>; };
template <typename T> struct PlanePlan<T, 64> { using P = FftPlan<64, 8, RadixList<8, 8>>; };
template <> struct PlanePlan<double, 96> { using P = FftPlan<96, 12, RadixList<4, 4, 6>>; };
template <> struct PlanePlan<float, 96> { using P = FftPlan<96, 24, RadixList<12, 8>>; };
template <typename T> struct PlanePlan<T, 128> { using P = FftPlan<128, 16, RadixList<16, 8>>; };
template <typename T> struct PlanePlan<T, 192> {
  using P = FftPlan<192, 12, RadixList<12, 4, 4>>;
};
template <typename T> struct PlanePlan<T, 256> { using P = FftPlan<256, 16, RadixList<16, 16>>; };
template <typename T> struct PlanePlan<T, 512> { using P = FftPlan<512, 8, RadixList<8, 8, 8>>; };
template <typename T, int N> struct PlaneRowPlan { using P = typename PlanePlan<T, N>::P; };
template <> struct PlaneRowPlan<double, 256> {
  using P = FftPlan<256, 8, RadixList<8, 8, 4>>;
};
template <> struct PlaneRowPlan<double, 128> { using P = FftPlan<128, 8, RadixList<8, 4, 4>>; };

// Calls f(Plan{}) for the column (ROW = false) or row plan of length n; false
// when there is none.
template <typename T, bool ROW, int N, typename F>
__host__ __device__ __forceinline__ void plane_call(F &&f) {
  if constexpr (ROW)
    f(typename PlaneRowPlan<T, N>::P{});
  else
    f(typename PlanePlan<T, N>::P{});
}
template <typename T, bool ROW, typename F>
__host__ __device__ __forceinline__ bool plane_plan(int n, F &&f) {
  switch (n) {
  case 8: plane_call<T, ROW, 8>(f); return true;
  case 12: plane_call<T, ROW, 12>(f); return true;
  case 16: plane_call<T, ROW, 16>(f); return true;
  case 24: plane_call<T, ROW, 24>(f); return true;
  case 32: plane_call<T, ROW, 32>(f); return true;
  case 48: plane_call<T, ROW, 48>(f); return true;
  case 64: plane_call<T, ROW, 64>(f); return true;
  case 96: plane_call<T, ROW, 96>(f); return true;
  case 128: plane_call<T, ROW, 128>(f); return true;
  case 192: plane_call<T, ROW, 192>(f); return true;
  case 256: plane_call<T, ROW, 256>(f); return true;
  case 512: plane_call<T, ROW, 512>(f); return true;
  default: return false;
  }
}

// ---- host side ------------------------------------------------------------------
constexpr size_t kPlaneLds = 160 * 1024; // LDS of a CU

template <typename T, bool ROW> int plane_lines_per_wave(int n) {
  int lpw = 0;
  plane_plan<T, ROW>(n, [&](auto p) { lpw = 64 / decltype(p)::TL; });
  return lpw;
}
template <typename T, bool ROW> std::vector<int> plane_radices(int n) {
  std::vector<int> r;
  plane_plan<T, ROW>(n, [&](auto p) { r = RadixOf<typename decltype(p)::List>::get(); });
  return r;
}
// Bytes of the plane's LDS image, 0 when the plane kernels do not take it.
template <typename T> size_t plane_lds(int nx, int ny) {
  if (nx % 2 || !plane_lines_per_wave<T, true>(nx / 2) || !plane_lines_per_wave<T, false>(ny))
    return 0;
  const size_t b = (size_t)(nx / 2 + 1) * ny * 2 * sizeof(T);
  return b <= kPlaneLds ? b : 0;
}
// Waves per block: enough that the axis with more line groups takes the
// fewest rounds a block of 16 waves can take.
template <typename T> int plane_waves(int nx, int ny) {
  const int ly = plane_lines_per_wave<T, false>(ny), lx = plane_lines_per_wave<T, true>(nx / 2);
  const int gy = (nx / 2 + 1 + ly - 1) / ly, gx = (ny + lx - 1) / lx;
  const int g = gy > gx ? gy : gx, rounds = (g + 15) / 16;
  return (g + rounds - 1) / rounds;
}

// Launches MODE over `planes` planes (all fields of a batched plan).
template <typename T> hipError_t plane_launch(int mode, PlaneArgs<T> a, long planes, hipStream_t s);
template <> hipError_t plane_launch<double>(int, PlaneArgs<double>, long, hipStream_t);
template <> hipError_t plane_launch<float>(int, PlaneArgs<float>, long, hipStream_t);

// Admits the LDS size of every plane kernel on the current device.
template <typename T> hipError_t plane_init();
template <> hipError_t plane_init<double>();
template <> hipError_t plane_init<float>();

} // namespace pfc_amd
