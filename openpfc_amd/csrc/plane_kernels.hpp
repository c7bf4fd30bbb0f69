// plane_kernels.hpp -- x and y passes of a whole (x, y) plane in one block.
//
// Where the half spectrum of one z plane ((nx/2+1) x ny complex values) fits
// the 160 KB of LDS of a CU, one block transforms the plane along both axes
// without a trip to memory in between: psi plane -> half spectrum (PL_FWD),
// half spectrum -> psi plane (PL_INV), or, between two z passes, inverse y,
// inverse x, the pointwise work in real space, forward x and forward y in one
// go (PL_BND for the PFC step boundary, PL_TUNG for the Tungsten nonlinearity,
// PL_ADJ for the adjoint's combine).  A PFC step then moves 2C + C (z pass) and
// C + 2C (boundary) instead of 2R + 12C, and a step of a multi-step run is two
// launches instead of five.
//
// What bounds these grids is latency, not bandwidth: their spectra stay in
// the last-level cache and a launch of the line passes takes 3.3 us at 32^3
// whatever it moves.  Every line transform here lies within one wavefront
// (TL threads of a line, 64/TL lines side by side), so its exchanges need
// wavefront ordering only and run in the line's own storage: the plane's LDS
// image is both the transpose buffer and the exchange buffer, and a block
// barrier stands only between the two axes.
//
// LDS image: element (kx, y) at y*pitch + kx, complex values interleaved, pitch
// = nx/2 + 1 (odd for even nx/2).  The lanes of a wave run over lines first:
// 8 (16-byte values) or 16 (8-byte values) consecutive lanes then touch
// columns kx, kx+1, ... of one row or, an odd pitch apart, rows y, y+1, ... of
// one column: distinct banks either way.
//
// Measured times stand at plane_variant_default() (pfc_hip.hip).
#pragma once

#include "plane.hpp"

namespace pfc_amd {

// Lines of a wave's group: lane -> (line, t).  Lanes past the last line work
// on a copy of it (the same values to the same slots) and store nothing.
template <typename Plan> struct PlaneLane {
  static constexpr int LPW = 64 / Plan::TL; // lines per wave
  int line, t;
  bool active;
  __device__ __forceinline__ PlaneLane(int g, int lane, int nlines) {
    const int l = g * LPW + lane % LPW;
    active = l < nlines;
    line = active ? l : nlines - 1;
    t = lane / LPW;
    // t is the same in every group: hide that, or the compiler keeps all
    // twiddles of the line in registers across the loop over groups
    asm volatile("" : "+v"(t));
  }
  __device__ __forceinline__ static int groups(int nlines) { return (nlines + LPW - 1) / LPW; }
};

// Keeps the operands of at most four elements in flight beside a line's own 12
// to 24 values: with all of them the 128 registers that a block of 16 waves
// leaves spill (PL_INV in double: 144 bytes of scratch a lane without the
// batches, 44 with; none in single).
template <typename T, int E> __device__ __forceinline__ void plane_batch(int e) {
  if (E > 8 && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
}

// Half-length merge and split with the factors exp(2 pi i k/nx) in double,
// also on single-precision values, rounded once: a factor rounded to single
// precision is off by the same amount in every step, and such errors grow
// along the unstable modes (FP32-mixed runs of 192x96x48 and of the uneven
// ensemble are then closer to the 64-bit result than with the packed
// nx-point transform of the row kernels, not further off).
template <typename T>
__device__ __forceinline__ cplx<T> plane_merge(cplx<T> xa, cplx<T> xmk, cplx<double> w, bool k0) {
  const cplx<double> r = c2r_merge(cplx<double>{xa.x, xa.y}, cplx<double>{xmk.x, xmk.y}, w, k0);
  return cplx<T>{(T)r.x, (T)r.y};
}
template <typename T>
__device__ __forceinline__ cplx<T> plane_split(cplx<T> zk, cplx<T> zmk, cplx<double> w) {
  const cplx<double> r = r2c_split(cplx<double>{zk.x, zk.y}, cplx<double>{zmk.x, zmk.y}, w);
  return cplx<T>{(T)r.x, (T)r.y};
}

// Column kx of the plane: memory -> inverse y -> LDS.
template <typename T, typename Plan>
__device__ __forceinline__ void plane_y_inv(const cplx<T> *__restrict__ src, int pitch_m,
                                            typename Vec2<T>::type *lds, int pitch, int W,
                                            const cplx<T> *__restrict__ tw) {
  constexpr int TL = Plan::TL, E = Plan::E;
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64, nw = blockDim.x / 64;
  for (int g = wid; g < PlaneLane<Plan>::groups(W); g += nw) {
    const PlaneLane<Plan> p(g, lane, W);
    cplx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = src[(long)(p.t + TL * e) * pitch_m + p.line];
    const LdsCplx<T> ll{lds, p.line, pitch};
    LineFft<T, Plan, +1, false, false, true>::run(v, p.t, ll, tw);
#pragma unroll
    for (int e = 0; e < E; ++e) ll.put(p.t + TL * e, v[e]);
  }
}

// LDS -> forward y -> memory.
template <typename T, typename Plan>
__device__ __forceinline__ void plane_y_fwd(cplx<T> *__restrict__ dst, int pitch_m,
                                            typename Vec2<T>::type *lds, int pitch, int W,
                                            const cplx<T> *__restrict__ tw) {
  constexpr int TL = Plan::TL, E = Plan::E;
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64, nw = blockDim.x / 64;
  for (int g = wid; g < PlaneLane<Plan>::groups(W); g += nw) {
    const PlaneLane<Plan> p(g, lane, W);
    const LdsCplx<T> ll{lds, p.line, pitch};
    cplx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ll.get(p.t + TL * e);
    lds_sync<true>(); // the column becomes its own exchange area
    LineFft<T, Plan, -1, false, false, true>::run(v, p.t, ll, tw);
    if (p.active) {
#pragma unroll
      for (int e = 0; e < E; ++e) dst[(long)(p.t + TL * e) * pitch_m + p.line] = v[e];
    }
  }
}

// Rows of the plane with the nx/2-point plan: C2R of the LDS image (every mode
// but PL_FWD), the pointwise work, R2C back into the LDS image (PL_FWD, PL_BND,
// PL_TUNG).  row0: index of the plane's first real row; `second`: PL_ADJ's
// second field.
template <typename T, typename Plan, int MODE>
__device__ __forceinline__ void plane_x(const PlaneArgs<T> &a, const Nonlin<T> &nl, int field,
                                        typename Vec2<T>::type *lds, int pitch, long row0,
                                        bool second) {
  constexpr int TL = Plan::TL, E = Plan::E, M = Plan::N;
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64, nw = blockDim.x / 64;
  for (int g = wid; g < PlaneLane<Plan>::groups(a.ny); g += nw) {
    const PlaneLane<Plan> p(g, lane, a.ny);
    const LdsCplx<T> row{lds, p.line * pitch, 1};
    const long ro = (row0 + p.line) * (2L * M);
    cplx<T> v[E];
    if constexpr (MODE == PL_FWD) {
      const cplx<T> *__restrict__ in =
          reinterpret_cast<const cplx<T> *>((field == 2 ? a.lam_in : a.psi_in) + ro);
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = in[p.t + TL * e];
      } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = p.t + TL * e;
        v[e] = plane_merge(row.get(k), row.get(M - k), a.wn[k], k == 0);
        plane_batch<T, E>(e);
      }
      lds_sync<true>(); // the row becomes its own exchange area
      LineFft<T, Plan, +1, false, false, true>::run(v, p.t, row, a.tw_x);
    }
    // v[e] = (u[2k], u[2k+1]), k = t + TL*e
    if constexpr (MODE == PL_INV) {
      if (p.active) {
        cplx<T> *__restrict__ out = reinterpret_cast<cplx<T> *>(a.psi_out + ro);
#pragma unroll
        for (int e = 0; e < E; ++e) out[p.t + TL * e] = c_scale(v[e], a.scale);
      }
    } else if constexpr (MODE == PL_ADJ) {
      if (p.active) {
        cplx<T> *out = reinterpret_cast<cplx<T> *>(a.psi_out + ro);
        if (!second) { // parked in the result; the same thread combines it below
#pragma unroll
          for (int e = 0; e < E; ++e) out[p.t + TL * e] = v[e];
        } else {
          const cplx<T> *__restrict__ ps = reinterpret_cast<const cplx<T> *>(a.psi_in + ro);
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const cplx<T> w = ps[p.t + TL * e], f = out[p.t + TL * e];
            const T ux = a.mean + w.x, uy = a.mean + w.y;
            out[p.t + TL * e] = cplx<T>{f.x + (((T)3 * (ux * ux)) * v[e].x),
                                        f.y + (((T)3 * (uy * uy)) * v[e].y)};
            plane_batch<T, E>(e);
          }
        }
      }
    } else {
      if constexpr (MODE == PL_TUNG) {
        if (a.mf_out && p.active) {
          cplx<T> *__restrict__ mo = reinterpret_cast<cplx<T> *>(a.mf_out + ro);
#pragma unroll
          for (int e = 0; e < E; ++e) mo[p.t + TL * e] = v[e];
        }
        const cplx<T> *__restrict__ ps = reinterpret_cast<const cplx<T> *>(a.psi_in + ro);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const cplx<T> u = ps[p.t + TL * e];
          v[e] = cplx<T>{a.tnl(u.x, v[e].x), a.tnl(u.y, v[e].y)};
          plane_batch<T, E>(e);
        }
      } else {
        if (field == 1) {
#pragma unroll
          for (int e = 0; e < E; ++e) v[e] = cplx<T>{nl(v[e].x), nl(v[e].y)};
        }
      }
      LineFft<T, Plan, -1, false, false, true>::run(v, p.t, row, a.tw_x);
      // R2C split: the mirror element through the row's storage
#pragma unroll
      for (int e = 0; e < E; ++e) row.put(p.t + TL * e, v[e]);
      lds_sync<true>();
      const cplx<T> xm{v[0].x - v[0].y, (T)0}; // X[M], on t == 0
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = p.t + TL * e;
        v[e] = plane_split(v[e], row.get(k == 0 ? 0 : M - k), a.wn[k]);
        plane_batch<T, E>(e);
      }
      lds_sync<true>();
#pragma unroll
      for (int e = 0; e < E; ++e) row.put(p.t + TL * e, v[e]);
      if (p.t == 0) row.put(M, xm);
    }
  }
}

// NT: threads a block may have.  Planes of up to 8 waves run the 512-thread
// build, whose 256 registers hold every double path without spilling.
template <typename T, int MODE, int NT>
__global__ void __launch_bounds__(NT) k_plane(PlaneArgs<T> a) {
  extern __shared__ __align__(16) unsigned char plane_smem[];
  auto *lds = reinterpret_cast<typename Vec2<T>::type *>(plane_smem);
  const int W = a.nx / 2 + 1, pitch = W;
  const long pz = blockIdx.x;
  const long row0 = pz * a.ny;
  const int field = blockIdx.y;
  Nonlin<T> nl = a.nl;
  if constexpr (MODE == PL_FWD || MODE == PL_BND) {
    if (a.mnl) {
      const long b = pz / a.nz;
      nl.c1 = a.mnl[2 * b];
      nl.c2 = a.mnl[2 * b + 1];
    }
  }
  auto y_inv = [&](const cplx<T> *src) {
    plane_plan<T, false>(a.ny, [&](auto p) {
      plane_y_inv<T, decltype(p)>(src + row0 * a.pitch, a.pitch, lds, pitch, W, a.tw_y);
    });
    __syncthreads();
  };
  auto x_pass = [&](bool second) {
    plane_plan<T, true>(a.nx / 2, [&](auto p) {
      plane_x<T, decltype(p), MODE>(a, nl, field, lds, pitch, row0, second);
    });
  };
  if constexpr (MODE != PL_FWD) y_inv(a.src);
  x_pass(false);
  if constexpr (MODE == PL_ADJ) {
    __syncthreads();
    y_inv(a.src2);
    x_pass(true);
  }
  if constexpr (MODE == PL_FWD || MODE == PL_BND || MODE == PL_TUNG) {
    __syncthreads();
    plane_plan<T, false>(a.ny, [&](auto p) {
      plane_y_fwd<T, decltype(p)>(a.dst[field] + row0 * a.pitch, a.pitch, lds, pitch, W, a.tw_y);
    });
  }
}

template <typename T, int MODE> hipError_t plane_init_mode() {
  const void *fn[2] = {reinterpret_cast<const void *>(&k_plane<T, MODE, 512>),
                       reinterpret_cast<const void *>(&k_plane<T, MODE, 1024>)};
  for (const void *f : fn)
    if (hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kPlaneLds);
        e != hipSuccess)
      return e;
  return hipSuccess;
}

template <typename T, int MODE>
hipError_t plane_launch_mode(const PlaneArgs<T> &a, long planes, hipStream_t s) {
  const size_t lds = plane_lds<T>(a.nx, a.ny);
  if (!lds || planes < 1 || planes > 0x7fffffffL) return hipErrorInvalidValue;
  const int nf = (MODE == PL_FWD || MODE == PL_BND) ? a.nfields : 1;
  int nt = 64 * plane_waves<T>(a.nx, a.ny);
  // A CU runs one block of 9 to 16 waves at a time (128 registers a thread), and its
  // loads, transforms and stores follow each other.  With more blocks than the
  // 256 CUs, and room in the LDS for two, 8 waves a block let two blocks overlap.
  // Single precision, us of a step of a run with 16 | 8 waves: 128x128x256
  // 52.9 | 46.3, 128x128x512 105 | 89, 96x192x512 121 | 103, 256x64x512 96 | 84,
  // 192x96x512 102 | 98.  At 256 blocks and below both take the same time or
  // 8 waves lose (128x128x64: 25.5 | 26.4), as they do in the inverse pass alone
  // (25.5 | 26.2 at 128x128x512); doubles differ by 1 % either way.
  if constexpr (sizeof(T) == 4 && (MODE == PL_FWD || MODE == PL_BND)) {
    if (nt > 512 && planes * nf > 256 && 2 * lds <= 160 * 1024) nt = 512;
  }
  const dim3 grid((unsigned)planes, (unsigned)nf);
  if (nt <= 512)
    hipLaunchKernelGGL((k_plane<T, MODE, 512>), grid, dim3(nt), lds, s, a);
  else
    hipLaunchKernelGGL((k_plane<T, MODE, 1024>), grid, dim3(nt), lds, s, a);
  return hipGetLastError();
}

#define PFC_AMD_DEFINE_PLANE(T)                                                             \
  template <> hipError_t plane_launch<T>(int mode, PlaneArgs<T> a, long planes, hipStream_t s) { \
    switch (mode) {                                                                         \
    case PL_FWD: return plane_launch_mode<T, PL_FWD>(a, planes, s);                         \
    case PL_INV: return plane_launch_mode<T, PL_INV>(a, planes, s);                         \
    case PL_BND: return plane_launch_mode<T, PL_BND>(a, planes, s);                         \
    case PL_TUNG: return plane_launch_mode<T, PL_TUNG>(a, planes, s);                       \
    case PL_ADJ:                                                                            \
      if constexpr (sizeof(T) == 8) return plane_launch_mode<T, PL_ADJ>(a, planes, s);      \
      [[fallthrough]];                                                                      \
    default: return hipErrorInvalidValue;                                                   \
    }                                                                                       \
  }                                                                                         \
  template <> hipError_t plane_init<T>() {                                                  \
    for (hipError_t e : {plane_init_mode<T, PL_FWD>(), plane_init_mode<T, PL_INV>(),        \
                         plane_init_mode<T, PL_BND>(), plane_init_mode<T, PL_TUNG>()})      \
      if (e != hipSuccess) return e;                                                        \
    if constexpr (sizeof(T) == 8) return plane_init_mode<T, PL_ADJ>();                      \
    return hipSuccess;                                                                      \
  }

} // namespace pfc_amd
