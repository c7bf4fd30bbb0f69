// adjoint_z.hpp -- operator derivatives of the adjoint step and its fused z pass.
#pragma once

#include "fft_kernels.hpp"

namespace pfc_amd {

// d opL / d eps and d opN / d eps for one mode (unscaled).
__device__ __forceinline__ void pfc_op_deriv(const PfcOp &o, double kxy, double kz,
                                             double &opL, double &opN, double &dL,
                                             double &dN) {
#pragma clang fp contract(off)
  const double k2 = (kxy + (kz * kz));
  const double k2_lap = -k2;
  const double one_m = 1.0 - k2;
  const double L = (k2_lap * (o.eps + (one_m * one_m)));
  const double oL = exp((L * o.dt));
  opL = oL;
  if (fabs(L) > 1e-14) {
    opN = ((oL - 1.0) / L * k2_lap);
    // dt*opL*L - (opL - 1) = x e^x - expm1(x), x = L dt
    const double x = L * o.dt;
    const double num = (x * oL) - expm1(x);
    dN = ((k2_lap * k2_lap) * num) / (L * L);
  } else {
    opN = (o.dt * k2_lap);
    dN = 0.0;
  }
  dL = (o.dt * k2_lap) * oL;
}

// Spectral part of the adjoint step fused with its z transforms (natural layout,
// double fields): for L adjacent kx columns at one ky, from spectra transformed
// along x and y,
//   Lam <- Fz(lam), and with want_dr P <- Fz(P), N <- Fz(N),
//   partial[block] = sum w_kx Re(conj(Lam) (dopL P + dopN N)),
//   P = Fz^-1(opL Lam), N = Fz^-1(opN Lam).
// The separate z passes, the spectral kernel and the inverse z passes it
// replaces moved 15 half spectra (6 + 5 + 4); this reads 3 and writes 2.
// kz enters as kz*kz only, so up to kZTabMax points the four multipliers of a
// column come from an LDS table of nz/2 + 1 entries (see k_pfc_z); beyond that
// they are evaluated per element.  Bound by memory and by the latency of the four
// or five dependent line transforms: at 128^3 FP64 27.2 us (5 spectra of 17 MB,
// 3.1 TB/s) against 3*16.3 + 15.5 + 2*11.0 = 86.4 us of the separate passes.
struct AdjZArgs {
  const cplx<double> *lam;
  cplx<double> *P, *N;
  const cplx<double> *tw;
  PfcOp op;
  double *partial;
  long s_pos; // pitch*ny
  int pitch, W, ntx;
  int want_dr;
};

template <typename Plan, int L>
__global__ void __launch_bounds__(L *Plan::TL) k_adj_z(AdjZArgs a) {
  constexpr int TL = Plan::TL, E = Plan::E, N = Plan::N, NH = N / 2 + 1, NT = L * TL;
  constexpr int NP = row_padded(N);
  constexpr bool TAB = N <= kZTabMax;
  constexpr int XCH = 2 * L * NP > NT ? 2 * L * NP : NT;
  __shared__ double lds[XCH];
  __shared__ double tab[TAB ? 4 * L * NH : 1];
  const int c = threadIdx.x % L, t = threadIdx.x / L;
  const unsigned bid = xcd_block<double, L>(blockIdx.x, gridDim.x);
  const int x = (int)(bid % (unsigned)a.ntx) * L + c;
  const int y = (int)(bid / (unsigned)a.ntx);
  const bool active = x < a.W;
  const long base = (long)y * a.pitch + x;
  const LdsLine<double> ll{lds, c, L, L * NP};
  const double kxy = pfc_kxy(a.op, x, y);
  auto at = [&](int e) { return base + (long)(t + TL * e) * a.s_pos; };
  auto load = [&](const cplx<double> *p, cplx<double>(&v)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = active ? p[at(e)] : cplx<double>{0, 0};
  };
  double mul[TAB ? 1 : 4 * E];
  auto op = [&](int m, int e) {
    if constexpr (TAB) {
      const int k = t + TL * e;
      return tab[(m * NH + (k <= N / 2 ? k : N - k)) * L + c];
    } else {
      return mul[m * E + e];
    }
  };

  cplx<double> lam[E], v[E];
  load(a.lam, lam);
  if constexpr (TAB) {
    for (int k = t; k < NH; k += TL) {
      double oL, oN, dL, dN;
      pfc_op_deriv(a.op, kxy, pfc_kc(k, a.op.nz, a.op.fz), oL, oN, dL, dN);
      tab[(0 * NH + k) * L + c] = oL * a.op.scale;
      tab[(1 * NH + k) * L + c] = oN * a.op.scale;
      tab[(2 * NH + k) * L + c] = dL;
      tab[(3 * NH + k) * L + c] = dN;
    }
    __syncthreads(); // the table is complete
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      double oL, oN;
      pfc_op_deriv(a.op, kxy, pfc_kc(t + TL * e, a.op.nz, a.op.fz), oL, oN, mul[2 * E + e],
                   mul[3 * E + e]);
      mul[e] = oL * a.op.scale;
      mul[E + e] = oN * a.op.scale;
    }
  }
  LineFft<double, Plan, -1, false, true>::run(lam, t, ll, a.tw);
  if (a.want_dr) {
    double acc = 0.0;
#pragma unroll 1
    for (int f = 0; f < 2; ++f) {
      load(f ? a.N : a.P, v);
      LineFft<double, Plan, -1, false, true>::run(v, t, ll, a.tw);
#pragma unroll
      for (int e = 0; e < E; ++e)
        acc += (f ? op(3, e) : op(2, e)) * (lam[e].x * v[e].x + lam[e].y * v[e].y);
    }
    acc = active ? (x == 0 || 2 * x == a.op.nx ? acc : 2.0 * acc) : 0.0;
    __syncthreads(); // the exchange area is free
    lds[threadIdx.x] = acc;
    __syncthreads();
    for (int n = NT; n > 1;) { // fixed-order tree over any count
      const int h = (n + 1) / 2;
      if ((int)threadIdx.x + h < n) lds[threadIdx.x] += lds[threadIdx.x + h];
      n = h;
      __syncthreads();
    }
    if (threadIdx.x == 0) a.partial[blockIdx.x] = lds[0];
    __syncthreads(); // lds becomes the exchange area again
  }
#pragma unroll 1
  for (int f = 0; f < 2; ++f) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = c_scale(lam[e], f ? op(1, e) : op(0, e));
    LineFft<double, Plan, +1, false, true>::run(v, t, ll, a.tw);
    cplx<double> *out = f ? a.N : a.P;
    if (active) {
#pragma unroll
      for (int e = 0; e < E; ++e) out[at(e)] = v[e];
    }
  }
}

// Launch for columns of op.nz points, with the twiddles of line plan
// adj_z_plan(n).  8 columns are a whole 128-byte line of a row; at 1024 points
// they would be 1024 threads of 128 registers, which spill.
constexpr int adj_cols(int nz) { return nz >= 1024 ? 4 : 8; }
constexpr int adj_z_blocks(int W, int ny, int nz) {
  return (W + adj_cols(nz) - 1) / adj_cols(nz) * ny;
}
hipError_t adj_z_launch(AdjZArgs a, hipStream_t s);
int adj_z_plan(int n);

} // namespace pfc_amd
