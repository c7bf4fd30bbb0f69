// Fused z pass of the adjoint step, double precision.
#include "variants_impl.hpp"

#include "adjoint_z.hpp"

namespace pfc_amd {

// Line plan of an n-point column: the one with the fewest values a thread, since
// the kernel holds two lines (lambda and the one being transformed).
template <int N> constexpr int adj_pid() {
  return N == 96 || N == 128 || N == 256 || N == 1024 ? 1 : 0;
}
template <int I, typename P, typename... Ps> auto adj_plan_at(PlanList<P, Ps...>) {
  if constexpr (I == 0)
    return P{};
  else
    return adj_plan_at<I - 1>(PlanList<Ps...>{});
}

int adj_z_plan(int n) {
  PFC_AMD_SWITCH_LEN(n, return adj_pid<N_>();)
  return 0;
}

template <int N> hipError_t adj_z_n(AdjZArgs a, hipStream_t s) {
  using P = decltype(adj_plan_at<adj_pid<N>()>(typename Plans<N>::L{}));
  constexpr int L = adj_cols(N);
  a.ntx = (a.W + L - 1) / L;
  hipLaunchKernelGGL((k_adj_z<P, L>), dim3((unsigned)adj_z_blocks(a.W, a.op.ny, N)),
                     dim3(L * P::TL), 0, s, a);
  return hipGetLastError();
}

hipError_t adj_z_launch(AdjZArgs a, hipStream_t s) {
  PFC_AMD_SWITCH_LEN(a.op.nz, return adj_z_n<N_>(a, s);)
  return hipErrorInvalidValue;
}

} // namespace pfc_amd
