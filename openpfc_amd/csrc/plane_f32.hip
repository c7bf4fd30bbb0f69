// Plane kernels (x and y passes of a whole plane per block), single precision.
//
// A boundary pass (PL_BND) has to give the bits of PL_INV followed by PL_FWD, so
// products and sums are fused where the source writes them in one expression
// and nowhere else; with the compiler's default it chooses per kernel which
// product of a sum to fuse, and the same line transform rounds differently in
// two kernels.
#pragma clang fp contract(on)

#include "plane_kernels.hpp"

namespace pfc_amd {
PFC_AMD_DEFINE_PLANE(float)
} // namespace pfc_amd
