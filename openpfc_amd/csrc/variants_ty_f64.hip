// Transposed-step variant lists and kernels for double precision: the y passes.
#include "variants_impl.hpp"

namespace pfc_amd {
PFC_AMD_DEFINE_T_Y_LISTS(double)
} // namespace pfc_amd
