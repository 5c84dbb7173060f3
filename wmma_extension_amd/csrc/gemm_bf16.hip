// The driver's kernels for bfloat16: two terms with error correction, and one
// term.
#include "gemm_launch.hpp"

namespace wmmae_driver {
const PolicyKernels &kernels_bf16x2_ec() {
  static constexpr PolicyKernels k =
      make_policy_kernels<w::bfloat16, __bf16, 2, false>();
  return k;
}
const PolicyKernels &kernels_bf16_noec() {
  static constexpr PolicyKernels k =
      make_policy_kernels<w::bfloat16, __bf16, 1, false>();
  return k;
}
} // namespace wmmae_driver
