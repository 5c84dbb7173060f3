// The driver's kernels for three bf16 terms.
#include "gemm_launch.hpp"

namespace wmmae_driver {
const PolicyKernels &kernels_bf16x3_ec() {
  static constexpr PolicyKernels k =
      make_policy_kernels<w::precision::tf32, __bf16, 3, true>();
  return k;
}
} // namespace wmmae_driver
