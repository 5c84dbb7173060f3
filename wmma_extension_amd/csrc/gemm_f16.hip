// The driver's kernels for fp16: hi + lo with error correction, and one term.
#include "gemm_launch.hpp"

namespace wmmae_driver {
const PolicyKernels &kernels_f16_ec() {
  static constexpr PolicyKernels k =
      make_policy_kernels<w::half, _Float16, 2, true>();
  return k;
}
const PolicyKernels &kernels_f16_noec() {
  static constexpr PolicyKernels k =
      make_policy_kernels<w::half, _Float16, 1, false>();
  return k;
}
} // namespace wmmae_driver
