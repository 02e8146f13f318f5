// C8 and C4 products: 64x64 tiles of complex elements, with two k-groups per
// workgroup (tile choice 1) or one (0).
#define XT_GEMM_KERNELS
#include "gemm_native.hpp"

namespace xt {

int launch_native_cx(const Product &q, int kind, int tile, hipStream_t s)
{
  if (kind == C8) {
    if (tile == 1) return launch_modes<double, true, 64, 64, 16, 2, 2>(q, s);
    return launch_modes<double, true, 64, 64, 16, 1, 2>(q, s);
  }
  if (tile == 1) return launch_modes<float, true, 64, 64, 16, 2, 2>(q, s);
  return launch_modes<float, true, 64, 64, 16, 1, 2>(q, s);
}

}  // namespace xt
