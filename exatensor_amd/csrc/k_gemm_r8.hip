// R8 (FP64) products: tile choices 0 (128x128), 1 (64x64, four k-groups per
// workgroup) and 2 (64x64).
#define XT_GEMM_KERNELS
#include "gemm_native.hpp"

namespace xt {

int launch_native_r8(const Product &q, int tile, hipStream_t s)
{
  if (tile == 2) return launch_modes<double, false, 64, 64, 16, 1, 4>(q, s);
  if (tile == 1) return launch_modes<double, false, 64, 64, 16, 4, 4>(q, s);
  return launch_modes<double, false, 128, 128, 16, 1, 2>(q, s);
}

}  // namespace xt
