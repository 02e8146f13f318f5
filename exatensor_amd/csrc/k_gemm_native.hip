// The native-precision products of one data kind and tile choice: the makefile
// compiles this file once for each (XT_KIND, XT_TILE). A code object of its own
// for each is what a process loads at its first product: with the three choices
// of a real kind in one, a first R8 contraction took 2.8 ms instead of 2.0.
#define XT_GEMM_KERNELS
#include "gemm_native.hpp"

namespace xt {

template <>
int launch_native<XT_KIND, XT_TILE>(const Product &q, hipStream_t s)
{
  typedef typename std::conditional<XT_KIND == R8 || XT_KIND == C8, double, float>::type Real;
  constexpr bool CPLX = XT_KIND == C8 || XT_KIND == C4;
  constexpr TileShape ts = tile_shape(XT_KIND, XT_TILE);
  // waves per SIMD that the registers have to leave room for
  constexpr int occ = CPLX || ts.bm == 128 ? 2 : 4;
  return launch_modes<Real, CPLX, ts.bm, ts.bn, ts.bk, ts.groups, occ>(q, s);
}

}  // namespace xt
