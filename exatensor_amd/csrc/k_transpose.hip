// DLF tensor permutation for gfx950 (the engine's transpose/copy kernel).
//
// Replaces the reference's gpu_tensor_block_copy_dlf__ /
// gpu_tensor_block_copy_scatter_dlf__ (TALSH/tensor_algebra_gpu_nvidia.cu:1125-1457,
// :2172-2260). Semantics: out[idx'] = in[idx], input dimension i becoming output
// dimension o2n[i]; pure data movement, bit-exact.
//
// Design:
//  * host planner: drop unit extents, fuse input dimensions that stay adjacent
//    and in order in the output, then pick an LDS tile = the union of an
//    input-minor dimension group and an output-minor dimension group, walked
//    until both contiguous runs are long enough;
//  * two forms. Tiles that divide the tensor and whose runs are whole cache
//    lines of 16-byte vectors: k_permute_tiled, streaming accesses. Everything
//    else: k_permute_runs, vectors along the runs whatever their alignment;
//  * LDS padding is chosen on the host by simulating the bank conflicts of the
//    store phase for each candidate padding period;
//  * persistent kernels (two resident 512-thread workgroups per CU): each thread decodes
//    the intra-tile offsets of its vectors once and keeps them in registers, so
//    the per-tile work is one base-offset decode per workgroup plus one
//    coalesced load and one coalesced store per vector.
// The run form against the lane-masked single-element tiles it replaces, kernel
// time: R4 37,29,41,23,31 -> 2,4,1,0,3 132 to 60 us; R8 119,70,65,34 reversed
// 113 to 69; C8 14,23,104,3,35 43 to 32; 25 instead of 34 us in the geometric
// mean of 34 random shapes. A permuted addition in one pass: rank-6 extent-24
// R8 1567 to 890 us.
#include <algorithm>
#include <mutex>
#include <string>
#include <unordered_map>
#include <cstring>
#include <numeric>

#include "kernels.hpp"

namespace xt {
namespace {

constexpr int kNT = 256;           // threads per workgroup (copy and scatter kernels)
constexpr int kTNT = 512;          // threads per workgroup of the tiled kernel
constexpr int kMaxTileDims = 8;    // dimensions inside one tile
constexpr int kMaxGridDims = 16;   // fused rank handled by the tiled path
constexpr int kMaxEPT = 8;         // tile vectors per thread (more cost occupancy)
constexpr int kTiledPerCU = 2;     // persistent workgroups per CU (16 waves)
constexpr int kTileMaxBytes = 65536;  // LDS tile (before padding)
constexpr long kTileMinVol = 8192;    // tiles are grown to at least this many elements
// Tiles of the run form: at most kRunEPT vectors per thread, counted with the
// partial last one of every run (eight hold 76 registers per thread in R4 and
// keep a workgroup's loads and stores apart for longer: R4 37x29x41x23x31 88 us
// with 64 KB tiles, 60 with these, 67 with 26 KB; 4001 x 4003 transposed 53, 33
// and 34), grown to 16 KB.
constexpr int kRunEPT = 4;
constexpr long kRunTileMaxBytes = 34 << 10, kRunTileMinBytes = 16 << 10;
constexpr int kLine = 128;            // cache line bytes

struct DevDiv { uint32_t d, m, s; };

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const DevDiv &f)
{
  // d == 0 encodes "no division" (result 0); d == 1 is the identity
  if (f.d == 0) return 0;
  return (f.d == 1) ? n : ((__umulhi(n, f.m) + n) >> f.s);
}

struct TileParams {
  // tile dimensions in input (load) order
  int nt;
  DevDiv t_in[kMaxTileDims];       // tile extents, load order
  uint64_t is_in[kMaxTileDims];    // input strides, load order
  // tile dimensions in output (store) order
  DevDiv t_out[kMaxTileDims];      // tile extents, store order
  uint64_t os_out[kMaxTileDims];   // output strides, store order
  uint32_t ls_out[kMaxTileDims];   // LDS (load-order linear) strides, store order
  // grid over all fused dims
  int ng;
  DevDiv gdiv[kMaxGridDims];       // number of tiles along each dim
  uint64_t g_is[kMaxGridDims];     // input stride * tile extent
  uint64_t g_os[kMaxGridDims];     // output stride * tile extent
  uint32_t vol_tile;               // elements per tile
  uint32_t ntiles;
  DevDiv pad;                      // LDS slot = e + e / pad.d (pad.d = 0: no padding)
  DevDiv tv_in0, tv_out0;          // first tile extent on each side divided by the vector width
};

// Elements move as integer words of their size (pure data movement, so the
// result is bit-exact by construction); conjugation flips the sign bit of the
// imaginary half of a complex word.
template <typename W, bool CONJ>
__device__ __forceinline__ W conj_if(W v) { return v; }
template <>
__device__ __forceinline__ uint2 conj_if<uint2, true>(uint2 v) { v.y ^= 0x80000000u; return v; }
template <>
__device__ __forceinline__ uint4 conj_if<uint4, true>(uint4 v) { v.w ^= 0x80000000u; return v; }

template <typename W, int VEC>
struct __align__(sizeof(W) * VEC) Pack { W w[VEC]; };

// Hides a value's origin from the optimizer, so that addresses derived from it
// are recomputed where they are used instead of being hoisted out of the tile
// loop and held in registers for every element.
__device__ __forceinline__ void opaque(uint32_t &x) { asm volatile("" : "+v"(x)); }

// Streaming (nontemporal) global accesses: every element is read once and
// written once, so the data should not displace useful lines from L2/MALL.
// For tiles whose runs are whole cache lines only (rank-6 extent-24 R8: 595 us
// against 620 without the hint); a line shared with a neighbouring tile has to
// wait for the rest of it.
typedef unsigned int nt1 __attribute__((ext_vector_type(1)));
typedef unsigned int nt2 __attribute__((ext_vector_type(2)));
typedef unsigned int nt4 __attribute__((ext_vector_type(4)));
template <int BYTES>
struct NtWord;
template <>
struct NtWord<4> { typedef unsigned int type; };
template <>
struct NtWord<8> { typedef nt2 type; };
template <>
struct NtWord<16> { typedef nt4 type; };

template <typename P>
__device__ __forceinline__ P ld_stream(const P *p)
{
  typedef typename NtWord<sizeof(P)>::type U;
  const U u = __builtin_nontemporal_load(reinterpret_cast<const U *>(p));
  return __builtin_bit_cast(P, u);
}
template <typename P>
__device__ __forceinline__ void st_stream(P *p, const P &v)
{
  typedef typename NtWord<sizeof(P)>::type U;
  __builtin_nontemporal_store(__builtin_bit_cast(U, v), reinterpret_cast<U *>(p));
}

// Accesses of runs that begin and end inside cache lines, aligned to a 4-byte
// word only. They are left to the caches (no streaming hint): the rest of a
// line is the neighbouring tile's, and with the hint the R4 body of extents
// 37,29,41,23,31 took 124 us instead of 90.
typedef unsigned int un2 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned int un4 __attribute__((ext_vector_type(4), aligned(4)));
template <int BYTES>
struct RunWord;
template <>
struct RunWord<4> { typedef unsigned int type; };
template <>
struct RunWord<8> { typedef un2 type; };
template <>
struct RunWord<16> { typedef un4 type; };
template <typename P>
__device__ __forceinline__ P ld_run(const void *p)
{
  return __builtin_bit_cast(P, *static_cast<const typename RunWord<sizeof(P)>::type *>(p));
}
template <typename P>
__device__ __forceinline__ void st_run(void *p, const P &v)
{
  *static_cast<typename RunWord<sizeof(P)>::type *>(p) = __builtin_bit_cast(typename RunWord<sizeof(P)>::type, v);
}

// One workgroup walks tiles (persistent grid). Each thread owns EPT vectors of
// VEC consecutive elements along the input-minor dimension for the load and
// along the output-minor dimension for the store, so global accesses are
// 16-byte wide whenever both minor extents allow it.
//
// Register budget: a thread keeps per vector only its input offset, output
// offset and LDS read base; the LDS slots
// are recomputed per tile from those (a few integer operations) instead of
// being held for every element, which keeps the common instantiations at
// 30-60 VGPRs, i.e. at full occupancy.
template <typename W, int VEC, int EPT, bool CONJ, typename OffT>
__global__ __launch_bounds__(kTNT) void k_permute_tiled(const W *__restrict__ in, W *__restrict__ out,
                                                        const TileParams p)
{
  typedef Pack<W, VEC> P;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  W *lds = reinterpret_cast<W *>(lds_raw);
  const uint32_t tid = threadIdx.x;
  const uint32_t nvec = p.vol_tile / VEC;
  OffT in_off[EPT], out_off[EPT];
  uint32_t st_ls[EPT];
  // one-time decode of this thread's tile vectors (kept in registers)
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const uint32_t v = tid + (uint32_t)k * kTNT;
    uint32_t r = v;
    OffT io = 0, oo = 0;
    uint32_t ls = 0;
    for (int j = 0; j < p.nt; ++j) {
      const DevDiv &dv = j == 0 ? p.tv_in0 : p.t_in[j];
      const uint32_t q = fdiv(r, dv);
      uint32_t c = r - q * dv.d;
      if (j == 0) c *= VEC;
      r = q;
      io += (OffT)c * (OffT)p.is_in[j];
    }
    r = v;
    for (int j = 0; j < p.nt; ++j) {
      const DevDiv &dv = j == 0 ? p.tv_out0 : p.t_out[j];
      const uint32_t q = fdiv(r, dv);
      uint32_t c = r - q * dv.d;
      if (j == 0) c *= VEC;
      r = q;
      oo += (OffT)c * (OffT)p.os_out[j];
      ls += c * p.ls_out[j];
    }
    in_off[k] = io;
    out_off[k] = oo;
    st_ls[k] = ls;
  }
  const uint32_t step = p.ls_out[0];
  // tile base decode (uniform across the workgroup)
  auto decode = [&](uint32_t tile, OffT &bin, OffT &bout) {
    bin = bout = 0;
    uint32_t r = tile;
    for (int g = 0; g < p.ng; ++g) {
      const uint32_t q = fdiv(r, p.gdiv[g]);
      const uint32_t c = r - q * p.gdiv[g].d;
      r = q;
      bin += (OffT)c * (OffT)p.g_is[g];
      bout += (OffT)c * (OffT)p.g_os[g];
    }
  };
  P val[EPT];
  auto load = [&](OffT bin) {
#pragma unroll
    for (int k = 0; k < EPT; ++k)
      if (tid + (uint32_t)k * kTNT < nvec) val[k] = ld_stream(reinterpret_cast<const P *>(in + (bin + in_off[k])));
  };
  // the padding period is a multiple of VEC (checked by the planner), so the
  // VEC slots of one loaded vector are consecutive: base slot + j
  auto to_lds = [&]() {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      uint32_t v = tid + (uint32_t)k * kTNT;
      if (v < nvec) {
        opaque(v);
        const uint32_t e0 = v * VEC;
        const uint32_t b = e0 + fdiv(e0, p.pad);
#pragma unroll
        for (int j = 0; j < VEC; ++j) lds[b + j] = val[k].w[j];
      }
    }
  };
  auto from_lds = [&](OffT bout) {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      if (tid + (uint32_t)k * kTNT < nvec) {
        uint32_t base = st_ls[k];
        opaque(base);
        P o;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          const uint32_t e = base + j * step;
          o.w[j] = conj_if<W, CONJ>(lds[e + fdiv(e, p.pad)]);
        }
        st_stream(reinterpret_cast<P *>(out + (bout + out_off[k])), o);
      }
    }
  };
  uint32_t tile = blockIdx.x;
  if (tile >= p.ntiles) return;
  OffT bin, bout;
  decode(tile, bin, bout);
  load(bin);
  // software pipeline: the next tile's loads are in flight while the current
  // tile drains from LDS to memory
  while (true) {
    to_lds();
    __syncthreads();
    const uint32_t next = tile + gridDim.x;
    const OffT cur = bout;
    if (next < p.ntiles) {
      decode(next, bin, bout);
      load(bin);
    }
    from_lds(cur);
    if (next >= p.ntiles) break;
    __syncthreads();
    tile = next;
  }
}

// ---------------------------------------------------------------------------
// Permutation by runs: the form for tiles whose minor extents hold no whole
// vectors (odd extents), for bodies aligned to an element only, and for D +=
// f * L.
//
// A tile's contiguous run on each side may span several dimensions. A thread
// takes vectors of VEC consecutive elements of a run, whatever the alignment
// (global accesses need an element's only); a run's last vector starts early
// enough to be whole, so it repeats elements of the one before. A dimension
// that its tile extent does not divide is covered by tiles that overlap in
// the same way. Copies write repeated elements twice, with the same value; in
// the accumulating form the repeats are skipped. No access is masked, so a
// thread's loads fly together: with one masked 4-byte access at a time, a
// 31 M element R4 body of extents 37,29,41,23,31 took 130 us (1.9 TB/s).
struct RunParams {
  int nri, nro;                     // tile dimensions after the run, load / store order
  uint32_t ri, ro;                  // run lengths (elements)
  DevDiv nvi, nvo;                  // vectors per run
  uint32_t vecs_i, vecs_o;          // vectors per tile
  DevDiv t_in[kMaxTileDims];        // extents after the run, load order
  uint64_t is_in[kMaxTileDims];
  DevDiv t_run[kMaxTileDims];       // extents inside the output run
  uint32_t ls_run[kMaxTileDims];    // their LDS strides
  int nrun;
  DevDiv t_out[kMaxTileDims];       // extents after the run, store order
  uint64_t os_out[kMaxTileDims];
  uint32_t ls_out[kMaxTileDims];
  int g_out[kMaxTileDims];          // grid dimension of t_out[j]
  int g_run;                        // grid dimension of the run's last dimension
  uint32_t unit;                    // run elements per step of that dimension
  int ng;
  DevDiv gdiv[kMaxGridDims];        // tiles along each dimension, output order
  uint64_t g_is[kMaxGridDims], g_os[kMaxGridDims];
  uint32_t g_t[kMaxGridDims], g_last[kMaxGridDims];  // tile extent, start of the last tile
  uint32_t ntiles;
  DevDiv pad;                       // LDS slot = e + e / pad.d (pad.d = 0: no padding)
};

// Arithmetic view of a word for D += f * L (products and sums rounded
// separately, as the element-wise kernels do).
#pragma clang fp contract(off)
template <int KIND>
struct Acc1;
template <>
struct Acc1<R4> {
  typedef uint32_t W;
  __device__ __forceinline__ static W run(W d, W l, double fr, double)
  {
    const float t = __uint_as_float(l) * (float)fr;
    return __float_as_uint(__uint_as_float(d) + t);
  }
};
template <>
struct Acc1<R8> {
  typedef uint2 W;
  __device__ __forceinline__ static W run(W d, W l, double fr, double)
  {
    const double t = __builtin_bit_cast(double, l) * fr;
    return __builtin_bit_cast(uint2, __builtin_bit_cast(double, d) + t);
  }
};
template <>
struct Acc1<C4> {
  typedef uint2 W;
  __device__ __forceinline__ static W run(W d, W l, double fr, double fi)
  {
    const float re = __uint_as_float(l.x), im = __uint_as_float(l.y), f0 = (float)fr, f1 = (float)fi;
    const float a = re * f0, b = im * f1, c = re * f1, e = im * f0;
    const float tr = a - b, ti = c + e;
    return make_uint2(__float_as_uint(__uint_as_float(d.x) + tr), __float_as_uint(__uint_as_float(d.y) + ti));
  }
};
template <>
struct Acc1<C8> {
  typedef uint4 W;
  struct D2 { double re, im; };
  __device__ __forceinline__ static W run(W d, W l, double fr, double fi)
  {
    const D2 x = __builtin_bit_cast(D2, l), y = __builtin_bit_cast(D2, d);
    const double a = x.re * fr, b = x.im * fi, c = x.re * fi, e = x.im * fr;
    const double tr = a - b, ti = c + e;
    return __builtin_bit_cast(uint4, D2{y.re + tr, y.im + ti});
  }
};
// KIND 0: out[..] = conj?(in[..]); a data kind: out[..] += f * conj?(in[..]).
template <typename W, int VEC, int EPT, bool CONJ, typename OffT, int KIND>
__global__ __launch_bounds__(kTNT) void k_permute_runs(const W *__restrict__ in, W *__restrict__ out,
                                                       const RunParams p, double fr, double fi)
{
  typedef Pack<W, VEC> P;
  constexpr int NS = (VEC + 1) / 2;       // LDS slots of a vector, two to a register
  extern __shared__ __align__(16) unsigned char lds_raw[];
  W *lds = reinterpret_cast<W *>(lds_raw);
  const uint32_t tid = threadIdx.x;
  OffT in_off[EPT], out_off[EPT];
  uint32_t lslot[EPT][NS], sslot[EPT][NS];
  uint32_t skip[KIND ? EPT : 1];          // leading elements that repeat the vector before
  uint32_t ocrd[KIND ? EPT : 1];          // position inside the run, for overlapping tiles
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    {
      const uint32_t v = min(tid + (uint32_t)k * kTNT, p.vecs_i - 1);
      uint32_t q = fdiv(v, p.nvi);
      const uint32_t s = min((v - q * p.nvi.d) * VEC, p.ri - VEC);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const uint32_t sl = s + p.ri * q + e, slot = sl + fdiv(sl, p.pad);
        if (e & 1) lslot[k][e / 2] |= slot << 16;
        else lslot[k][e / 2] = slot;
      }
      OffT io = s;
      for (int j = 0; j < p.nri; ++j) {
        const uint32_t n = fdiv(q, p.t_in[j]);
        io += (OffT)(q - n * p.t_in[j].d) * (OffT)p.is_in[j];
        q = n;
      }
      in_off[k] = io;
    }
    const uint32_t v = min(tid + (uint32_t)k * kTNT, p.vecs_o - 1);
    uint32_t q = fdiv(v, p.nvo);
    const uint32_t s0 = (v - q * p.nvo.d) * VEC, s = min(s0, p.ro - VEC);
    if (KIND) {
      skip[k] = tid + (uint32_t)k * kTNT < p.vecs_o ? s0 - s : VEC;
      ocrd[k] = v;
    }
    OffT oo = s;
    uint32_t base = 0;
    for (int j = 0; j < p.nro; ++j) {
      const uint32_t n = fdiv(q, p.t_out[j]), c = q - n * p.t_out[j].d;
      oo += (OffT)c * (OffT)p.os_out[j];
      base += c * p.ls_out[j];
      q = n;
    }
    out_off[k] = oo;
    uint32_t r[VEC], sl[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      r[e] = s + e;
      sl[e] = base;
    }
    // (dimensions outside, elements inside: one wait for the arguments of a
    // dimension, not one per element)
    for (int j = 0; j < p.nrun; ++j) {
      const DevDiv t = p.t_run[j];
      const uint32_t ls = p.ls_run[j];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const uint32_t n = fdiv(r[e], t);
        sl[e] += (r[e] - n * t.d) * ls;
        r[e] = n;
      }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const uint32_t x = sl[e] + fdiv(sl[e], p.pad);
      if (e & 1) sslot[k][e / 2] |= x << 16;
      else sslot[k][e / 2] = x;
    }
  }
  // Place `at` of the grid-stride order -> tile: each XCD (workgroups go round
  // robin over eight) takes a contiguous range, so that the tiles sharing a
  // line meet in one L2 (1-3% over the plain order).
  const uint32_t per_xcd = p.ntiles / 8;
  auto tile_at = [&](uint32_t at) { return at < per_xcd * 8 ? at % 8 * per_xcd + at / 8 : at; };
  // tile index -> start along each dimension (the last tile of a dimension
  // ends at its end); lap: whether it repeats elements of the tile before
  auto decode = [&](uint32_t place, OffT &bi, OffT &bo, bool &lap) {
    bi = bo = 0;
    lap = false;
    uint32_t r = tile_at(place);
    for (int g = 0; g < p.ng; ++g) {
      const uint32_t q = fdiv(r, p.gdiv[g]), c = r - q * p.gdiv[g].d;
      r = q;
      const uint32_t at = min(c * p.g_t[g], p.g_last[g]);
      lap = lap || at != c * p.g_t[g];
      bi += (OffT)at * (OffT)p.g_is[g];
      bo += (OffT)at * (OffT)p.g_os[g];
    }
  };
  // elements of tile `tile` along grid dimension g that the tile before holds
  auto lap_of = [&](uint32_t place, int g) {
    uint32_t r = tile_at(place), c = 0;
    for (int i = 0; i <= g; ++i) {
      const uint32_t q = fdiv(r, p.gdiv[i]);
      c = r - q * p.gdiv[i].d;
      r = q;
    }
    return c * p.g_t[g] - min(c * p.g_t[g], p.g_last[g]);
  };
  uint32_t tile = blockIdx.x;
  if (tile >= p.ntiles) return;
  auto slot = [](const uint32_t (&x)[NS], int e) { return (e & 1) ? x[e / 2] >> 16 : x[e / 2] & 0xFFFFu; };
  P val[EPT], d[KIND ? EPT : 1];
  OffT bi, bo;
  bool lap;
  decode(tile, bi, bo, lap);
  auto load = [&]() {
#pragma unroll
    for (int k = 0; k < EPT; ++k) val[k] = ld_run<P>(in + (bi + in_off[k]));
  };
  load();
  while (true) {
    // D before the next tile's loads: both are waited for in issue order
    if constexpr (KIND != 0) {
#pragma unroll
      for (int k = 0; k < EPT; ++k) d[k] = ld_run<P>(out + (bo + out_off[k]));
    }
#pragma unroll
    for (int k = 0; k < EPT; ++k)
#pragma unroll
      for (int e = 0; e < VEC; ++e) lds[slot(lslot[k], e)] = val[k].w[e];
    __syncthreads();
    const uint32_t next = tile + gridDim.x;
    const OffT bo_cur = bo;
    const bool lap_cur = lap;
    if (next < p.ntiles) {
      decode(next, bi, bo, lap);
      load();
    }
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      P o;
#pragma unroll
      for (int e = 0; e < VEC; ++e) o.w[e] = conj_if<W, CONJ>(lds[slot(sslot[k], e)]);
      W *dst = out + (bo_cur + out_off[k]);
      if constexpr (KIND == 0) {
        st_run<P>(dst, o);
      } else {
        uint32_t first = skip[k];
        if (lap_cur && first < VEC) {  // elements that the tile before holds
          uint32_t q = fdiv(ocrd[k], p.nvo);
          const uint32_t s = min((ocrd[k] - q * p.nvo.d) * VEC, p.ro - VEC), run = lap_of(tile, p.g_run) * p.unit;
          if (run > s) first = max(first, min(run - s, (uint32_t)VEC));
          for (int j = 0; j < p.nro; ++j) {
            const uint32_t n = fdiv(q, p.t_out[j]);
            if (q - n * p.t_out[j].d < lap_of(tile, p.g_out[j])) first = VEC;
            q = n;
          }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) o.w[e] = Acc1<KIND>::run(d[k].w[e], o.w[e], fr, fi);
        if (first == 0) {
          st_run<P>(dst, o);
        } else {
#pragma unroll
          for (int e = 0; e < VEC; ++e)
            if ((uint32_t)e >= first) dst[e] = o.w[e];
        }
      }
    }
    if (next >= p.ntiles) break;
    __syncthreads();
    tile = next;
  }
}

// Generic per-element fallback (any rank): decode the input index, scatter.
struct ScatterParams {
  int rank;
  uint64_t vol;
  uint64_t ext[kMaxRank];
  uint64_t ostr[kMaxRank];
};

template <typename T, bool CONJ>
__global__ __launch_bounds__(kNT) void k_permute_scatter(const T *__restrict__ in, T *__restrict__ out,
                                                          const ScatterParams p)
{
  const uint64_t stride = (uint64_t)gridDim.x * kNT;
  for (uint64_t i = (uint64_t)blockIdx.x * kNT + threadIdx.x; i < p.vol; i += stride) {
    uint64_t r = i, o = 0;
    for (int d = 0; d < p.rank; ++d) {
      const uint64_t q = r / p.ext[d];
      o += (r - q * p.ext[d]) * p.ostr[d];
      r = q;
    }
    out[o] = conj_if<T, CONJ>(in[i]);
  }
}

template <typename T, bool CONJ>
__global__ __launch_bounds__(kNT) void k_copy(const T *__restrict__ in, T *__restrict__ out, uint64_t n)
{
  const uint64_t stride = (uint64_t)gridDim.x * kNT;
  for (uint64_t i = (uint64_t)blockIdx.x * kNT + threadIdx.x; i < n; i += stride) out[i] = conj_if<T, CONJ>(in[i]);
}

// Identity permutation of a 16-byte aligned body: one 16-byte streaming
// access per thread in one-wave workgroups, one workgroup per KiB. The
// dispatcher hands the workgroups out in index order, so the lines in flight
// at any moment form a compact window that sweeps the body; on this part
// that moves more bytes per second than any persistent grid-stride form
// (measured: 6.4-6.7 TB/s against 5.5-5.8 TB/s).
constexpr int kCopyNT = 64;
template <typename W, bool CONJ>
__global__ __launch_bounds__(kCopyNT) void k_copy16(const nt4 *__restrict__ in, nt4 *__restrict__ out, uint64_t n16)
{
  const uint64_t i = (uint64_t)blockIdx.x * kCopyNT + threadIdx.x;
  if (i >= n16) return;
  nt4 v = __builtin_nontemporal_load(in + i);
  if (CONJ) {  // complex words: flip the sign bit of each imaginary part
    if (sizeof(W) == 8) { v.y ^= 0x80000000u; v.w ^= 0x80000000u; }
    else v.w ^= 0x80000000u;
  }
  __builtin_nontemporal_store(v, out + i);
}

// ---------------------------------------------------------------------------
// host planning

struct Fused {
  int rank = 0;
  std::vector<int> ext;   // fused extents, input order
  std::vector<int> o2n;   // output position of each fused dim
};

Fused fuse_dims(int rank, const int *dims, const int *o2n)
{
  // keep non-unit dims, re-rank their output positions
  std::vector<int> keep;
  for (int i = 0; i < rank; ++i)
    if (dims[i] > 1) keep.push_back(i);
  std::vector<int> order(keep.size());
  std::iota(order.begin(), order.end(), 0);
  std::sort(order.begin(), order.end(), [&](int a, int b) { return o2n[keep[a]] < o2n[keep[b]]; });
  std::vector<int> pos(keep.size());
  for (size_t q = 0; q < order.size(); ++q) pos[order[q]] = (int)q;
  // fuse runs i, i+1 with pos[i+1] == pos[i] + 1 while the fused extent stays
  // an int (a run left unfused is still a valid description of the copy)
  Fused f;
  std::vector<int> grp_pos;
  for (size_t i = 0; i < keep.size(); ++i) {
    if (i > 0 && pos[i] == pos[i - 1] + 1 && (int64_t)f.ext.back() * dims[keep[i]] <= INT32_MAX) {
      f.ext.back() *= dims[keep[i]];
    } else {
      f.ext.push_back(dims[keep[i]]);
      grp_pos.push_back(pos[i]);
    }
  }
  f.rank = (int)f.ext.size();
  std::vector<int> ord(f.rank);
  std::iota(ord.begin(), ord.end(), 0);
  std::sort(ord.begin(), ord.end(), [&](int a, int b) { return grp_pos[a] < grp_pos[b]; });
  f.o2n.assign(f.rank, 0);
  for (int q = 0; q < f.rank; ++q) f.o2n[ord[q]] = q;
  return f;
}

// Smallest divisor of ext in [need, 2*need], else need itself. With
// unit_bytes > 0 (the bytes of the contiguous run the split extends), the
// smallest divisor in [need, 4*need] that makes the run a whole number of
// cache lines is preferred: runs that end mid-line leave lines split between
// tiles.
int pick_split(int ext, int need, long unit_bytes = 0)
{
  if (unit_bytes > 0)
    for (int t = need; t <= std::min(ext, 4 * need); ++t)
      if (ext % t == 0 && (unit_bytes * t) % kLine == 0) return t;
  for (int t = need; t <= std::min(ext, 2 * need); ++t)
    if (ext % t == 0) return t;
  return std::min(ext, need);
}

struct TilePlan {
  std::vector<int> t;   // tile extent per fused dim (0: not a tile dim)
  long vol = 0;
  int in_run = 0, out_run = 0;
};

TilePlan choose_tile(const Fused &f, int target_in, int target_out, int align_es)
{
  const int r = f.rank;
  std::vector<int> n2o(r);
  for (int i = 0; i < r; ++i) n2o[f.o2n[i]] = i;
  TilePlan tp;
  tp.t.assign(r, 0);
  long run = 1;
  for (int i = 0; i < r; ++i) {
    const long need = (target_in + run - 1) / run;
    if (need >= f.ext[i]) {
      tp.t[i] = f.ext[i];
      run *= f.ext[i];
      if (run >= target_in) break;
    } else {
      tp.t[i] = pick_split(f.ext[i], (int)need, run * align_es);
      run *= tp.t[i];
      break;
    }
  }
  tp.in_run = (int)std::min<long>(run, 1 << 30);
  run = 1;
  for (int q = 0; q < r; ++q) {
    const int i = n2o[q];
    const long need = (target_out + run - 1) / run;
    if (tp.t[i] > 0 && tp.t[i] < f.ext[i] && tp.t[i] < need)
      tp.t[i] = pick_split(f.ext[i], (int)std::min<long>(need, f.ext[i]), run * align_es);
    if (tp.t[i] == 0) tp.t[i] = need >= f.ext[i] ? f.ext[i] : pick_split(f.ext[i], (int)need, run * align_es);
    run *= tp.t[i];
    if (tp.t[i] < f.ext[i] || run >= target_out) break;
  }
  tp.out_run = (int)std::min<long>(run, 1 << 30);
  // the input run may have grown through the output walk
  run = 1;
  for (int i = 0; i < r; ++i) {
    if (tp.t[i] == 0) break;
    run *= tp.t[i];
    if (tp.t[i] < f.ext[i]) break;
  }
  tp.in_run = (int)std::min<long>(run, 1 << 30);
  tp.vol = 1;
  for (int i = 0; i < r; ++i)
    if (tp.t[i]) tp.vol *= tp.t[i];
  return tp;
}

// Grows a tile that meets its run targets but is too small to keep a
// workgroup busy (e.g. when the input- and output-minor dimensions coincide):
// alternately extends the input-order and output-order prefixes (doubling the
// first partial dimension, or opening the next one) until vol >= min_vol.
void grow_tile(const Fused &f, TilePlan &tp, long min_vol, long max_vol)
{
  const int r = f.rank;
  std::vector<int> n2o(r);
  for (int i = 0; i < r; ++i) n2o[f.o2n[i]] = i;
  auto volume = [&]() {
    long v = 1;
    for (int i = 0; i < r; ++i)
      if (tp.t[i]) v *= tp.t[i];
    return v;
  };
  int side = 0, stuck = 0;
  while (volume() < min_vol && stuck < 2) {
    int dim = -1;
    for (int q = 0; q < r; ++q) {
      const int i = side == 0 ? q : n2o[q];
      if (tp.t[i] < f.ext[i]) { dim = i; break; }
    }
    side ^= 1;
    if (dim < 0) { ++stuck; continue; }
    const int old = tp.t[dim];
    const int want = old == 0 ? 2 : old * 2;
    const int nt = pick_split(f.ext[dim], std::min(want, f.ext[dim]));
    const long nv = volume() / std::max(old, 1) * nt;
    if (nv > max_vol) { ++stuck; continue; }
    stuck = 0;
    tp.t[dim] = nt;
  }
  tp.vol = volume();
  long run = 1;
  for (int i = 0; i < r; ++i) {
    if (tp.t[i] == 0) break;
    run *= tp.t[i];
    if (tp.t[i] < f.ext[i]) break;
  }
  tp.in_run = (int)std::min<long>(run, 1 << 30);
  run = 1;
  for (int q = 0; q < r; ++q) {
    const int i = n2o[q];
    if (tp.t[i] == 0) break;
    run *= tp.t[i];
    if (tp.t[i] < f.ext[i]) break;
  }
  tp.out_run = (int)std::min<long>(run, 1 << 30);
}

// LDS bank-conflict degree of the store phase for a padding period.
int conflict_cost(const std::vector<uint32_t> &slots, int words_per_elem, uint32_t period)
{
  int cost = 0;
  for (int banks : {32, 64}) {
    for (size_t base = 0; base + 1 <= slots.size(); base += 64) {
      std::vector<std::vector<uint32_t>> hit(banks);
      for (size_t l = base; l < std::min(slots.size(), base + 64); ++l) {
        const uint32_t s = slots[l];
        const uint32_t slot = period ? s + s / period : s;
        for (int w = 0; w < words_per_elem; ++w) {
          const uint32_t word = slot * words_per_elem + w;
          auto &v = hit[word % banks];
          if (std::find(v.begin(), v.end(), word) == v.end()) v.push_back(word);
        }
      }
      int mx = 0;
      for (auto &v : hit) mx = std::max<int>(mx, (int)v.size());
      cost += mx;
    }
  }
  return cost;
}

DevDiv to_dev(uint32_t d)
{
  if (d == 0) return DevDiv{0, 0, 0};  // "no division" marker
  FastDiv f(d);
  return DevDiv{f.d, f.m, f.s};
}

struct Planned {
  int path = 0;  // 0 copy, 1 tiled, 2 scatter, 3 tiled by runs
  Fused f;
  TileParams tp{};
  RunParams rp{};
  int ept = 0;
  size_t lds_bytes = 0;
  int grid = 0;
  int vec = 1;        // elements per global access
  bool wide = false;  // 64-bit element offsets
  int cus = 0;        // compute units the grid was sized for
  TilePlan tile;
};

int num_cus_current()
{
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0) cus = prop.multiProcessorCount;
  }
  return cus;
}

// Vector width the kernel can use for a tile: both minor dimensions (the first
// tile dimension in input and in output order) and their tile extents must be
// multiples of it, so that every vector is aligned and whole.
int tile_vec(const Fused &f, const TilePlan &tp, int es)
{
  int i0 = -1, o0 = -1;
  for (int i = 0; i < f.rank && i0 < 0; ++i)
    if (tp.t[i] > 0) i0 = i;
  std::vector<int> n2o(f.rank);
  for (int i = 0; i < f.rank; ++i) n2o[f.o2n[i]] = i;
  for (int q = 0; q < f.rank && o0 < 0; ++q)
    if (tp.t[n2o[q]] > 0) o0 = n2o[q];
  if (i0 < 0 || o0 < 0) return 1;
  for (int cand = 16 / es; cand >= 2; cand /= 2)
    if (f.ext[i0] % cand == 0 && tp.t[i0] % cand == 0 && f.ext[o0] % cand == 0 && tp.t[o0] % cand == 0) return cand;
  return 1;
}

// Tile of the run form: an input-minor and an output-minor group of
// dimensions, each walked until it covers `target` elements. A dimension that
// is cut gets tiles of nearly equal extent (the last one overlaps its
// neighbour by less than the number of tiles); one of sixteen tiles and more
// gets whole lines (a step is `run` elements) where they are at most a quarter
// longer: its last tile repeats a sixteenth at most, and with 65 columns instead
// of 64 every line between two tiles is read twice and written in parts (C4
// 2350648 x 16 transposed 136 us with 65, 118 with 64).
int cut_extent(int ext, long need, long run, int es)
{
  if (need >= ext) return ext;
  long step = kLine / es;
  while (step > 1 && run % 2 == 0) { step /= 2; run /= 2; }
  const long lines = (need + step - 1) / step * step;
  if (4 * lines <= 5 * need && ext >= 16 * lines) return (int)lines;
  const int n = std::max<int>(1, (int)(ext / need));  // tiles of at least `need`
  return (ext + n - 1) / n;
}

bool plan_runs(int es, const Fused &f, int cus, int vec, Planned &pl, bool choose_pad)
{
  const int r = f.rank;
  std::vector<int> n2o(r);
  for (int i = 0; i < r; ++i) n2o[f.o2n[i]] = i;
  uint64_t vol = 1;
  for (int e : f.ext) vol *= (uint64_t)e;
  const long max_vol = kRunTileMaxBytes / es;
  const long min_vol =
      std::min<long>({max_vol, kRunTileMinBytes / es, std::max<long>(1024, (long)(vol / (4 * (uint64_t)std::max(cus, 1))))});
  std::vector<int> t(r);
  auto volume = [&] {
    long v = 1;
    for (int x : t) v *= std::max(x, 1);
    return v;
  };
  // whether the tile's vectors, those at the runs' ends included, fit the threads
  auto fits = [&] {
    for (bool in : {true, false}) {
      long run = 1;
      for (int q = 0; q < r; ++q) {
        const int i = in ? q : n2o[q];
        run *= std::max(t[i], 1);
        if (t[i] < f.ext[i]) break;
      }
      if ((run + vec - 1) / vec * (volume() / run) > (long)kTNT * kRunEPT) return false;
    }
    return volume() <= max_vol;
  };
  auto walk = [&](long target, bool in) {
    long run = 1;
    for (int q = 0; q < r; ++q) {
      const int i = in ? q : n2o[q];
      const int want = cut_extent(f.ext[i], (target + run - 1) / run, run, es);
      t[i] = std::max(t[i], want);
      run *= t[i];
      if (t[i] < f.ext[i] || run >= target) break;
    }
  };
  auto try_target = [&](long target) {
    std::fill(t.begin(), t.end(), 0);
    walk(target, true);
    walk(target, false);
    return fits() && std::count_if(t.begin(), t.end(), [](int x) { return x > 0; }) <= kMaxTileDims;
  };
  // (tiles of at most a sixth of a CU's share: a 31 MB body in 1.5 tiles per
  // resident workgroup took 48 us, in 6 smaller ones 30)
  const long share = std::max<long>(2048, (long)(vol / (6 * (uint64_t)std::max(cus, 1))));
  long target = std::max(8, 512 / es);
  while (target > 1 && (!try_target(target) || (volume() > share && target * es > kLine))) target /= 2;
  if (!try_target(target)) return false;
  // grow towards min_vol, alternating sides
  for (int side = 0, stuck = 0; volume() < min_vol && stuck < 2; side ^= 1) {
    int dim = -1;
    long run = 1;
    for (int q = 0; q < r && dim < 0; ++q) {
      const int i = side == 0 ? q : n2o[q];
      if (t[i] < f.ext[i]) dim = i;
      else run *= t[i];
    }
    if (dim < 0) { ++stuck; continue; }
    const int old = t[dim];
    t[dim] = cut_extent(f.ext[dim], std::max(2l, 2l * old), run, es);
    if (!fits() || volume() > share ||
        std::count_if(t.begin(), t.end(), [](int x) { return x > 0; }) > kMaxTileDims) {
      t[dim] = old;
      ++stuck;
      continue;
    }
    stuck = 0;
  }
  RunParams &P = pl.rp;
  std::memset(&P, 0, sizeof(P));
  std::vector<uint64_t> istr(r), ostr(r);
  uint64_t st = 1;
  for (int i = 0; i < r; ++i) { istr[i] = st; st *= (uint64_t)f.ext[i]; }
  st = 1;
  for (int q = 0; q < r; ++q) { ostr[n2o[q]] = st; st *= (uint64_t)f.ext[n2o[q]]; }
  std::vector<uint32_t> ls(r, 0);
  uint32_t lv = 1;
  for (int i = 0; i < r; ++i)
    if (t[i] > 0) { ls[i] = lv; lv *= (uint32_t)t[i]; }
  // run prefixes
  P.ri = P.ro = 1;
  bool run = true;
  for (int i = 0; i < r; ++i) {
    if (run && t[i] > 0) P.ri *= (uint32_t)t[i];
    else if (t[i] > 0) {
      P.t_in[P.nri] = to_dev((uint32_t)t[i]);
      P.is_in[P.nri++] = istr[i];
    }
    if (t[i] < f.ext[i]) run = false;
  }
  run = true;
  P.unit = 1;
  for (int q = 0; q < r; ++q) {
    const int i = n2o[q];
    if (run && t[i] > 0) {
      P.unit = P.ro;
      P.ro *= (uint32_t)t[i];
      P.t_run[P.nrun] = to_dev((uint32_t)t[i]);
      P.ls_run[P.nrun++] = ls[i];
      P.g_run = q;
    } else if (t[i] > 0) {
      P.t_out[P.nro] = to_dev((uint32_t)t[i]);
      P.os_out[P.nro] = ostr[i];
      P.ls_out[P.nro] = ls[i];
      P.g_out[P.nro++] = q;
    }
    if (t[i] < f.ext[i]) run = false;
  }
  if (P.ri < (uint32_t)vec || P.ro < (uint32_t)vec) return false;
  const uint32_t tv = lv;
  P.nvi = to_dev((P.ri + vec - 1) / vec);
  P.nvo = to_dev((P.ro + vec - 1) / vec);
  P.vecs_i = P.nvi.d * (tv / P.ri);
  P.vecs_o = P.nvo.d * (tv / P.ro);
  uint64_t ntiles = 1;
  P.ng = r;
  for (int q = 0; q < r; ++q) {  // output order (see plan)
    const int i = n2o[q], ti = std::max(t[i], 1), n = (f.ext[i] + ti - 1) / ti;
    P.gdiv[q] = to_dev((uint32_t)n);
    P.g_is[q] = istr[i];
    P.g_os[q] = ostr[i];
    P.g_t[q] = (uint32_t)ti;
    P.g_last[q] = (uint32_t)(f.ext[i] - ti);
    ntiles *= (uint64_t)n;
  }
  if (ntiles >= (1ull << 31)) return false;
  P.ntiles = (uint32_t)ntiles;
  // LDS padding: simulated bank conflicts of the first vectors' store-phase
  // reads (a millisecond or so per plan: not for a plan that is only described)
  std::vector<uint32_t> slots;
  for (uint32_t v = 0; choose_pad && v < std::min<uint32_t>(P.vecs_o, kTNT); ++v) {
    uint32_t q = v / P.nvo.d, s = std::min((v % P.nvo.d) * (uint32_t)vec, P.ro - (uint32_t)vec), l = 0;
    for (int j = 0; j < P.nro; ++j) { l += q % P.t_out[j].d * P.ls_out[j]; q /= P.t_out[j].d; }
    for (int j = 0; j < P.nrun; ++j) { l += s % P.t_run[j].d * P.ls_run[j]; s /= P.t_run[j].d; }
    slots.push_back(l);
  }
  const int words = std::max(1, es / 4);
  std::vector<uint32_t> cands = {4, 8, 16, 32, 64, 128, 256, P.ri};
  uint32_t best = 0;
  int bestc = choose_pad ? conflict_cost(slots, words, 0) : 0;
  for (uint32_t c : cands) {
    if (!choose_pad || c < 4 || c >= tv) continue;
    const int cc = conflict_cost(slots, words, c);
    if (cc < bestc) { bestc = cc; best = c; }
  }
  P.pad = to_dev(best);
  const uint32_t nv = std::max(P.vecs_i, P.vecs_o);
  int ept = 1;
  while ((uint32_t)ept * kTNT < nv) ept *= 2;
  if (ept > kRunEPT) return false;
  pl.ept = ept;
  pl.vec = vec;
  pl.wide = vol >= (1ull << 32);
  pl.lds_bytes = (tv + (best ? tv / best + 1 : 0)) * (size_t)es;
  pl.cus = cus;
  const int per_cu = std::max(1, std::min(kTiledPerCU, (int)(160 * 1024 / std::max<size_t>(pl.lds_bytes, 1))));
  pl.grid = (int)std::min<uint64_t>(ntiles, (uint64_t)cus * per_cu);
  pl.path = 3;
  return true;
}

// align: bytes that both bodies are aligned to (at most 16).
int plan(int es, int rank, const int *dims, const int *o2n, Planned &pl, int cus, int align, bool choose_pad = true)
{
  pl.f = fuse_dims(rank, dims, o2n);
  const Fused &f = pl.f;
  bool identity = true;
  for (int i = 0; i < f.rank; ++i) identity = identity && f.o2n[i] == i;
  if (f.rank <= 1 || identity) { pl.path = 0; return 0; }
  if (f.rank > kMaxGridDims) { pl.path = 2; return 0; }
  uint64_t vol = 1;
  for (int e : f.ext) vol *= (uint64_t)e;
  // a small tensor gets tiles small enough for about four per CU (a tile
  // takes one workgroup and the grid would otherwise leave CUs idle)
  const long min_vol = std::min<long>(kTileMinVol, std::max<long>(1024, (long)(vol / (4 * (uint64_t)std::max(cus, 1)))));
  // two attempts: first with splits that keep runs whole cache lines, then
  // without, if the aligned tile would need more vectors per thread than the
  // kernel is instantiated for
  TilePlan tp;
  bool ok = false;
  for (int attempt = 0; attempt < 2 && !ok; ++attempt) {
    const int align_es = attempt == 0 ? es : 0;
    // the second attempt bounds the tile by one element per vector, so that
    // it always fits the kernel's vector slots
    const long max_vol = std::min<long>((long)kTNT * kMaxEPT * (attempt == 0 ? 16 / es : 1), kTileMaxBytes / es);
    int target = std::max(8, 256 / es);
    while (true) {
      tp = choose_tile(f, target, target, align_es);
      int ntd = 0;
      for (int x : tp.t) ntd += x > 0;
      if ((tp.vol <= max_vol && ntd <= kMaxTileDims) || target <= 1) break;
      target = std::max(1, target / 2);
    }
    TilePlan g = tp;
    grow_tile(f, g, std::min(min_vol, max_vol), max_vol);
    int gd = 0;
    for (int x : g.t) gd += x > 0;
    if (gd <= kMaxTileDims) tp = g;
    ok = tp.vol <= max_vol && (tp.vol + (long)kTNT * tile_vec(f, tp, es) - 1) / ((long)kTNT * tile_vec(f, tp, es)) <= kMaxEPT;
  }
  int ntd = 0, nrag = 0;
  for (int i = 0; i < f.rank; ++i) {
    if (tp.t[i] > 0) ++ntd;
    if (tp.t[i] > 0 && f.ext[i] % tp.t[i] != 0) ++nrag;
  }
  uint64_t ntiles = 1;
  for (int i = 0; i < f.rank; ++i) ntiles *= (uint64_t)((f.ext[i] + std::max(tp.t[i], 1) - 1) / std::max(tp.t[i], 1));
  // The vector form takes tiles that divide the tensor, with 16-byte vectors
  // along both minor dimensions and runs of whole cache lines on both sides;
  // everything else goes by runs (shapes of either kind that could go both
  // ways: within 1% on 60 random ones)
  const bool tiled = ok && ntd <= kMaxTileDims && nrag == 0 && ntiles < (1ull << 31) && align >= 16 &&
                     tile_vec(f, tp, es) * es == 16 && (long)tp.in_run * es % kLine == 0 &&
                     (long)tp.out_run * es % kLine == 0;
  if (!tiled) {
    pl.path = plan_runs(es, f, cus, 16 / es, pl, choose_pad) ? 3 : 2;
    return 0;
  }
  pl.path = 1;
  pl.tile = tp;
  TileParams &P = pl.tp;
  std::memset(&P, 0, sizeof(P));
  // strides
  std::vector<uint64_t> istr(f.rank), ostr_out(f.rank), ostr(f.rank);
  uint64_t s = 1;
  for (int i = 0; i < f.rank; ++i) { istr[i] = s; s *= (uint64_t)f.ext[i]; }
  std::vector<int> n2o(f.rank);
  for (int i = 0; i < f.rank; ++i) n2o[f.o2n[i]] = i;
  s = 1;
  for (int q = 0; q < f.rank; ++q) { ostr_out[q] = s; s *= (uint64_t)f.ext[n2o[q]]; }
  for (int i = 0; i < f.rank; ++i) ostr[i] = ostr_out[f.o2n[i]];
  // tile dims in load order
  std::vector<int> tin, tout;
  for (int i = 0; i < f.rank; ++i)
    if (tp.t[i] > 0) tin.push_back(i);
  for (int q = 0; q < f.rank; ++q)
    if (tp.t[n2o[q]] > 0) tout.push_back(n2o[q]);
  P.nt = (int)tin.size();
  std::vector<uint32_t> lstride(f.rank, 0);
  uint32_t ls = 1;
  for (int j = 0; j < P.nt; ++j) {
    P.t_in[j] = to_dev((uint32_t)tp.t[tin[j]]);
    P.is_in[j] = istr[tin[j]];
    lstride[tin[j]] = ls;
    ls *= (uint32_t)tp.t[tin[j]];
  }
  for (int j = 0; j < P.nt; ++j) {
    P.t_out[j] = to_dev((uint32_t)tp.t[tout[j]]);
    P.os_out[j] = ostr[tout[j]];
    P.ls_out[j] = lstride[tout[j]];
  }
  // grid: tile index decoded fastest along the output's minor dimension, then
  // in output order, so that the tiles in flight at once (consecutive indices
  // across the persistent grid) write neighbouring regions of the output.
  // Measured against input order on the 174-transpose workload (+1.9%
  // geometric mean) and on 40 random shapes of ranks 2-6 (+5.9%).
  P.ng = f.rank;
  for (int q = 0; q < f.rank; ++q) {
    const int i = n2o[q];
    const uint32_t t = (uint32_t)std::max(tp.t[i], 1);
    const uint32_t n = (uint32_t)((f.ext[i] + t - 1) / t);
    P.gdiv[q] = to_dev(n);
    P.g_is[q] = istr[i] * t;
    P.g_os[q] = ostr[i] * t;
  }
  P.vol_tile = (uint32_t)tp.vol;
  P.ntiles = (uint32_t)ntiles;
  // LDS padding by simulated store-phase conflicts (first 256 store slots)
  std::vector<uint32_t> st;
  for (uint32_t e = 0; e < std::min<uint32_t>(P.vol_tile, kTNT); ++e) {
    uint32_t r = e, l = 0;
    for (int j = 0; j < P.nt; ++j) {
      const uint32_t d = P.t_out[j].d;
      l += (r % d) * P.ls_out[j];
      r /= d;
    }
    st.push_back(l);
  }
  const int words = std::max(1, es / 4);
  std::vector<uint32_t> cands = {0, 4, 8, 16, 32, 64, 128, 256};
  uint32_t prod = 1;
  for (int j = 0; j < P.nt && j < 3; ++j) { prod *= P.t_in[j].d; cands.push_back(prod); }
  uint32_t best = 0;
  int bestc = choose_pad ? conflict_cost(st, words, 0) : 0;
  for (uint32_t c : cands) {
    if (!choose_pad || c == 0 || c >= P.vol_tile) continue;
    const int cc = conflict_cost(st, words, c);
    if (cc < bestc) { bestc = cc; best = c; }
  }
  P.pad = to_dev(best);
  const int vec = 16 / es;
  // the kernel writes one vector to consecutive LDS slots, so a vector must
  // not straddle a padding period
  if (best % (uint32_t)vec != 0) best = 0;
  P.pad = to_dev(best);
  pl.vec = vec;
  P.tv_in0 = to_dev((uint32_t)(tp.t[tin[0]] / vec));
  P.tv_out0 = to_dev((uint32_t)(tp.t[tout[0]] / vec));
  int ept = 1;
  while ((long)ept * kTNT * vec < tp.vol) ept *= 2;
  pl.ept = ept;
  pl.wide = vol >= (1ull << 32);
  const size_t slots = P.vol_tile + (best ? P.vol_tile / best + 1 : 0);
  pl.lds_bytes = slots * (size_t)es;
  // resident workgroups per CU: measured on the transpose workload, 16 waves
  // per CU move more bytes per second than 32 (the DRAM sees fewer concurrent
  // streams); LDS may allow fewer
  const int per_cu = std::max(1, std::min(kTiledPerCU, (int)(160 * 1024 / std::max<size_t>(pl.lds_bytes, 1))));
  pl.cus = cus;
  pl.grid = (int)std::min<uint64_t>(ntiles, (uint64_t)cus * per_cu);
  return 0;
}

// Workgroups of one kernel instantiation that a CU holds at once as far as its
// registers allow (LDS is accounted for by the planner); the persistent grid
// is capped at this so that every workgroup is resident from the start.
template <typename W, int VEC, int EPT, bool CONJ, typename OffT>
int resident_per_cu()
{
  static const int n = [] {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_permute_tiled<W, VEC, EPT, CONJ, OffT>, kTNT, 0) !=
            hipSuccess || b <= 0)
      b = 1;
    return b;
  }();
  return n;
}

template <typename W, bool CONJ, typename OffT>
int launch_tiled_o(const Planned &pl, const void *in, void *out, hipStream_t s)
{
  constexpr int VEC = 16 / (int)sizeof(W);
  const W *a = static_cast<const W *>(in);
  W *b = static_cast<W *>(out);
  switch (pl.ept) {
#define XT_CASE(E)                                                                                             \
  case E: {                                                                                                    \
    const int cap = pl.cus * resident_per_cu<W, VEC, E, CONJ, OffT>();                                         \
    const dim3 g(std::min(pl.grid, cap));                                                                      \
    hipLaunchKernelGGL((k_permute_tiled<W, VEC, E, CONJ, OffT>), g, dim3(kTNT), pl.lds_bytes, s, a, b, pl.tp); \
    break;                                                                                                     \
  }
    XT_CASE(1) XT_CASE(2) XT_CASE(4) XT_CASE(8)
#undef XT_CASE
  default: return TALSH_FAILURE;
  }
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

template <typename W, bool CONJ>
int launch_tiled_t(const Planned &pl, const void *in, void *out, hipStream_t s)
{
  return pl.wide ? launch_tiled_o<W, CONJ, uint64_t>(pl, in, out, s) : launch_tiled_o<W, CONJ, uint32_t>(pl, in, out, s);
}

// Launches the run form (KIND 0: copy; a data kind: accumulate f times the
// permuted input).
template <typename W, bool CONJ, int KIND, typename OffT>
int launch_runs_o(const Planned &pl, const void *in, void *out, double fr, double fi, hipStream_t s)
{
  constexpr int VEC = 16 / (int)sizeof(W);
  const W *a = static_cast<const W *>(in);
  W *b = static_cast<W *>(out);
  switch (pl.ept) {
#define XT_CASE(E)                                                                                              \
  case E:                                                                                                       \
    hipLaunchKernelGGL((k_permute_runs<W, VEC, E, CONJ, OffT, KIND>), dim3(pl.grid), dim3(kTNT), pl.lds_bytes, s, \
                       a, b, pl.rp, fr, fi);                                                                    \
    break;
    XT_CASE(1) XT_CASE(2) XT_CASE(4)
#undef XT_CASE
  default: return TALSH_FAILURE;
  }
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}
template <typename W, bool CONJ, int KIND>
int launch_runs(const Planned &pl, const void *in, void *out, double fr, double fi, hipStream_t s)
{
  return pl.wide ? launch_runs_o<W, CONJ, KIND, uint64_t>(pl, in, out, fr, fi, s)
                 : launch_runs_o<W, CONJ, KIND, uint32_t>(pl, in, out, fr, fi, s);
}

template <typename W, bool CONJ>
int launch_copy_t(const void *in, void *out, uint64_t n, hipStream_t s, int cus)
{
  const uint64_t bytes = n * sizeof(W);
  if (bytes % 16 == 0 && ((uintptr_t)in % 16) == 0 && ((uintptr_t)out % 16) == 0) {
    const uint64_t n16 = bytes / 16;
    const uint64_t blocks = (n16 + kCopyNT - 1) / kCopyNT;
    // one launch covers up to 2^31 - 1 workgroups of 1 KiB (2 TiB): always
    // enough for a body that fits in device memory
    if (blocks >= (1ull << 31)) return TALSH_INVALID_ARGS;
    hipLaunchKernelGGL((k_copy16<W, CONJ>), dim3((unsigned)blocks), dim3(kCopyNT), 0, s,
                       static_cast<const nt4 *>(in), static_cast<nt4 *>(out), n16);
    return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
  }
  const uint64_t blocks = std::min<uint64_t>((n + kNT - 1) / kNT, (uint64_t)cus * 16);
  if (blocks == 0) return 0;
  hipLaunchKernelGGL((k_copy<W, CONJ>), dim3((unsigned)blocks), dim3(kNT), 0, s, static_cast<const W *>(in),
                     static_cast<W *>(out), n);
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

template <typename W, bool CONJ>
int launch_scatter_t(const Fused &f, const void *in, void *out, hipStream_t s, int cus)
{
  ScatterParams h;
  std::memset(&h, 0, sizeof(h));
  h.rank = f.rank;
  h.vol = 1;
  std::vector<int> n2o(f.rank);
  for (int i = 0; i < f.rank; ++i) n2o[f.o2n[i]] = i;
  std::vector<uint64_t> ostr_out(f.rank);
  uint64_t st = 1;
  for (int q = 0; q < f.rank; ++q) { ostr_out[q] = st; st *= (uint64_t)f.ext[n2o[q]]; }
  for (int i = 0; i < f.rank; ++i) {
    h.ext[i] = (uint64_t)f.ext[i];
    h.ostr[i] = ostr_out[f.o2n[i]];
    h.vol *= h.ext[i];
  }
  const uint64_t blocks = std::min<uint64_t>((h.vol + kNT - 1) / kNT, (uint64_t)cus * 16);
  hipLaunchKernelGGL((k_permute_scatter<W, CONJ>), dim3((unsigned)std::max<uint64_t>(blocks, 1)), dim3(kNT), 0, s,
                     static_cast<const W *>(in), static_cast<W *>(out), h);
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

template <typename W, bool CONJ>
int dispatch(const Planned &pl, const void *in, void *out, uint64_t vol, hipStream_t s, int cus)
{
  if (pl.path == 0) return launch_copy_t<W, CONJ>(in, out, vol, s, cus);
  if (pl.path == 1) return launch_tiled_t<W, CONJ>(pl, in, out, s);
  if (pl.path == 3) return launch_runs<W, CONJ, 0>(pl, in, out, 0.0, 0.0, s);
  return launch_scatter_t<W, CONJ>(pl.f, in, out, s, cus);
}

int compute_units()
{
  static const int cus = num_cus_current();
  return cus;
}

// The plan of a permutation (add: of its accumulating form, path 3 or none).
// Plans are memoized per (form, element size, alignment, extents,
// permutation): planning (fusion, tile choice, bank-conflict simulation) costs
// far more host time than a launch.
Planned planned(int es, int rank, const int *dims, const int *o2n, const void *in, const void *out, bool add)
{
  static std::mutex mu;
  static std::unordered_map<std::string, Planned> cache;
  const uintptr_t addr = (uintptr_t)in | (uintptr_t)out;
  const int align = add || addr % 16 == 0 ? 16 : addr % 8 == 0 ? 8 : 4;
  std::string key;
  key.reserve(8 * rank + 8);
  key.append(std::to_string(add ? -es : es)).push_back('@');
  key.append(std::to_string(align)).push_back(':');
  for (int i = 0; i < rank; ++i) key.append(std::to_string(dims[i])).append(",").append(std::to_string(o2n[i])).push_back(';');
  std::lock_guard<std::mutex> g(mu);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  Planned pl;
  if (add) {
    pl.f = fuse_dims(rank, dims, o2n);
    if (pl.f.rank < 2 || pl.f.rank > kMaxGridDims || !plan_runs(es, pl.f, compute_units(), 16 / es, pl, true)) pl.path = 2;
  } else {
    plan(es, rank, dims, o2n, pl, compute_units(), align);
  }
  if (cache.size() >= 4096) cache.clear();
  cache.emplace(key, pl);
  return pl;
}

bool valid_permutation(int rank, const int *dims, const int *o2n)
{
  std::vector<int> seen(std::max(rank, 1), 0);
  for (int i = 0; i < rank; ++i) {
    if (dims[i] <= 0 || o2n[i] < 0 || o2n[i] >= rank || seen[o2n[i]]) return false;
    seen[o2n[i]] = 1;
  }
  return true;
}

}  // namespace

int plan_permute_info(int kind, int rank, const int *dims_in, const int *o2n, PermuteInfo *info, bool with_padding)
{
  const int es = kind_size(kind);
  if (es == 0 || rank < 0 || rank > kMaxRank) return TALSH_INVALID_ARGS;
  Planned pl;
  plan(es, rank, dims_in, o2n, pl, 256, 16, with_padding);
  info->fused_rank = pl.f.rank;
  if (pl.path == 3) {
    info->path = 1;
    info->tile_volume = (int)(pl.rp.ri * (pl.rp.vecs_i / pl.rp.nvi.d));
    info->in_run = (int)pl.rp.ri;
    info->out_run = (int)pl.rp.ro;
    info->grid = pl.grid;
    info->vec = pl.vec;
    return 0;
  }
  info->path = pl.path;
  info->tile_volume = pl.path == 1 ? (int)pl.tile.vol : 0;
  info->in_run = pl.path == 1 ? pl.tile.in_run : 0;
  info->out_run = pl.path == 1 ? pl.tile.out_run : 0;
  info->grid = pl.grid;
  info->vec = pl.path == 1 ? pl.vec : 1;
  return 0;
}

int launch_permute(const void *in, void *out, int kind, int rank, const int *dims_in, const int *o2n, bool conj,
                   hipStream_t s)
{
  const int es = kind_size(kind);
  if (es == 0 || rank < 0 || rank > kMaxRank) return TALSH_INVALID_ARGS;
  if (!valid_permutation(rank, dims_in, o2n)) return TALSH_INVALID_ARGS;
  uint64_t vol = 1;
  for (int i = 0; i < rank; ++i) vol *= (uint64_t)dims_in[i];
  if (vol == 0) return 0;
  if (in == out) return TALSH_INVALID_ARGS;  // out-of-place only
  const Planned pl = planned(es, rank, dims_in, o2n, in, out, false);
  // the persistent grid and the per-thread vector slots must cover the tile
  if (pl.path == 1 && ((long)pl.ept * kTNT * pl.vec < (long)pl.tp.vol_tile || pl.grid <= 0 || pl.ept > kMaxEPT))
    return TALSH_FAILURE;
  const int cus = compute_units();
  const bool cj = conj && kind_complex(kind);
  hipEvent_t pr[2];
  prof_begin(s, kKTranspose, pr);  // timing brackets the launch only
  int e = TALSH_INVALID_ARGS;
  switch (kind) {
  case R4: e = dispatch<uint32_t, false>(pl, in, out, vol, s, cus); break;
  case R8: e = dispatch<uint2, false>(pl, in, out, vol, s, cus); break;
  case C4: e = cj ? dispatch<uint2, true>(pl, in, out, vol, s, cus) : dispatch<uint2, false>(pl, in, out, vol, s, cus); break;
  case C8: e = cj ? dispatch<uint4, true>(pl, in, out, vol, s, cus) : dispatch<uint4, false>(pl, in, out, vol, s, cus); break;
  default: break;
  }
  prof_end(s, kKTranspose, pr);
  return e;
}

bool permute_add_planned(int kind, int rank, const int *dims_in, const int *o2n)
{
  const int es = kind_size(kind);
  if (es == 0 || rank < 0 || rank > kMaxRank || !valid_permutation(rank, dims_in, o2n)) return false;
  return planned(es, rank, dims_in, o2n, nullptr, nullptr, true).path == 3;
}

int launch_permute_add(const void *in, void *out, int kind, int rank, const int *dims_in, const int *o2n, bool conj,
                       double re, double im, hipStream_t s)
{
  if (in == out || !permute_add_planned(kind, rank, dims_in, o2n)) return TALSH_INVALID_ARGS;
  const Planned pl = planned(kind_size(kind), rank, dims_in, o2n, in, out, true);
  const double f = real_factor(re, im);
  hipEvent_t pr[2];
  prof_begin(s, kKTranspose, pr);
  int e = TALSH_INVALID_ARGS;
  switch (kind) {
  case R4: e = launch_runs<uint32_t, false, R4>(pl, in, out, f, 0.0, s); break;
  case R8: e = launch_runs<uint2, false, R8>(pl, in, out, f, 0.0, s); break;
  case C4: e = conj ? launch_runs<uint2, true, C4>(pl, in, out, re, im, s) : launch_runs<uint2, false, C4>(pl, in, out, re, im, s); break;
  case C8: e = conj ? launch_runs<uint4, true, C8>(pl, in, out, re, im, s) : launch_runs<uint4, false, C8>(pl, in, out, re, im, s); break;
  default: break;
  }
  prof_end(s, kKTranspose, pr);
  return e;
}

}  // namespace xt
