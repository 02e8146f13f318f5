// Native-precision matrix products (FP64 / FP32 16x16x4 MFMAs, real and
// complex): kernels, and the launchers that the translation units of each kind
// and tile choice instantiate (k_gemm_native.hip).
//
// Every operand is addressed by two index groups (rows and k, GatherMaps): a
// matricized operand has one dimension per group, a tensor read in place up
// to kGatherMaxDims. Offsets are digit arithmetic in the kernel, so a product
// is one launch with no tables in memory.
//
// Workgroup: KG groups of 256 threads = 2x2 waves; each wave owns a (BM/2) x
// (BN/2) sub-tile of 16x16 MFMA blocks. Groups take alternate k-tiles of the
// same output tile and their sums meet in LDS at the end: with few output
// tiles that fills a CU's SIMDs with four waves each, without partials in
// memory (one 64x64 tile per CU, K 8192: FP64 54 TFLOP/s with four groups
// against 41 with one, FP32 105 against 85; the 1024^3 product 48 us in FP64
// against 55 in two K pieces, 29 against 32 in FP32).
//
// Staging, along the operand's contiguous side:
//  * row-fast: lanes along rows, row pairs when every run along the rows holds
//    whole pairs, each thread several consecutive k, which go to LDS in one
//    store;
//  * k-fast: BK / VW lanes take one row's k-values in VW-element vectors
//    (VW = 16 bytes when every run along k holds whole vectors, else 1).
// Loads need no bounds checks and no alignment beyond an element's: row and k
// indices are clamped into range (rows past the edge feed only results that
// are not stored; k-values past the end are zeroed on their way to LDS, in
// the last k-tile only), so odd extents run the same instructions as round
// ones. A 1537 x 1581 x 2491 product runs at 41 (FP64) and 75 (FP32) TFLOP/s,
// with the lane-masked loads this replaces at 33 and 38.
//
// What bounds the loop, the MFMAs aside, is the other instructions a wave
// issues between them: with 45 vector instructions of address arithmetic per
// 16 FP64 MFMAs a 64x64 tile per CU ran at 35 TFLOP/s, without them at 41; a
// branch per loaded k-value cost as much. So, wherever a k-tile starts at one
// offset for all lanes (mode kVec, kUni), the tile's start is a scalar that
// steps by carries, the lanes' offsets are loop invariant, and one compare per
// k-tile decides what the last tile needs. 128x128 tiles reach 64 (FP64) and
// 127 (FP32) TFLOP/s, 82% of the matrix peak, and C8 64x64 tiles 64. Everywhere
// else (modes kTab, kTabLong) one lane per k-value works out its offsets for 64
// k-values ahead into LDS, and the loads add what they read there to their
// row's offset.
// With a digit walk per lane and k-value instead, kernel times were, in us:
// R8 ranks 10, extents 4 (groups of five dimensions) 116 against 72, extents 3
// 106 against 22; ranks 8, extents 4 53 against 21; R4 the same three 107, 98
// and 62 against 52, 20 and 16; R4 24^4 29.6 against 23; R8 1537 x 1581 x
// 2491 (a call) 300 against 286; C4 with runs of a few elements and a deep K 55
// against 60. (32-bit offsets in the tables, and reading them ahead of the
// stores to LDS, changed nothing beyond 1%.)
//
// Operand tiles sit in LDS with k fastest ([row][k], padded rows). Inside a
// 16-deep k slice, lane group g = lane/16 feeds k = 4g+s at MFMA step s, so a
// lane's four steps use four consecutive k and its fragment for the whole
// slice is one contiguous LDS read (summation order over k is immaterial).
//
// Pipeline: at k-tile t the registers holding tile t+1 go to the other LDS
// buffer first, the loads of tile t+2 follow into the same registers, then
// tile t is multiplied.
#pragma once

#include <algorithm>
#include <type_traits>

#include "bf16x3.hpp"
#include "kernels.hpp"

namespace xt {

struct DevDivisor { uint32_t d, m, s; };
// An index group of up to N dimensions.
template <int N>
struct DevGroup {
  int nd;
  DevDivisor div[N - 1];   // of every dimension but the last, whose digit is the quotient; 1 beyond those
  int64_t str[N];          // in the long form, str[N - 1] is the last dimension's
};

// Kernel arguments. Groups of up to kSmallDims dimensions go in the short form
// (0.6 KB in all): with 2 KB of arguments every launch took about 1 us longer
// (calls by offset tables: R8 8^4 40.4 against 38.3 us, R8 1537 x 1581 x 2491
// 291 against 286).
constexpr int kSmallDims = 4;
template <int N>
struct GemmParams {
  const void *a;
  const void *b;
  void *c;
  int64_t m, n, k;
  int64_t a_line, b_line;    // row stride of an operand whose rows are one dimension, else 0
  int64_t k0;                // this launch covers k-values [k0, k), at most kMaxDepth
  double alpha_re, alpha_im;
  int beta_zero;
  int conj_a, conj_b;
  int tiles_m, tiles_n;
  // split K: tiles [0, full) run over all of K, every later tile in `parts`
  // pieces of kchunk k-values whose raw sums go to part (piece z at z *
  // zstride elements); full == 0: the tiles' blocks are stored unpadded
  void *part;
  int full, parts;
  int64_t kchunk, zstride;
  DevGroup<N> a_row, a_k, b_row, b_k, c_row, c_col;
};

constexpr int64_t kMaxDepth = 1ll << 30;

// How an operand pair walks along k.
enum GemmMode {
  kVec,   // a k-tile starts at one offset for all lanes; k-fast operands load 16-byte vectors, row-fast ones
          // row pairs (whole vectors everywhere: even rows and k-values in eights there)
  kUni,   // the same, element loads
  kTab,   // offsets from tables in LDS: runs along k of any length, 64-bit offsets
  kTabLong  // the same with arguments in the long form, for groups of up to kGatherMaxDims dimensions
};
constexpr int group_dims(GemmMode mode) { return mode == kTabLong ? kGatherMaxDims : kSmallDims; }
constexpr bool tabled(GemmMode mode) { return mode == kTab || mode == kTabLong; }

// A product ready to launch.
struct Product {
  GemmParams<kGatherMaxDims> p{};
  bool a_kfast = false, b_kfast = false;
  GemmMode mode = kTab;
};

// Output tiles of the native-precision kernels: rows x columns, the k-depth of
// one LDS stage (128 bytes of a row; complex kinds hold two planes) and the
// k-groups of a workgroup.
struct TileShape { int bm, bn, bk, groups; };
constexpr TileShape tile_shape(int kind, int tile)
{
  const int bk = kind == R4 ? 32 : 16;
  if (kind == C8 || kind == C4) return {64, 64, bk, tile == 1 ? 2 : 1};
  return tile == 2 ? TileShape{64, 64, bk, 1} : tile == 1 ? TileShape{64, 64, bk, 4} : TileShape{128, 128, bk, 1};
}

// One translation unit (k_gemm_native.hip) for each kind and tile choice.
template <int KIND, int TILE>
int launch_native(const Product &q, hipStream_t s);

// The output-tile order: first gather the workgroups that the dispatcher
// places on one XCD (round-robin over 8) into a contiguous range, then walk
// that range in column groups of G M-tiles so neighbouring workgroups share B
// panels (and A panels within a group) in their XCD's L2.
template <int G = 8>
__device__ __forceinline__ void tile_walk(int t, int tiles_m, int tiles_n, int &tm, int &tn)
{
  const int per_group = G * tiles_n;
  const int group = t / per_group;
  const int first_m = group * G;
  const int gm = min(tiles_m - first_m, G);
  const int r = t - group * per_group;
  tm = first_m + r % gm;
  tn = r / gm;
}
__device__ __forceinline__ int xcd_order(int b, int nb) { return (nb % 8) == 0 ? (b % 8) * (nb / 8) + b / 8 : b; }

#ifdef XT_GEMM_KERNELS
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Acc;
template <>
struct Acc<double> { typedef d4 type; };
template <>
struct Acc<float> { typedef f4 type; };

__device__ __forceinline__ d4 mfma(double a, double b, d4 c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma(float a, float b, f4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The kernels read their arguments through the kernel-argument segment (the
// one argument starts it): a by-value struct whose arrays are indexed at run
// time may be copied to scratch memory, and in some instantiations was.
template <int N>
using ArgParams = const __attribute__((address_space(4))) GemmParams<N>;
template <int N>
using ArgGroup = const __attribute__((address_space(4))) DevGroup<N>;
template <int N>
__device__ __forceinline__ ArgParams<N> &gemm_args_of_kernel()
{
  return *(ArgParams<N> *)__builtin_amdgcn_kernarg_segment_ptr();
}

template <typename D>
__device__ __forceinline__ uint32_t gg_div(uint32_t x, const D &f) { return (__umulhi(x, f.m) + x) >> f.s; }

// Element offset of index x of a group. The long form takes three dimensions at
// a time: a loop over single ones waits for the arguments of each in turn. The
// short form's groups mostly have two (R8 32^4: 147 us against 150).
template <int N>
__device__ __forceinline__ int64_t group_off(ArgGroup<N> &g, int64_t x)
{
  constexpr int STEP = N > kSmallDims ? 3 : 1;
  if (g.nd <= 1) return x * g.str[0];
  uint32_t r = (uint32_t)x;
  int64_t o = 0;
  for (int j = 0; j + 1 < g.nd; j += STEP) {
#pragma unroll
    for (int i = j; i < j + STEP; ++i) {
      const uint32_t q = gg_div(r, g.div[i]);
      o += (int64_t)(r - q * g.div[i].d) * g.str[i];
      r = q;
    }
  }
  return o + (int64_t)r * g.str[N > kSmallDims ? N - 1 : g.nd - 1];
}

// A position along a k group of up to three dimensions, the same for all lanes,
// advanced STEP k-values at a time by carries (a few scalar additions; no
// division, no read of the arguments). Offsets in bytes.
template <int STEP, int ES, int N>
struct KWalk {
  int64_t at, step, s0, fix0, fix1;  // offset, its change per STEP and per k, its corrections on carries
  uint32_t c0, c1, b0, b1, d0, d1;
  __device__ __forceinline__ void init(ArgGroup<N> &g, int64_t x0)
  {
    const uint32_t x = (uint32_t)x0;
    s0 = g.str[0] * ES;
    const int64_t s1 = g.str[1] * ES, s2 = g.str[2] * ES;
    d0 = d1 = 0x7fffffffu;
    c0 = c1 = b0 = b1 = 0;
    step = STEP * s0;
    if (g.nd > 1) {
      const uint32_t q0 = gg_div(x, g.div[0]);
      d0 = g.div[0].d;
      c0 = x - q0 * d0;
      const uint32_t bq = STEP / d0;
      b0 = STEP - bq * d0;
      if (g.nd > 2) d1 = g.div[1].d;
      c1 = g.nd > 2 ? q0 - gg_div(q0, g.div[1]) * d1 : q0;
      b1 = bq % d1;
      step = b0 * s0 + b1 * s1 + (int64_t)(bq / d1) * s2;
    }
    fix0 = s1 - d0 * s0;
    fix1 = s2 - d1 * s1;
    at = group_off(g, x0) * ES;
  }
  __device__ __forceinline__ void advance()
  {
    at += step;
    c0 += b0;
    c1 += b1;
    if (c0 >= d0 || c1 >= d1) {
      const bool k0 = c0 >= d0;
      c0 -= k0 ? d0 : 0u;
      at += k0 ? fix0 : 0;
      c1 += k0 ? 1u : 0u;
      const bool k1 = c1 >= d1;
      c1 -= k1 ? d1 : 0u;
      at += k1 ? fix1 : 0;
    }
  }
};

__device__ __forceinline__ double flip_sign(double x, uint32_t m)
{
  return __hiloint2double(__double2hiint(x) ^ (int)m, __double2loint(x));
}
__device__ __forceinline__ float flip_sign(float x, uint32_t m) { return __uint_as_float(__float_as_uint(x) ^ m); }

// Staging of one operand tile (BX rows x BK k-values) by the 256 threads of a
// group, one k-tile in KG.
template <typename T, bool CPLX, bool KF, int BX, int BK, int KG, GemmMode MODE>
struct Staging {
  static constexpr bool TAB = tabled(MODE);
  typedef typename std::conditional<TAB, uint64_t, uint32_t>::type OffT;
  static constexpr int N = group_dims(MODE);
  static constexpr bool VEC = MODE == kVec && !CPLX;
  static constexpr int NP = CPLX ? 2 : 1;
  static constexpr int KP = BK + (sizeof(T) == 4 ? 4 : 2);  // padded k extent of an LDS row
  // a thread loads W contiguous elements at a time: VW along k (k-fast) or RV
  // along rows (row-fast, vector form)
  static constexpr int VW = KF && VEC ? 16 / (int)sizeof(T) : 1;
  static constexpr int RV = !KF && VEC ? 2 : 1;
  static constexpr int W = VW * RV;
  // k-fast: LR lanes per row, NR rows per thread; row-fast: LR lanes along the
  // rows (64 in the element form, so that a wave's loads share each k), NR
  // row groups, KV consecutive k per thread
  static constexpr int LR = KF ? BK / VW : RV == 1 ? 64 : BX / RV;
  static constexpr int RS = KF ? 256 / LR : LR * RV;        // rows between a thread's rows
  static constexpr int NR = BX / RS;
  static constexpr int KV = KF ? 1 : BK * LR / 256;
  static constexpr int NE = NR * KV * W;
  static constexpr int ES = (int)sizeof(T) * NP;
  static constexpr int STEP = BK * KG;
  typedef T LdsRow[KP];
  OffT ro[NR];
  int row, kk;
  KWalk<STEP, ES, N> walk;  // at the start of a k-tile

  __device__ __forceinline__ void place(int tid, int wave)
  {
    if (KF) { kk = (tid % LR) * VW; row = tid / LR; }
    else { kk = (RV == 1 ? wave : tid / LR) * KV; row = tid % LR * RV; }
  }
  __device__ __forceinline__ void init(ArgGroup<N> &g, ArgGroup<N> &gk, int64_t line, int64_t r0, int64_t rows,
                                       int64_t kbeg, int64_t k0, int64_t kend, int tid, int wave)
  {
    place(tid, wave);
    const int64_t last = rows - RV;
    walk.init(gk, k0 < kend ? k0 : kbeg);
    // lanes hold offsets from the tile's first row where rows are one
    // dimension (line: its stride, else 0), so that 32 bits do for operands of
    // any size
    const int64_t first = r0 * line;
    walk.at += first * ES;
    // (element-form row-fast loads add their k offset as a scalar)
    const OffT lane_k = KF || RV > 1 ? (OffT)(kk * walk.s0) : OffT(0);
#pragma unroll
    for (int i = 0; i < NR; ++i) ro[i] = (OffT)((group_off(g, min(r0 + row + i * RS, last)) - first) * ES) + lane_k;
  }
  // TAB: rows from the tile's table of row offsets (in bytes; rows past the
  // edge repeat the last)
  __device__ __forceinline__ void init_tab(const uint64_t *rows, int tid, int wave)
  {
    place(tid, wave);
#pragma unroll
    for (int i = 0; i < NR; ++i) ro[i] = rows[row + i * RS];
  }
  // Loads the k-tile whose offsets start at kt (in bytes; k-values past the
  // end repeat the last), elements as load() does.
  __device__ __forceinline__ void load_tab(const char *base, const uint64_t *kt, T (&r)[NE * NP]) const
  {
    constexpr int J = KF ? 1 : KV;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const char *p = base + kt[kk + j];
#pragma unroll
      for (int i = 0; i < NR; ++i) load_one(p + ro[i], &r[(i * J + j) * W * NP]);
    }
  }
  // In the last k-tile, `left` k-values deep, lanes past the end read the
  // tile's first k-values (a lane's KV k-values lie on one side of the end)
  __device__ __forceinline__ void clamp_k(int left)
  {
    if (KF || RV > 1) {
      const OffT back = kk < left ? OffT(0) : (OffT)(kk * walk.s0);
#pragma unroll
      for (int i = 0; i < NR; ++i) ro[i] -= back;
    }
  }
  __device__ __forceinline__ void load_one(const char *p, T *r) const
  {
    constexpr int N = W * NP;
    typedef T TV __attribute__((ext_vector_type(N), aligned(sizeof(T))));
    if constexpr (N == 1) {
      r[0] = *reinterpret_cast<const T *>(p);
    } else {
      const TV v = *reinterpret_cast<const TV *>(p);
#pragma unroll
      for (int e = 0; e < N; ++e) r[e] = v[e];
    }
  }
  // Loads the k-tile the walk stands at; left: k-values from the tile's start
  // to the end. r[e * NP + q]: element e, component q; k-fast e = row * VW +
  // k, row-fast e = (row group * KV + k) * RV + row.
  __device__ __forceinline__ void load(const char *base, int left, T (&r)[NE * NP]) const
  {
    if constexpr (KF) {
      const char *p = base + walk.at;
#pragma unroll
      for (int i = 0; i < NR; ++i) load_one(p + ro[i], &r[i * W * NP]);
    } else {
#pragma unroll
      for (int j = 0; j < KV; ++j) {
        const int x = RV > 1 ? j : kk + j;
        const char *p = base + (walk.at + (x < left ? x : 0) * walk.s0);
#pragma unroll
        for (int i = 0; i < NR; ++i) load_one(p + ro[i], &r[(i * KV + j) * W * NP]);
      }
    }
  }
  // Zeroes what a k-tile of `left` k-values does not hold.
  __device__ __forceinline__ void zero_past(T (&r)[NE * NP], int left) const
  {
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const bool ok = kk + (KF ? e % VW : e / RV % KV) < left;
#pragma unroll
      for (int q = 0; q < NP; ++q) r[e * NP + q] = ok ? r[e * NP + q] : T(0);
    }
  }
  __device__ __forceinline__ void to_lds(LdsRow *S, const T (&r)[NE * NP], uint32_t conj) const
  {
    constexpr int L = KF ? VW : KV;                       // consecutive k of one row
    constexpr int SV = L * (int)sizeof(T) >= 16 ? 16 / (int)sizeof(T) : L;
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int v = 0; v < RV; ++v) {
          T *dst = &S[q * BX + row + i * RS + v][kk];
#pragma unroll
          for (int e = 0; e < L; e += SV) {
            typedef T TS __attribute__((ext_vector_type(SV)));
            T x[SV];
#pragma unroll
            for (int u = 0; u < SV; ++u) {
              x[u] = r[((i * L + e + u) * RV + v) * NP + q];
              if (q) x[u] = flip_sign(x[u], conj);
            }
            if constexpr (SV == 1) {
              dst[e] = x[0];
            } else {
              TS y;
#pragma unroll
              for (int u = 0; u < SV; ++u) y[u] = x[u];
              *reinterpret_cast<TS *>(dst + e) = y;
            }
          }
        }
  }
};

// C = alpha * acc + beta * C (beta 0 or 1) for the FM x FN blocks of a wave;
// get(i, j, r, q) is component q of the accumulator's element r, rows(x) and
// cols(x) the offsets of row and column x (clamped into C).
// Per 16-row block the offsets (-1: outside C), then every C load of the
// block at once (clamped addresses, no lane-masked branches), one wait, then
// the stores; a load-add-store per element would wait for each load in turn
// behind the stores already issued.
template <typename T, bool CPLX, int FM, int FN, int N, typename Get, typename Rows, typename Cols>
__device__ __forceinline__ void store_c(ArgParams<N> &p, int64_t m0, int64_t n0, int lane, Get get, Rows rows, Cols cols)
{
  constexpr int NP = CPLX ? 2 : 1;
  T *C = static_cast<T *>(p.c);
  const int fr = lane & 15, fk = (lane >> 4) & 3;
  const T ar = (T)p.alpha_re, ai = (T)p.alpha_im;
  int64_t gcol[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t col = n0 + j * 16 + fr;
    gcol[j] = col < p.n ? cols(col) : -1;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    int64_t off[FN][4];
    T cv[FN][4][NP];
    // accumulator layout: FP32 16x16x4 keeps rows 4*(lane/16)+r in a lane,
    // FP64 16x16x4 keeps rows lane/16 + 4*r
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = m0 + i * 16 + (sizeof(T) == 8 ? fk + 4 * r : fk * 4 + r);
      const int64_t grow = rows(min(row, p.m - 1));
#pragma unroll
      for (int j = 0; j < FN; ++j) off[j][r] = (row < p.m && gcol[j] >= 0) ? grow + gcol[j] : -1;
    }
    if (!p.beta_zero) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int q = 0; q < NP; ++q) cv[j][r][q] = C[NP * (off[j][r] < 0 ? 0 : off[j][r]) + q];
      wait_all_vmem();  // on every lane, before the lane-masked stores
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int q = 0; q < NP; ++q) cv[j][r][q] = T(0);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (off[j][r] < 0) continue;
        if (CPLX) {
          const T xr = get(i, j, r, 0), xi = get(i, j, r, 1);
          C[2 * off[j][r]] = ar * xr - ai * xi + cv[j][r][0];
          C[2 * off[j][r] + 1] = ar * xi + ai * xr + cv[j][r][1 % NP];
        } else {
          C[off[j][r]] = ar * get(i, j, r, 0) + cv[j][r][0];
        }
      }
  }
}

// Place of a split tile's element (row r, column c of the tile) in a piece of
// the partials: row-major, tiles padded (full > 0) or their stored part only.
template <int BM, int BN>
struct PartLayout {
  int64_t base;
  int cols;
  template <int N>
  __device__ __forceinline__ PartLayout(ArgParams<N> &p, int tile, int64_t m0, int64_t n0)
  {
    if (p.full > 0) {
      base = (int64_t)(tile - p.full) * (BM * BN);
      cols = BN;
    } else {
      cols = (int)min((int64_t)BN, p.n - n0);
      base = n0 * p.m + m0 * cols;
    }
  }
};

template <typename T, bool CPLX, bool AK, bool BKF, int BM, int BN, int BK, int KG, int OCC, GemmMode MODE>
__global__ __launch_bounds__(256 * KG, OCC) void k_gemm_mfma(const GemmParams<group_dims(MODE)>)
{
  ArgParams<group_dims(MODE)> &p = gemm_args_of_kernel<group_dims(MODE)>();
  constexpr int NP = CPLX ? 2 : 1;                 // LDS planes (re, im)
  constexpr int FM = BM / 32, FN = BN / 32;        // MFMA blocks per wave along m / n
  constexpr int HS = 16 / (int)sizeof(T);          // k-steps per 16-byte fragment read
  typedef Staging<T, CPLX, AK, BM, BK, KG, MODE> SA;
  typedef Staging<T, CPLX, BKF, BN, BK, KG, MODE> SB;
  constexpr int KP = SA::KP;
  typedef typename Acc<T>::type AccT;
  typedef T LdsRow[KP];
  __shared__ __align__(16) T As[KG][2][NP * BM][KP];
  __shared__ __align__(16) T Bs[KG][2][NP * BN][KP];
  // TAB: offsets in bytes of the tile's rows of A and B and of two chunks of
  // 64 k-values per k-group, in elements of its rows and columns of C.
  constexpr bool TAB = tabled(MODE);
  constexpr int TN = TAB ? 64 : 1, TPC = 64 / BK;  // k-tiles per chunk
  __shared__ uint64_t t_ab[TAB ? BM + BN : 1], t_k[TAB ? KG : 1][2][2][TN];
  __shared__ int64_t t_c[TAB ? BM + BN : 1];

  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  int tile, z = 0;
  int64_t kbeg = p.k0, kend = p.k;
  const bool split = (int)blockIdx.x >= p.full;
  if (!split) {
    tile = xcd_order(blockIdx.x, p.full);
  } else {
    const int s = blockIdx.x - p.full;
    tile = p.full + s / p.parts;
    z = s % p.parts;
    kbeg += z * p.kchunk;
    kend = min(p.k, kbeg + p.kchunk);
  }
  int tm, tn;
  tile_walk(tile, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
  const char *A = static_cast<const char *>(p.a), *B = static_cast<const char *>(p.b);
  const uint32_t ca = p.conj_a ? 0x80000000u : 0u, cb = p.conj_b ? 0x80000000u : 0u;
  LdsRow *la = As[grp][0], *lb = Bs[grp][0];

  AccT acc[NP][FM][FN];
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[q][i][j] = AccT{0, 0, 0, 0};

  if constexpr (TAB) {
    for (int x = threadIdx.x; x < 2 * (BM + BN); x += 256 * KG) {
      const int y = x % (BM + BN);
      const bool row = y < BM;
      const int64_t at = row ? min(m0 + y, p.m - 1) : min(n0 + y - BM, p.n - 1);
      if (x < BM + BN) t_ab[y] = (uint64_t)((row ? group_off(p.a_row, at) : group_off(p.b_row, at)) * SA::ES);
      else t_c[y] = row ? group_off(p.c_row, at) : group_off(p.c_col, at);
    }
    __syncthreads();
  }
  const int fr = lane & 15, fg = (lane >> 4) * 4;
  const int nt = (int)((kend - kbeg + BK * KG - 1) / (BK * KG));  // steps: k-tiles per group
  if (nt > 0) {
    SA sa;
    SB sb;
    const int64_t k0 = kbeg + grp * BK;
    constexpr int ES = SA::ES;
    auto k_table = [&](int c) {  // chunk c of this k-group: wave 0 for A, wave 1 for B
      if (wave > 1) return;
      const int64_t x = min(k0 + (int64_t)(c * TPC + lane / BK) * (BK * KG) + lane % BK, kend - 1);
      const int64_t o = wave == 0 ? group_off(p.a_k, x) : group_off(p.b_k, x);
      t_k[TAB ? grp : 0][wave][c & 1][TAB ? lane : 0] = (uint64_t)(o * ES);
    };
    if constexpr (TAB) {
      k_table(0);
      __syncthreads();
      sa.init_tab(t_ab, tid, wave);
      sb.init_tab(t_ab + BM, tid, wave);
    } else {
      sa.init(p.a_row, p.a_k, p.a_line, m0, p.m, kbeg, k0, kend, tid, wave);
      sb.init(p.b_row, p.b_k, p.b_line, n0, p.n, kbeg, k0, kend, tid, wave);
    }
    int lt = 0;  // TAB: k-tiles loaded
    // k-values from the next k-tile's start to the end: of the tile to load
    // (walks stay at the last tile), of the tile to store
    int left_s = (int)(kend - k0), left_l = left_s <= 0 ? (int)min(kend - kbeg, (int64_t)BK) : left_s;
    if (!TAB && left_l < BK) {
      sa.clamp_k(left_l);
      sb.clamp_k(left_l);
    }
    T ra[SA::NE * NP], rb[SB::NE * NP];
    auto load = [&]() {  // the next k-tile
      if constexpr (TAB) {
        const int c = lt / TPC;
        // the chunk after this one, over the one before (the last read of
        // which lies a barrier back)
        if (lt % TPC == 0) k_table(c + 1);
        sa.load_tab(A, &t_k[grp][0][c & 1][lt % TPC * BK], ra);
        sb.load_tab(B, &t_k[grp][1][c & 1][lt % TPC * BK], rb);
        ++lt;
        return;
      }
      sa.load(A, left_l, ra);
      sb.load(B, left_l, rb);
      if (left_l > BK * KG) {
        left_l -= BK * KG;
        sa.walk.advance();
        sb.walk.advance();
        if (left_l < BK) {
          sa.clamp_k(left_l);
          sb.clamp_k(left_l);
        }
      }
    };
    auto store = [&](int buf) {  // the loaded k-tile into LDS buffer buf
      if (left_s < BK) {  // the last, partial k-tile, or none left for this group
        sa.zero_past(ra, left_s);
        sb.zero_past(rb, left_s);
      }
      sa.to_lds(la + buf * NP * BM, ra, ca);
      sb.to_lds(lb + buf * NP * BN, rb, cb);
      left_s -= BK * KG;
    };
    auto compute = [&](int buf) {
      const LdsRow *xa = la + buf * NP * BM + wm + fr, *xb = lb + buf * NP * BN + wn + fr;
#pragma unroll
      for (int ks = 0; ks < BK; ks += 16)
#pragma unroll
        for (int h = 0; h < 4; h += HS) {
          typedef T TH __attribute__((ext_vector_type(HS)));
          TH fa[NP][FM], fb[NP][FN];
#pragma unroll
          for (int q = 0; q < NP; ++q) {
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[q][i] = *reinterpret_cast<const TH *>(&xa[q * BM + i * 16][ks + fg + h]);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[q][j] = *reinterpret_cast<const TH *>(&xb[q * BN + j * 16][ks + fg + h]);
          }
#pragma unroll
          for (int st = 0; st < HS; ++st)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
              for (int j = 0; j < FN; ++j) {
                if (CPLX) {
                  // (ar + i ai)(br + i bi) = (ar br - ai bi) + i (ar bi + ai br)
                  const T a0 = fa[0][i][st], a1 = fa[1 % NP][i][st], b0 = fb[0][j][st], b1 = fb[1 % NP][j][st];
                  acc[0][i][j] = mfma(a0, b0, acc[0][i][j]);
                  acc[1 % NP][i][j] = mfma(a0, b1, acc[1 % NP][i][j]);
                  acc[0][i][j] = mfma(-a1, b1, acc[0][i][j]);
                  acc[1 % NP][i][j] = mfma(a1, b0, acc[1 % NP][i][j]);
                } else {
                  acc[0][i][j] = mfma(fa[0][i][st], fb[0][j][st], acc[0][i][j]);
                }
              }
        }
    };
    load();
    store(0);
    load();
    __syncthreads();
    // (past the last k-tile, stores and loads go on harmlessly: into the
    // buffer that is not read any more, from addresses in range)
    for (int t = 0, buf = 0; t < nt; ++t, buf ^= 1) {
      store(buf ^ 1);
      load();
      compute(buf);
      __syncthreads();
    }
  }

  // blocks that this wave finishes: all of its own with one group, else a
  // share of the four (OM x ON of them from block (oi, oj) on) summed over the
  // groups through LDS
  constexpr int OM = KG == 1 ? FM : 1, ON = KG == 4 ? 1 : FN;
  static_assert(KG == 1 || (FM == 2 && FN == 2 && (KG == 2 || KG == 4)), "block shares of the groups");
  const int oi = KG == 1 ? 0 : KG == 2 ? grp : grp >> 1, oj = KG == 4 ? grp & 1 : 0;
  if constexpr (KG > 1) {
    constexpr int NB = FM * FN * NP * 4;
    static_assert(sizeof(As) >= sizeof(T) * KG * 4 * NB * 64 / 2 && sizeof(Bs) >= sizeof(T) * KG * 4 * NB * 64 / 2,
                  "the sums fit the operand buffers");
    // value v of a lane: the first half in As, the second in Bs
    auto slot = [&](int g, int v) -> T * {
      T *h = v < NB / 2 ? &As[0][0][0][0] : &Bs[0][0][0][0];
      return h + ((g * 4 + wave) * (NB / 2) + v % (NB / 2)) * 64 + lane;
    };
    auto at = [&](int q, int i, int j, int r) { return ((i * FN + j) * NP + q) * 4 + r; };
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) *slot(grp, at(q, i, j, r)) = acc[q][i][j][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int j = 0; j < ON; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T s = *slot(0, at(q, oi, oj + j, r));
#pragma unroll
          for (int g = 1; g < KG; ++g) s += *slot(g, at(q, oi, oj + j, r));
          acc[q][0][j][r] = s;
        }
  }
  const int64_t mw = m0 + wm + oi * 16, nw = n0 + wn + oj * 16;
  if (!split) {
    store_c<T, CPLX, OM, ON>(p, mw, nw, lane, [&](int i, int j, int r, int q) { return acc[q][i][j][r]; },
                             [&](int64_t x) { return TAB ? t_c[x - m0] : group_off(p.c_row, x); },
                             [&](int64_t x) { return TAB ? t_c[BM + (x - n0)] : group_off(p.c_col, x); });
    return;
  }
  const PartLayout<BM, BN> pl(p, tile, m0, n0);
  T *P = static_cast<T *>(p.part) + NP * (z * p.zstride + pl.base);
  const int fk = (lane >> 4) & 3;
#pragma unroll
  for (int i = 0; i < OM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wm + (oi + i) * 16 + (sizeof(T) == 8 ? fk + 4 * r : fk * 4 + r);
#pragma unroll
      for (int j = 0; j < ON; ++j) {
        const int col = wn + (oj + j) * 16 + fr;
        if (m0 + row < p.m && n0 + col < p.n) {
#pragma unroll
          for (int q = 0; q < NP; ++q) P[NP * (row * pl.cols + col) + q] = acc[q][i][j][r];
        }
      }
    }
}

// C = alpha * sum of the pieces (+ C) of the split tiles, summed in FP64. One
// workgroup per 16 rows of a tile, lanes along the columns (which hold C's
// stride-1 index whenever the product was free to choose).
template <typename T, bool CPLX, int BM, int BN, int N>
__global__ __launch_bounds__(256) void k_splitk_sum(const GemmParams<N>)
{
  ArgParams<N> &p = gemm_args_of_kernel<N>();
  constexpr int NP = CPLX ? 2 : 1, RB = BM / 16;
  const int tile = p.full + blockIdx.x / RB;
  int tm, tn;
  tile_walk(tile, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const PartLayout<BM, BN> pl(p, tile, m0, n0);
  const T *P = static_cast<const T *>(p.part) + NP * pl.base;
  T *C = static_cast<T *>(p.c);
  const int c = threadIdx.x % BN;
  const int64_t col = n0 + c;
  if (col >= p.n) return;
  const int64_t gcol = group_off(p.c_col, col);
#pragma unroll
  for (int e = 0; e < 16 * BN / 256; ++e) {
    const int r = (blockIdx.x % RB) * 16 + threadIdx.x / BN + e * (256 / BN);
    if (m0 + r >= p.m) break;
    const T *src = P + NP * (r * pl.cols + c);
    double s[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) s[q] = 0.0;
#pragma unroll 4
    for (int z = 0; z < p.parts; ++z)
#pragma unroll
      for (int q = 0; q < NP; ++q) s[q] += (double)src[NP * z * p.zstride + q];
    T *d = C + NP * (group_off(p.c_row, m0 + r) + gcol);
    if (CPLX) {
      double vr = p.alpha_re * s[0] - p.alpha_im * s[1 % NP], vi = p.alpha_re * s[1 % NP] + p.alpha_im * s[0];
      if (!p.beta_zero) { vr += (double)d[0]; vi += (double)d[1 % NP]; }
      d[0] = (T)vr;
      d[1 % NP] = (T)vi;
    } else {
      double v = p.alpha_re * s[0];
      if (!p.beta_zero) v += (double)d[0];
      d[0] = (T)v;
    }
  }
}

// The arguments with groups of N dimensions (the caller has checked they fit).
template <int N>
GemmParams<N> shortened(const GemmParams<kGatherMaxDims> &f)
{
  if constexpr (N == kGatherMaxDims) {
    return f;
  } else {
    GemmParams<N> p{};
    p.a = f.a; p.b = f.b; p.c = f.c;
    p.m = f.m; p.n = f.n; p.k = f.k; p.k0 = f.k0;
    p.a_line = f.a_line; p.b_line = f.b_line;
    p.alpha_re = f.alpha_re; p.alpha_im = f.alpha_im;
    p.beta_zero = f.beta_zero;
    p.conj_a = f.conj_a; p.conj_b = f.conj_b;
    p.tiles_m = f.tiles_m; p.tiles_n = f.tiles_n;
    p.part = f.part;
    p.full = f.full; p.parts = f.parts;
    p.kchunk = f.kchunk; p.zstride = f.zstride;
    auto group = [](DevGroup<N> &d, const DevGroup<kGatherMaxDims> &g) {
      d.nd = g.nd;
      for (int j = 0; j < N; ++j) d.str[j] = g.str[j];
      for (int j = 0; j + 1 < N; ++j) d.div[j] = g.div[j];
    };
    group(p.a_row, f.a_row); group(p.a_k, f.a_k);
    group(p.b_row, f.b_row); group(p.b_k, f.b_k);
    group(p.c_row, f.c_row); group(p.c_col, f.c_col);
    return p;
  }
}

template <typename T, bool CPLX, bool AK, bool BKF, int BM, int BN, int BK, int KG, int OCC, GemmMode MODE>
int launch_tile(const Product &q, hipStream_t s)
{
  constexpr int N = group_dims(MODE);
  const GemmParams<N> p = shortened<N>(q.p);
  const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
  const int64_t blocks = p.full + (tiles - p.full) * p.parts;
  hipLaunchKernelGGL((k_gemm_mfma<T, CPLX, AK, BKF, BM, BN, BK, KG, OCC, MODE>), dim3((unsigned)blocks),
                     dim3(256 * KG), 0, s, p);
  if (tiles > p.full)
    hipLaunchKernelGGL((k_splitk_sum<T, CPLX, BM, BN, N>), dim3((unsigned)((tiles - p.full) * (BM / 16))), dim3(256), 0, s,
                       p);
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

template <typename T, bool CPLX, int BM, int BN, int BK, int KG, int OCC, GemmMode MODE>
int launch_orient(const Product &q, hipStream_t s)
{
  if (q.a_kfast && q.b_kfast) return launch_tile<T, CPLX, true, true, BM, BN, BK, KG, OCC, MODE>(q, s);
  if (q.a_kfast) return launch_tile<T, CPLX, true, false, BM, BN, BK, KG, OCC, MODE>(q, s);
  if (q.b_kfast) return launch_tile<T, CPLX, false, true, BM, BN, BK, KG, OCC, MODE>(q, s);
  return launch_tile<T, CPLX, false, false, BM, BN, BK, KG, OCC, MODE>(q, s);
}

template <typename T, bool CPLX, int BM, int BN, int BK, int KG, int OCC>
int launch_modes(const Product &q, hipStream_t s)
{
  if constexpr (!CPLX) {
    if (q.mode == kVec) return launch_orient<T, CPLX, BM, BN, BK, KG, OCC, kVec>(q, s);
  }
  if (q.mode == kTab) return launch_orient<T, CPLX, BM, BN, BK, KG, OCC, kTab>(q, s);
  if (q.mode == kTabLong) return launch_orient<T, CPLX, BM, BN, BK, KG, OCC, kTabLong>(q, s);
  return launch_orient<T, CPLX, BM, BN, BK, KG, OCC, kUni>(q, s);
}

}  // namespace
#endif  // XT_GEMM_KERNELS

}  // namespace xt
