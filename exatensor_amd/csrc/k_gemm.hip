// Matrix-core GEMMs for gfx950: the compute step of a tensor contraction
// (D(ll,lr) += alpha * L(lc,ll)^T * R(lc,lr) after matricization).
//
// Replaces the reference's cuBLAS calls and gpu_matrix_multiply_tn__
// (TALSH/tensor_algebra_gpu_nvidia.cu:6852-7056, :2263-2312) with in-house
// kernels:
//   R8 / C8 : v_mfma_f64_16x16x4_f64, FP64 accumulation;
//   R4 / C4 : v_mfma_f32_16x16x4_f32, FP32 accumulation ("native FP32");
//   R4 fast : three-way BF16 split on v_mfma_f32_16x16x32_bf16 (six partial
//             products per pair, two-level FP32 accumulation per K chunk,
//             FP64 sum over the chunks) -- see k_gemm_bf16x3 below.
// Operands: A stored k x m with k fastest ("T") or m x k with m fastest ("N");
// B stored k x n with k fastest ("N") or n x k with n fastest ("T");
// C is m x n column-major. Complex operands are interleaved (re, im) and are
// split into real/imaginary LDS planes while staging.
#include <algorithm>
#include <type_traits>

#include "gemm_native.hpp"

namespace xt {
namespace {

// ---------------------------------------------------------------------------
// Three-way BF16 split (helpers in bf16x3.hpp): six bf16 products per k-step
// on the bf16 MFMAs, FP32 accumulation folded every 256 k-values into a
// second FP32 sum (two-level summation), split K over gridDim.y chunks of at
// most kB3Chunk k-values whose partial tiles k_splitk_reduce sums in FP64.
//
// Operand layout ("tile-blocked"): the split pass stores each operand as three
// bf16 planes cut into blocks of RB rows x KB k-values, 1 KB each, laid out
// exactly as the matrix kernel's LDS stage holds them (rows of KB values,
// 16-byte chunks swizzled against LDS bank conflicts). One wave-wide
// global_load_lds_dwordx4 then moves one whole block, 1 KB contiguous in
// memory, straight into LDS. (Row-major planes moved 32 or 64 bytes per row
// per stage: partial 128-byte lines, and the memory path, not the MFMAs, set
// the kernel time.) Blocks of one row band follow each other along k; row
// bands are blk = RB * k_pad elements apart.
constexpr int kB3Chunk = 8192;
constexpr int kB3M = 256, kB3N = 128;   // output tile of one workgroup (8 waves)

// Split pass: FP32 operand -> three bf16 planes in the tile-blocked layout,
// zero-padded to rows_pad x k_pad, so the matrix kernel needs no bounds
// checks. Both forms write whole 1 KB blocks per wave (lane l fills the
// block's 16-byte slot l).
//
// k-fast source (rows of k contiguous): one wave per block, each lane reads
// the 8 k-values of its chunk straight from its row.
template <int RB, int KB>
__global__ __launch_bounds__(256) void k_split3(const float *__restrict__ x, int64_t rows, int64_t k, int64_t ld,
                                                 unsigned short *__restrict__ planes, int64_t rows_pad, int64_t k_pad,
                                                 int64_t blk, int64_t plane)
{
  typedef B3Layout<RB, KB> Lay;
  static_assert(RB * Lay::kChunks == 64, "one chunk per lane");
  const int lane = threadIdx.x & 63;
  const int64_t nkb = k_pad / KB;
  const int64_t nblocks = rows_pad / RB * nkb;
  const int rr = lane / Lay::kChunks;                    // slot l holds row l / 4 at position l % 4
  const int c = Lay::pos(rr, lane % Lay::kChunks);       // (the position map is an involution in c)
  const int64_t wst = (int64_t)gridDim.x * 4;
  // rows that start 16-byte aligned: two 16-byte loads per lane
  const bool vec = ((uintptr_t)x % 16 == 0) && (ld % 4 == 0);
  for (int64_t bi = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); bi < nblocks; bi += wst) {
    const int64_t band = bi / nkb, kb = bi % nkb;
    const int64_t r = band * RB + rr, k0 = kb * KB + c * 8;
    float v[8];
    if (vec && r < rows && k0 + 8 <= k) {
      const float4 *src = reinterpret_cast<const float4 *>(x + r * ld + k0);
      const float4 u0 = src[0], u1 = src[1];
      v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w; v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (r < rows && k0 + i < k) ? x[r * ld + k0 + i] : 0.f;
    }
    us8 h0, h1, h2;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      unsigned short e0, e1, e2;
      split3(v[i], e0, e1, e2);
      h0[i] = e0; h1[i] = e1; h2[i] = e2;
    }
    const int64_t off = band * blk + kb * (RB * KB) + lane * 8;
    *reinterpret_cast<us8 *>(planes + off) = h0;
    *reinterpret_cast<us8 *>(planes + plane + off) = h1;
    *reinterpret_cast<us8 *>(planes + 2 * plane + off) = h2;
  }
}

// Row-fast source (x[kk * ld + r]): a workgroup takes 64 rows x KB k-values
// (four blocks), reads them as KB runs of 64 contiguous floats into LDS, and
// each wave then splits one block out of LDS.
template <int RB, int KB>
__global__ __launch_bounds__(256) void k_split3_rows(const float *__restrict__ x, int64_t rows, int64_t k, int64_t ld,
                                                      unsigned short *__restrict__ planes, int64_t rows_pad,
                                                      int64_t k_pad, int64_t blk, int64_t plane)
{
  typedef B3Layout<RB, KB> Lay;
  static_assert(RB == 16 && KB == 32, "four 16-row blocks per 64-row tile, 8 threads per k-run");
  __shared__ float t[KB][64 + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t nkb = k_pad / KB;
  const int64_t ntiles = rows_pad / 64 * nkb;
  const bool vec = ((uintptr_t)x % 16 == 0) && (ld % 4 == 0);
  const int lk = tid >> 3, lr = (tid & 7) * 8;           // load: k-run lk, rows lr .. lr+7
  const int rr = lane / Lay::kChunks;
  const int c = Lay::pos(rr, lane % Lay::kChunks);
  for (int64_t ti = blockIdx.x; ti < ntiles; ti += gridDim.x) {
    const int64_t rt = ti / nkb, kb = ti % nkb;
    const int64_t r0 = rt * 64 + lr, kk = kb * KB + lk;
    float v[8];
    if (vec && kk < k && r0 + 8 <= rows) {
      const float4 *src = reinterpret_cast<const float4 *>(x + kk * ld + r0);
      const float4 u0 = src[0], u1 = src[1];
      v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w; v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (kk < k && r0 + i < rows) ? x[kk * ld + r0 + i] : 0.f;
    }
    __syncthreads();  // the previous tile's reads of t are done
#pragma unroll
    for (int i = 0; i < 8; ++i) t[lk][lr + i] = v[i];
    __syncthreads();
    us8 h0, h1, h2;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      unsigned short e0, e1, e2;
      split3(t[c * 8 + i][wave * 16 + rr], e0, e1, e2);
      h0[i] = e0; h1[i] = e1; h2[i] = e2;
    }
    const int64_t off = (rt * 4 + wave) * blk + kb * (RB * KB) + lane * 8;
    *reinterpret_cast<us8 *>(planes + off) = h0;
    *reinterpret_cast<us8 *>(planes + plane + off) = h1;
    *reinterpret_cast<us8 *>(planes + 2 * plane + off) = h2;
  }
}

// Complex operands (C4) under the three-way split run as one real product of
// the realified operands, with the contracted extent doubled (k' = 2k):
//   A'' (2m x k'):  row 2r   = [ Re a(r,:), -Im a(r,:) ]
//                   row 2r+1 = [ Im a(r,:),  Re a(r,:) ]
//   B'' (n x k'):   row j    = [ Re b(j,:),  Im b(j,:) ]
// so that (A'' B''^T)(2r, j) = Re c(r,j) and (2r+1, j) = Im c(r,j): the real
// product's column-major 2m x n output is the complex m x n output,
// interleaved. Conjugation negates the imaginary parts on the way in. The
// pass writes the same tile-blocked planes as k_split3, one wave per 1 KB
// block, reading the complex source element by element (k-fast or row-fast).
template <int RB, int KB, bool IS_A>
__global__ __launch_bounds__(256) void k_split3_cx(const float2 *__restrict__ x, int64_t rows, int64_t k, int64_t ld,
                                                    int kfast, int conj, unsigned short *__restrict__ planes,
                                                    int64_t rows_pad, int64_t k_pad, int64_t blk, int64_t plane)
{
  typedef B3Layout<RB, KB> Lay;
  static_assert(RB * Lay::kChunks == 64, "one chunk per lane");
  const int lane = threadIdx.x & 63;
  const int64_t nkb = k_pad / KB;
  const int64_t nblocks = rows_pad / RB * nkb;
  const int rr = lane / Lay::kChunks;
  const int c = Lay::pos(rr, lane % Lay::kChunks);
  const int64_t wst = (int64_t)gridDim.x * 4;
  const int64_t rrows = IS_A ? 2 * rows : rows;          // realified rows
  const float isign = conj ? -1.f : 1.f;
  for (int64_t bi = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); bi < nblocks; bi += wst) {
    const int64_t band = bi / nkb, kb = bi % nkb;
    const int64_t rp = band * RB + rr, k0 = kb * KB + c * 8;
    const int64_t r = IS_A ? rp >> 1 : rp;
    const int comp = IS_A ? (int)(rp & 1) : 0;
    us8 h0, h1, h2;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t kk2 = k0 + i;
      float v = 0.f;
      if (rp < rrows && kk2 < 2 * k) {
        const int half = kk2 >= k ? 1 : 0;
        const int64_t kk = kk2 - half * k;
        const float2 z = x[kfast ? r * ld + kk : kk * ld + r];
        const float zi = isign * z.y;
        // A: (comp, half) = (0,0) re, (0,1) -im, (1,0) im, (1,1) re; B: (0,0) re, (0,1) im
        v = (comp == half) ? z.x : (IS_A && half) ? -zi : zi;
      }
      unsigned short e0, e1, e2;
      split3(v, e0, e1, e2);
      h0[i] = e0; h1[i] = e1; h2[i] = e2;
    }
    const int64_t off = band * blk + kb * (RB * KB) + lane * 8;
    *reinterpret_cast<us8 *>(planes + off) = h0;
    *reinterpret_cast<us8 *>(planes + plane + off) = h1;
    *reinterpret_cast<us8 *>(planes + 2 * plane + off) = h2;
  }
}

struct B3Params {
  const unsigned short *a3;  // 3 tile-blocked planes of A, plane_a elements apart
  const unsigned short *b3;
  float *part;               // split-K partial C tiles, m x n column-major each
  int64_t m, n, k_pad, kchunk;
  int64_t blk;               // elements between row bands (both operands)
  int64_t plane_a, plane_b;
  int tiles_m, tiles_n;
};

// The workgroups walk columns of 4 M-tiles: the 32 workgroups an XCD runs at
// once then cover 4 x 8 tiles, the arrangement that reads the fewest operand
// rows per k-step for 32 tiles.
__device__ __forceinline__ void tile_of_b3(const B3Params &p, int &tm, int &tn)
{
  tile_walk<4>(xcd_order(blockIdx.x, gridDim.x), p.tiles_m, p.tiles_n, tm, tn);
}

// Issue the DMA of one k-stage: NL 1 KB blocks (A planes x row bands, then B),
// spread over the 8 waves; block idx lands at wr + idx * 512.
template <int RB, int KB, int NL>
__device__ __forceinline__ void b3_issue(unsigned short *__restrict__ wr, const unsigned short *__restrict__ ga,
                                         const unsigned short *__restrict__ gb, const B3Params &p, int64_t kb,
                                         int wave, int lane)
{
  constexpr int NA = 3 * (kB3M / RB);
  constexpr int PER = (NL + 7) / 8;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int idx = wave + 8 * u;
    if (NL % 8 != 0 && u == PER - 1 && idx >= NL) break;
    const unsigned short *g;
    if (idx < NA) g = ga + (idx / (kB3M / RB)) * p.plane_a + (idx % (kB3M / RB)) * p.blk;
    else g = gb + ((idx - NA) / (kB3N / RB)) * p.plane_b + ((idx - NA) % (kB3N / RB)) * p.blk;
    lds_dma16(g + kb * (RB * KB) + lane * 8, wr + idx * 512);
  }
}

// Form 16: k-stages of 32, 16x16x32 MFMAs, each wave 64x64 (4x4 blocks),
// LDS double-buffered (2 x 72 KB). (A form with k-stages of 16, 32x32x16
// MFMAs and four 36 KB stages in flight measured 4% slower.)
//
// A stage function both issues the DMA of a later stage into `wr` and
// multiplies the stage in `rd`. The pointers are restrict-qualified because
// they name different stage buffers: that lets the compiler's wait-count pass
// see that the LDS reads of `rd` do not depend on the DMA still in flight
// into other buffers (without it every LDS read waits for all outstanding
// loads and the stages serialise). The dependence the DMA does carry (stage
// kt written before it is read) is enforced by the caller's vmcnt wait and
// barrier.
template <int FORM>
struct B3Form;

template <>
struct B3Form<16> {
  static constexpr int RB = 16, KB = 32, S = 2;
  static constexpr int NL = 3 * (kB3M + kB3N) / RB;   // 72 blocks per stage, 9 per wave
  typedef f4 Acc;
  static constexpr int FB = 4;                        // MFMA blocks per wave side
  __device__ static void stage(const unsigned short *__restrict__ rd, unsigned short *__restrict__ wr, bool issue,
                               bool compute, const unsigned short *__restrict__ ga,
                               const unsigned short *__restrict__ gb, const B3Params &p, int64_t kb, int wave,
                               int lane, int wm, int wn, Acc (&acc)[FB][FB])
  {
    if (issue) b3_issue<RB, KB, NL>(wr, ga, gb, p, kb, wave, lane);
    if (!compute) return;
    typedef B3Layout<RB, KB> Lay;
    const int fr = lane & 15, fc = lane >> 4;
    const int fpos = Lay::pos(fr, fc) * 8;
    const unsigned short *rb = rd + 3 * kB3M * KB;
    us8 fb[3][FB];
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
#pragma unroll
      for (int j = 0; j < FB; ++j) fb[pl][j] = *reinterpret_cast<const us8 *>(rb + (pl * kB3N + wn + j * 16 + fr) * KB + fpos);
#pragma unroll
    for (int i = 0; i < FB; ++i) {
      us8 fa[3];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) fa[pl] = *reinterpret_cast<const us8 *>(rd + (pl * kB3M + wm + i * 16 + fr) * KB + fpos);
      // products outer, blocks inner: consecutive MFMAs write different
      // accumulators; smallest terms first
#pragma unroll
      for (int t = 0; t < 6; ++t) {
        const int qa = t == 0 ? 0 : t == 1 ? 1 : t == 2 ? 2 : t == 3 ? 0 : t == 4 ? 1 : 0;
        const int qb = t == 0 ? 2 : t == 1 ? 1 : t == 2 ? 0 : t == 3 ? 1 : t == 4 ? 0 : 0;
#pragma unroll
        for (int j = 0; j < FB; ++j) acc[i][j] = mfma_bf(fa[qa], fb[qb][j], acc[i][j]);
      }
    }
  }
  // item r of lane l: row 4 (l / 16) + r, column l % 16
  __device__ static int row_of(int lane, int r) { return 4 * (lane >> 4) + r; }
  __device__ static int col_of(int lane) { return lane & 15; }
  static constexpr int BS = 16, NR = 4;
};

template <int FORM>
__global__ __launch_bounds__(512, 1) void k_gemm_bf16x3(const B3Params p)
{
  typedef B3Form<FORM> F;
  constexpr int S = F::S, KB = F::KB, FB = F::FB;
  constexpr int kStage = 3 * (kB3M + kB3N) * KB;      // bf16 values per LDS stage (A planes, then B planes)
  constexpr int kFold = 256 / KB;                     // stages per FP32 fold (256 k-values)
  __shared__ __align__(16) unsigned short lds[S * kStage];
  int tm, tn;
  tile_of_b3(p, tm, tn);
  const int64_t m0 = (int64_t)tm * kB3M, n0 = (int64_t)tn * kB3N;
  const int64_t kbeg = (int64_t)blockIdx.y * p.kchunk;
  const int64_t kend = min(kbeg + p.kchunk, p.k_pad);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 3) * 64, wn = (wave >> 2) * 64;
  const unsigned short *ga = p.a3 + (m0 / F::RB) * p.blk, *gb = p.b3 + (n0 / F::RB) * p.blk;
  typename F::Acc acc[FB][FB], sum[FB][FB];
#pragma unroll
  for (int i = 0; i < FB; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      acc[i][j] = typename F::Acc{};
      sum[i][j] = typename F::Acc{};
    }
  const int64_t nk = (kend - kbeg) / KB, kb0 = kbeg / KB;
  for (int s = 0; s < S - 1; ++s)
    if (s < nk) F::stage(lds + (S - 1) * kStage, lds + s * kStage, true, false, ga, gb, p, kb0 + s, wave, lane, wm, wn, acc);
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int cur = (int)(kt % S);
    // this wave's DMA of stage kt has landed (the only stage in flight here)
    static_assert(S == 2, "stage count");
    wait_vmcnt<0>();
    stage_barrier();  // everyone's stage kt is in LDS; stage kt-1's buffer is free
    F::stage(lds + cur * kStage, lds + ((cur + S - 1) % S) * kStage, kt + S - 1 < nk, true, ga, gb, p,
             kb0 + kt + S - 1, wave, lane, wm, wn, acc);
    if ((kt + 1) % kFold == 0 || kt + 1 == nk) {
#pragma unroll
      for (int i = 0; i < FB; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = typename F::Acc{};
        }
    }
  }
  float *P = p.part + (int64_t)blockIdx.y * p.m * p.n;
#pragma unroll
  for (int i = 0; i < FB; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      const int64_t col = n0 + wn + j * F::BS + F::col_of(lane);
#pragma unroll
      for (int r = 0; r < F::NR; ++r) {
        const int64_t row = m0 + wm + i * F::BS + F::row_of(lane, r);
        if (row < p.m && col < p.n) P[row + col * p.m] = sum[i][j][r];
      }
    }
}

// C = alpha * sum_z part[z] (+ C): FP64 sum over the K chunks. C and the
// partials are all m x n column-major with leading dimension m, so this is a
// 1-D pass over mn values, four per thread when mn allows.
__global__ __launch_bounds__(256) void k_splitk_reduce(const float *__restrict__ part, int nz, int64_t mn,
                                                       float *__restrict__ c, double alpha, int beta_zero)
{
  const int64_t st = (int64_t)gridDim.x * 256;
  const int64_t n4 = (mn % 4 == 0 && ((uintptr_t)c & 15) == 0) ? mn / 4 : 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += st) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int z = 0; z < nz; ++z) {
      const float4 v = reinterpret_cast<const float4 *>(part + (int64_t)z * mn)[i];
      s0 += (double)v.x; s1 += (double)v.y; s2 += (double)v.z; s3 += (double)v.w;
    }
    float4 o;
    if (beta_zero) {
      o = make_float4((float)(alpha * s0), (float)(alpha * s1), (float)(alpha * s2), (float)(alpha * s3));
    } else {
      const float4 cv = reinterpret_cast<const float4 *>(c)[i];
      o = make_float4((float)(alpha * s0 + (double)cv.x), (float)(alpha * s1 + (double)cv.y),
                      (float)(alpha * s2 + (double)cv.z), (float)(alpha * s3 + (double)cv.w));
    }
    reinterpret_cast<float4 *>(c)[i] = o;
  }
  for (int64_t i = n4 * 4 + (int64_t)blockIdx.x * 256 + threadIdx.x; i < mn; i += st) {
    double s = 0.0;
    for (int z = 0; z < nz; ++z) s += (double)part[(int64_t)z * mn + i];
    double v = alpha * s;
    if (!beta_zero) v += (double)c[i];
    c[i] = (float)v;
  }
}

// Complex form (C4 under the three-way split): the partials hold the m x n
// complex result interleaved; C = alpha * sum_z part[z] (+ C) with complex
// alpha, summed in FP64.
__global__ __launch_bounds__(256) void k_splitk_reduce_cx(const float2 *__restrict__ part, int nz, int64_t mn,
                                                          float2 *__restrict__ c, double are, double aim,
                                                          int beta_zero)
{
  const int64_t st = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < mn; i += st) {
    double sr = 0.0, si = 0.0;
    for (int z = 0; z < nz; ++z) {
      const float2 v = part[(int64_t)z * mn + i];
      sr += (double)v.x;
      si += (double)v.y;
    }
    double orr = are * sr - aim * si, oi = are * si + aim * sr;
    if (!beta_zero) {
      const float2 cv = c[i];
      orr += (double)cv.x;
      oi += (double)cv.y;
    }
    c[i] = make_float2((float)orr, (float)oi);
  }
}

// Realified complex operands for the native-precision complex product (C8 on
// FP64, C4 on FP32 matrix cores) of large problems: the same layout as the
// three-way split's complex form (k' = 2k, k fastest),
//   A'' (2m x k'):  row 2r   = [ Re a(r,:), -Im a(r,:) ],  row 2r+1 = [ Im a(r,:), Re a(r,:) ]
//   B'' (n x k'):   row j    = [ Re b(j,:),  Im b(j,:) ]
// so that the real product A'' B''^T, column-major 2m x n, is the complex m x n
// product interleaved. Conjugation negates imaginary parts; a complex alpha
// (are, aim) is applied to A on the way in (the real product then runs with
// alpha 1). One thread per source element.
template <typename T, bool IS_A>
__global__ __launch_bounds__(256) void k_realify(const T *__restrict__ x, int64_t rows, int64_t k, int64_t ld,
                                                 int kfast, int conj, double are, double aim,
                                                 T *__restrict__ out)
{
  const int64_t k2 = 2 * k;
  const int64_t total = rows * k;  // source elements
  const T isign = conj ? T(-1) : T(1);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    // i walks the source in its storage order (k fastest or rows fastest),
    // so that the reads are coalesced
    int64_t r, kk;
    if (kfast) { r = i / k; kk = i - r * k; }
    else { kk = i / rows; r = i - kk * rows; }
    const int64_t src = kfast ? r * ld + kk : kk * ld + r;
    T re = x[2 * src], im = isign * x[2 * src + 1];
    if (IS_A) {
      if (aim != 0.0 || are != 1.0) {
        const T nr = (T)are * re - (T)aim * im, ni = (T)are * im + (T)aim * re;
        re = nr;
        im = ni;
      }
      T *r0 = out + (2 * r) * k2, *r1 = r0 + k2;
      r0[kk] = re;
      r0[k + kk] = -im;
      r1[kk] = im;
      r1[k + kk] = re;
    } else {
      T *r0 = out + r * k2;
      r0[kk] = re;
      r0[k + kk] = im;
    }
  }
}

// Element offset of index i of a group of at most kSmallDims dimensions.
__device__ __forceinline__ int64_t group_at(const DevGroup<kSmallDims> &g, int i)
{
  uint32_t r = (uint32_t)i;
  int64_t o = 0;
#pragma unroll
  for (int j = 0; j < kSmallDims; ++j) {
    if (j + 1 < kSmallDims && j + 1 < g.nd) {
      const uint32_t q = (__umulhi(r, g.div[j].m) + r) >> g.div[j].s;
      o += (int64_t)(r - q * g.div[j].d) * g.str[j];
      r = q;
    } else if (j + 1 == g.nd) {
      o += (int64_t)r * g.str[j];
    }
  }
  return o;
}

// Split pass straight from a tensor read in place (rows and k given as index
// groups): a workgroup takes 64 rows x 64 k-values, decodes their offsets once,
// reads them with lanes along the tensor's contiguous side into LDS, and each
// wave splits two blocks out of LDS. Replaces a transpose of the operand (a
// read and a write of it) and the re-read by k_split3.
template <bool ROWS>
__global__ __launch_bounds__(256) void k_split3_gather(const float *__restrict__ x, const DevGroup<kSmallDims> grow,
                                                       const DevGroup<kSmallDims> gk, int rows, int k,
                                                       unsigned short *__restrict__ planes, int rows_pad, int k_pad,
                                                       int64_t blk, int64_t plane)
{
  typedef B3Layout<16, 32> Lay;
  constexpr int TS = 64;
  __shared__ float t[TS][TS + 1];         // [k][row]
  __shared__ int64_t off[2][TS];          // rows, k
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nkt = (k_pad + TS - 1) / TS, ntiles = rows_pad / TS * nkt;
  const int rr = lane / Lay::kChunks, c = Lay::pos(rr, lane % Lay::kChunks);
  for (int ti = blockIdx.x; ti < ntiles; ti += gridDim.x) {
    const int rt = ti / nkt, r0 = rt * TS, k0 = (ti - rt * nkt) * TS;
    if (tid < TS) off[0][tid] = group_at(grow, min(r0 + tid, rows - 1));
    else if (tid < 2 * TS) off[1][tid - TS] = group_at(gk, min(k0 + tid - TS, k - 1));
    __syncthreads();
    float v[TS / 4];
#pragma unroll
    for (int u = 0; u < TS / 4; ++u) {
      const int i = ROWS ? lane : wave + 4 * u, j = ROWS ? wave + 4 * u : lane;  // row, k
      v[u] = x[off[0][i] + off[1][j]];
    }
#pragma unroll
    for (int u = 0; u < TS / 4; ++u) {
      const int i = ROWS ? lane : wave + 4 * u, j = ROWS ? wave + 4 * u : lane;
      t[j][i] = (r0 + i < rows && k0 + j < k) ? v[u] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (k0 + u * 32 >= k_pad) break;
      us8 h0, h1, h2;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        unsigned short e0, e1, e2;
        split3(t[u * 32 + c * 8 + e][wave * 16 + rr], e0, e1, e2);
        h0[e] = e0; h1[e] = e1; h2[e] = e2;
      }
      const int64_t o = (int64_t)(rt * 4 + wave) * blk + (int64_t)(k0 / 32 + u) * 512 + lane * 8;
      *reinterpret_cast<us8 *>(planes + o) = h0;
      *reinterpret_cast<us8 *>(planes + plane + o) = h1;
      *reinterpret_cast<us8 *>(planes + 2 * plane + o) = h2;
    }
    __syncthreads();
  }
}

// k_splitk_reduce into a tensor written in place: D element (r, c) sits at the
// offsets of its row and column groups. A wave takes 64 rows (which hold D's
// contiguous index) of 16 columns. Replaces the product's own pass, D's
// transpose back and, accumulating, its transpose in.
__global__ __launch_bounds__(256) void k_splitk_reduce_gather(const float *__restrict__ part, int nz, int m, int n,
                                                              const DevGroup<kSmallDims> grow,
                                                              const DevGroup<kSmallDims> gcol, float *__restrict__ d,
                                                              double alpha, int beta_zero)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  if (r >= m) return;
  const int64_t ro = group_at(grow, r), mn = (int64_t)m * n;
#pragma unroll 4
  for (int u = 0; u < 16; ++u) {
    const int c = blockIdx.y * 64 + wave * 16 + u;
    if (c >= n) break;
    double v = 0.0;
    for (int z = 0; z < nz; ++z) v += (double)part[(int64_t)z * mn + (int64_t)c * m + r];
    v *= alpha;
    float *dst = d + ro + group_at(gcol, c);
    if (!beta_zero) v += (double)*dst;
    *dst = (float)v;
  }
}

constexpr int kB3Form = 16;               // kernel form of the three-way split

int64_t round_up(int64_t x, int64_t q) { return (x + q - 1) / q * q; }

struct B3Geom {
  int64_t kp, mp, np, blk, plane_a, plane_b, nz;
};

// Geometry of the split planes; a complex product runs realified (2m rows of
// A, contracted extent 2k).
B3Geom b3_geom(const GemmArgs &g)
{
  B3Geom G;
  const int64_t cx = g.kind == C4 ? 2 : 1;
  G.kp = round_up(std::max<int64_t>(cx * (int64_t)g.k, 1), 32);
  G.mp = round_up(cx * (int64_t)g.m, kB3M);
  G.np = round_up((int64_t)g.n, kB3N);
  const int rb = B3Form<kB3Form>::RB;
  G.blk = rb * G.kp;
  G.plane_a = G.mp / rb * G.blk;
  G.plane_b = G.np / rb * G.blk;
  G.nz = (G.kp + kB3Chunk - 1) / kB3Chunk;
  return G;
}

// The matrix kernel over split planes a3 and b3, K-chunk partials behind them.
B3Params b3_product(const GemmArgs &g, const B3Geom &G, unsigned short *a3, unsigned short *b3, hipStream_t s)
{
  const bool cx = g.kind == C4;
  B3Params p{};
  p.a3 = a3; p.b3 = b3;
  p.part = reinterpret_cast<float *>(b3 + 3 * G.plane_b);
  p.m = (cx ? 2 : 1) * (int64_t)g.m; p.n = (int64_t)g.n; p.k_pad = G.kp;
  p.kchunk = std::min<int64_t>(G.kp, kB3Chunk);
  p.blk = G.blk; p.plane_a = G.plane_a; p.plane_b = G.plane_b;
  p.tiles_m = (int)(G.mp / kB3M);
  p.tiles_n = (int)(G.np / kB3N);
  hipLaunchKernelGGL(k_gemm_bf16x3<kB3Form>, dim3(p.tiles_m * p.tiles_n, (int)G.nz), dim3(512), 0, s, p);
  return p;
}

int launch_bf16x3(const GemmArgs &g, void *ws, hipStream_t s)
{
  typedef B3Form<kB3Form> F;
  if (!ws) return TALSH_INVALID_ARGS;
  const B3Geom G = b3_geom(g);
  unsigned short *a3 = static_cast<unsigned short *>(ws);
  unsigned short *b3 = a3 + 3 * G.plane_a;
  auto split = [&](const void *x, int64_t rows, bool kfast, unsigned short *out, int64_t rows_pad, int64_t plane) {
    const float *xf = static_cast<const float *>(x);
    if (kfast) {
      const int64_t nblocks = rows_pad / F::RB * (G.kp / F::KB);  // one wave each, 4 per workgroup
      const int blocks = (int)std::min<int64_t>((nblocks + 3) / 4, 65536);
      hipLaunchKernelGGL((k_split3<F::RB, F::KB>), dim3(blocks), dim3(256), 0, s, xf, rows, (int64_t)g.k,
                         (int64_t)g.k, out, rows_pad, G.kp, G.blk, plane);
    } else {
      const int64_t ntiles = rows_pad / 64 * (G.kp / F::KB);
      const int blocks = (int)std::min<int64_t>(ntiles, 65536);
      hipLaunchKernelGGL((k_split3_rows<F::RB, F::KB>), dim3(blocks), dim3(256), 0, s, xf, rows, (int64_t)g.k, rows,
                         out, rows_pad, G.kp, G.blk, plane);
    }
  };
  if (g.kind == R4) {
    split(g.a, (int64_t)g.m, g.a_kfast, a3, G.mp, G.plane_a);
    split(g.b, (int64_t)g.n, g.b_kfast, b3, G.np, G.plane_b);
  }
  const bool cx = g.kind == C4;
  if (cx) {
    const int64_t nblocks_a = G.mp / F::RB * (G.kp / F::KB), nblocks_b = G.np / F::RB * (G.kp / F::KB);
    const int ba = (int)std::min<int64_t>((nblocks_a + 3) / 4, 65536);
    const int bb = (int)std::min<int64_t>((nblocks_b + 3) / 4, 65536);
    const int64_t lda = g.a_kfast ? (int64_t)g.k : (int64_t)g.m, ldb = g.b_kfast ? (int64_t)g.k : (int64_t)g.n;
    hipLaunchKernelGGL((k_split3_cx<F::RB, F::KB, true>), dim3(ba), dim3(256), 0, s,
                       static_cast<const float2 *>(g.a), (int64_t)g.m, (int64_t)g.k, lda, g.a_kfast ? 1 : 0,
                       g.conj_a ? 1 : 0, a3, G.mp, G.kp, G.blk, G.plane_a);
    hipLaunchKernelGGL((k_split3_cx<F::RB, F::KB, false>), dim3(bb), dim3(256), 0, s,
                       static_cast<const float2 *>(g.b), (int64_t)g.n, (int64_t)g.k, ldb, g.b_kfast ? 1 : 0,
                       g.conj_b ? 1 : 0, b3, G.np, G.kp, G.blk, G.plane_b);
  }
  const B3Params p = b3_product(g, G, a3, b3, s);
  const int64_t mn = (int64_t)g.m * (int64_t)g.n;
  if (cx) {
    const int rb = (int)std::min<int64_t>((mn + 255) / 256, 8192);
    hipLaunchKernelGGL(k_splitk_reduce_cx, dim3(rb), dim3(256), 0, s, reinterpret_cast<const float2 *>(p.part),
                       (int)G.nz, mn, static_cast<float2 *>(g.c), g.alpha_re, g.alpha_im, g.beta_zero ? 1 : 0);
  } else {
    const int rb = (int)std::min<int64_t>((mn / 4 + 255) / 256 + 1, 8192);
    hipLaunchKernelGGL(k_splitk_reduce, dim3(rb), dim3(256), 0, s, p.part, (int)G.nz, mn, static_cast<float *>(g.c),
                       g.alpha_re, g.beta_zero ? 1 : 0);
  }
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

}  // namespace

int gemm_default_tile(int kind, R4Mode r4mode, size_t m, size_t n, size_t k);

int current_cus()
{
  static const int cus = []() {
    int dev = 0, c = 256;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
        prop.multiProcessorCount > 0)
      c = prop.multiProcessorCount;
    return c;
  }();
  return cus;
}

bool native_real(const GemmArgs &g) { return g.kind == R8 || (g.kind == R4 && g.r4mode == R4Mode::kNativeF32); }

constexpr int64_t kSplitMinK = 256;  // shortest K that is cut

// How a product's tiles are cut along K: tiles [0, full) run whole, the later
// ones in `parts` pieces of kchunk k-values.
struct SplitGeom {
  int64_t tiles = 0, full = 0, kchunk = 0, zstride = 0;
  int parts = 1;
  size_t bytes = 0;  // workspace of the partials
};

// Cost model of the cut. Workgroups of several k-groups fill a CU alone; of
// the others a CU holds two, and one alone hides its latencies worse (a 64x64
// FP64 tile per CU runs at 41 TFLOP/s, two at 51, a 128x128 one at 58 and 63).
// Whole rounds of tiles need no cut; what is left over is cut into the number
// of parts that ends soonest, the sum of the pieces (a launch and a pass over
// the partials) included. Pieces are at least 128 k-values deep. budget:
// bytes available for the partials.
SplitGeom split_geom(const GemmArgs &g, const TileShape &ts, int cus, size_t budget)
{
  SplitGeom G;
  const int64_t m = (int64_t)g.m, n = (int64_t)g.n, k = (int64_t)g.k;
  const int64_t tm = (m + ts.bm - 1) / ts.bm, tn = (n + ts.bn - 1) / ts.bn;
  G.tiles = G.full = tm * tn;
  G.kchunk = k;
  const int es = kind_size(g.kind);
  const bool cplx = g.kind == C8 || g.kind == C4, dp = g.kind == R8 || g.kind == C8;
  const int64_t round = (ts.groups > 1 ? 1 : 2) * (int64_t)cus;
  const int64_t full = G.tiles / round * round, rem = G.tiles - full;
  if (rem == 0 || k < kSplitMinK || k > kMaxDepth) return G;
  // microseconds of one tile on a CU of its own at 80% of its matrix rate
  const double tau = (cplx ? 8.0 : 2.0) * ts.bm * ts.bn * (double)k / (0.8 * (dp ? 78.6e6 : 157.3e6) / 256.0);
  auto cost = [&](int64_t parts) {
    const int64_t q = (rem * parts + cus - 1) / cus;  // pieces per CU
    const double eff = q > 1 || ts.groups > 1 ? 1.0 : 0.8;
    double c = tau * (double)q / (double)parts / eff;
    if (parts > 1) c += 8.0 + 2.0 * (double)rem * ts.bm * ts.bn * es * (double)parts / 4.0e6;
    return c;
  };
  double best = 0.95 * cost(1);
  for (int64_t parts = 2; parts <= 64 && k / parts >= 128; ++parts) {
    const int64_t chunk = ((k + parts - 1) / parts + ts.bk - 1) / ts.bk * ts.bk;
    if ((k + chunk - 1) / chunk != parts) continue;
    const int64_t zs = full > 0 ? rem * ts.bm * ts.bn : m * n;
    const size_t bytes = (size_t)parts * (size_t)zs * es;
    if (bytes > budget) break;
    const double c = cost(parts);
    if (c < best) {
      best = c;
      G.full = full;
      G.parts = (int)parts;
      G.kchunk = chunk;
      G.zstride = zs;
      G.bytes = bytes;
    }
  }
  return G;
}

bool gemm_vec_loads(int es, bool kfast, size_t rows, size_t k)
{
  return kfast ? k * (size_t)es % 16 == 0 : k % 8 == 0 && rows % 2 == 0;
}

bool gather_vec_loads(int es, bool kfast, const GatherGroup &row, const GatherGroup &kg, size_t k)
{
  const GatherGroup &x = kfast ? kg : row;
  return x.nd > 0 && x.str[0] == 1 && x.ext[0] % (kfast ? std::max(16 / es, 1) : 2) == 0 && (kfast || k % 8 == 0);
}

bool gather_uniform_k(int kind, const GatherMaps &mp)
{
  for (const GatherGroup *x : {&mp.a_row, &mp.a_k, &mp.b_row, &mp.b_k, &mp.c_row, &mp.c_col})
    if (x->nd > kSmallDims) return false;
  for (const GatherGroup *x : {&mp.a_k, &mp.b_k})
    if (x->nd > 3 || (x->nd > 1 && x->ext[0] % tile_shape(kind, 0).bk != 0)) return false;
  return true;
}

// Large complex products in native precision run realified through the real
// 128x128 kernels (which re-read operands from L2 half as often as the 64x64
// complex kernel), when the real product has enough 128x128 tiles to fill the
// chip twice and K is deep enough to amortise the realify pass.
bool complex_realified(const GemmArgs &g)
{
  if ((g.kind != C8 && g.kind != C4) || gemm_uses_split3(g)) return false;
  const size_t tiles = ((2 * g.m + 127) / 128) * ((g.n + 127) / 128);
  return tiles >= (size_t)(2 * current_cus()) && g.k >= 512;
}

size_t realified_bytes(const GemmArgs &g)
{
  const size_t es = g.kind == C8 ? 8 : 4, k2 = 2 * g.k;
  return ((2 * g.m * k2 * es + 255) / 256 * 256) + g.n * k2 * es + 16;
}

// Tile choice of the kernels: a caller's, or the default; complex kinds have
// one choice, their two forms are told apart here: two k-groups per workgroup
// when the tiles do not give every CU two workgroups and K is deep enough. Two
// groups share more than 64 k-values (C8 64x64, two groups and one: k 8 13 and
// 11 us, 48 18 and 15, 64 18 and 18, 128 26 and 27, 512 77 and 82); where a CU
// would run its two workgroups one after the other they need K deep enough for
// a cut of the last round besides (C8 1280x960: k 8 25 and 16 us, 160 62 and 53;
// 512, in pieces, 111 and 141; C4 16 and 12, 35 and 33, 60 and 81).
int resolved_tile(const GemmArgs &g)
{
  if (g.kind == C8 || g.kind == C4) {
    const int64_t tiles = (int64_t)((g.m + 63) / 64) * (int64_t)((g.n + 63) / 64);
    const int64_t cus = current_cus();
    return g.k > 64 && (tiles <= cus || (tiles < 2 * cus && g.k >= kSplitMinK)) ? 1 : 0;
  }
  return g.tile < 0 ? gemm_default_tile(g.kind, g.r4mode, g.m, g.n, g.k) : g.tile;
}

// Partials of the published workspace query (talshAmdGemmWorkspace): up to
// eight pieces of a real product with few 64x64 output tiles.
size_t gemm_workspace_bytes(const GemmArgs &g)
{
  if (!gemm_uses_split3(g)) {
    if (g.kind == C8 || g.kind == C4) return complex_realified(g) ? realified_bytes(g) : 0;
    if (resolved_tile(g) == 0 || g.k < 512) return 0;
    const int64_t tiles = (int64_t)((g.m + 63) / 64) * (int64_t)((g.n + 63) / 64);
    const int64_t want = 2 * (int64_t)current_cus();
    const int64_t nz = tiles >= want ? 1 : std::min<int64_t>({8, want / tiles, (int64_t)g.k / 256});
    return nz > 1 ? (size_t)nz * g.m * g.n * (size_t)kind_size(g.kind) + 16 : 0;
  }
  const B3Geom G = b3_geom(g);
  // split planes (bf16) + K-chunk partials (FP32, m x n each; complex: 2m x n)
  const int64_t cx = g.kind == C4 ? 2 : 1;
  return (size_t)(3 * (G.plane_a + G.plane_b)) * sizeof(unsigned short) +
         (size_t)(G.nz * cx * (int64_t)g.m * (int64_t)g.n) * 4 + 16;
}

// Bytes of partials worth having for a product whose workspace is free to
// choose (a contraction's temporaries); a product runs with less, or none.
size_t gemm_split_bytes(const GemmArgs &g)
{
  if (gemm_uses_split3(g) || complex_realified(g) || g.m == 0 || g.n == 0 || g.k == 0) return 0;
  return split_geom(g, tile_shape(g.kind, resolved_tile(g)), current_cus(), kSplitBytesMax).bytes;
}

// The partials, and room that keeps a gathered contraction subject to the
// arena's back-pressure like one with transposes (the kernels need none of
// it: they compute their offsets).
size_t gemm_gather_workspace_bytes(const GemmArgs &g)
{
  if (gemm_uses_split3(g)) return 0;
  const size_t room = ((2 * (g.m + g.n + g.k) + 10) * sizeof(int64_t) + 255) / 256 * 256;
  return room + (g.kind == C8 || g.kind == C4 ? 0 : gemm_workspace_bytes(g));
}

int launch_gemm(const GemmArgs &g, hipStream_t s) { return launch_gemm_ws(g, nullptr, 0, s); }

// Scratch of talshAmdGemmNoAlloc. In host code this name is a host-side
// stand-in, not a device address: only the pointer that
// gemm_noalloc_scratch returns may be handed to kernels or copies.
static __device__ __align__(256) unsigned char scratch[kGemmNoAllocScratchBytes];

int gemm_noalloc_scratch(void **ptr)
{
  *ptr = nullptr;
  if (!XT_HIP_OK(hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch)))) {
    *ptr = nullptr;
    return TALSH_FAILURE;
  }
  return 0;
}

bool gemm_uses_split3(const GemmArgs &g) { return (g.kind == R4 || g.kind == C4) && g.r4mode == R4Mode::kBF16x3; }

int gemm_tile_choices(int kind, R4Mode r4mode);

int gemm_default_tile(int kind, R4Mode r4mode, size_t m, size_t n, size_t k)
{
  if (gemm_tile_choices(kind, r4mode) == 1) return 0;
  const int cus = current_cus();
  // 128x128 tiles pay off only when there are enough of them to fill the
  // chip twice over and K is deep enough to amortise their prologue;
  // otherwise 64x64 tiles balance better (measured over random contractions)
  const size_t tiles128 = ((m + 127) / 128) * ((n + 127) / 128);
  return (tiles128 >= (size_t)(2 * cus) && k >= 2048) ? 0 : 2;
}

int gemm_splitk_count(int kind, R4Mode r4mode, size_t m, size_t n, size_t k, int tile, int cus)
{
  GemmArgs g{};
  g.kind = kind; g.r4mode = r4mode; g.m = m; g.n = n; g.k = k; g.tile = tile;
  if (gemm_uses_split3(g) || complex_realified(g) || k == 0) return 1;
  return split_geom(g, tile_shape(kind, tile), cus, kSplitBytesMax).parts;
}

int gemm_tile_choices(int kind, R4Mode r4mode)
{
  if (kind == R8 || (kind == R4 && r4mode == R4Mode::kNativeF32)) return 3;
  return 1;
}

void gemm_tile_shape(int kind, R4Mode r4mode, int tile, int *bm, int *bn, int *occupancy)
{
  *bm = *bn = 128;
  *occupancy = 2;
  if (kind == R4 && r4mode == R4Mode::kBF16x3) { *occupancy = 1; return; }
  const TileShape ts = tile_shape(kind, tile);
  *bm = ts.bm;
  *bn = ts.bn;
  if (ts.groups > 1) *occupancy = 1;
}

namespace {

typedef DevGroup<kGatherMaxDims> FullGroup;

FullGroup dev_group(const GatherGroup &g)
{
  FullGroup d{};
  d.nd = g.nd;
  for (int j = 0; j < g.nd; ++j) {
    d.str[j] = g.str[j];
    if (j + 1 < g.nd) {
      const FastDiv f((uint32_t)g.ext[j]);
      d.div[j] = DevDivisor{f.d, f.m, f.s};
    }
  }
  for (int j = std::max(g.nd - 1, 0); j + 1 < kGatherMaxDims; ++j) d.div[j] = DevDivisor{1, 0, 0};
  if (g.nd > 0) d.str[kGatherMaxDims - 1] = g.str[g.nd - 1];
  return d;
}

FullGroup line_group(int64_t stride)
{
  FullGroup d{};
  d.nd = 1;
  d.str[0] = stride;
  return d;
}

// Whether the offsets that a lane of the uniform modes holds (of its rows, from
// the tile's first row where they are one dimension, and of its k-values inside
// a k-tile) fit 32 bits.
bool lane_offsets_fit(const FullGroup &row, const FullGroup &kg, int64_t rows, int es)
{
  int64_t o = 0;
  if (row.nd <= 1) {
    o = 127 * row.str[0];
  } else {
    int64_t n = 1;
    for (int j = 0; j + 1 < row.nd; ++j) {
      o += (int64_t)(row.div[j].d - 1) * row.str[j];
      n *= row.div[j].d;
    }
    o += (rows / n - 1) * row.str[row.nd - 1];
  }
  const int64_t k0 = kg.str[0];
  return o < (1ll << 32) && k0 < (1ll << 32) && (o + 31 * k0) * es + 16 < (1ll << 32);
}

// Launches product q of g's shape (g.m, g.n after any exchange of A and B) on
// tile choice `tile`, cutting K as the workspace allows.
int launch_product(Product &q, const GemmArgs &g, int tile, void *ws, size_t ws_bytes, hipStream_t s)
{
  const TileShape ts = tile_shape(g.kind, tile);
  const int64_t tm = ((int64_t)g.m + ts.bm - 1) / ts.bm, tn = ((int64_t)g.n + ts.bn - 1) / ts.bn;
  if (tm >= (1ll << 31) || tn >= (1ll << 31) || tm * tn >= (1ll << 31) - 65536) return TALSH_LIMIT_EXCEEDED;
  auto &p = q.p;
  p.a_line = p.a_row.nd <= 1 ? p.a_row.str[0] : 0;
  p.b_line = p.b_row.nd <= 1 ? p.b_row.str[0] : 0;
  p.tiles_m = (int)tm;
  p.tiles_n = (int)tn;
  const SplitGeom G = split_geom(g, ts, current_cus(), ws ? ws_bytes : 0);
  p.part = ws;
  p.full = (int)G.full;
  p.parts = G.parts;
  p.kchunk = G.kchunk;
  p.zstride = G.zstride;
  // K beyond kMaxDepth runs in stretches that accumulate in C, one after the
  // other
  for (int64_t k0 = 0; k0 < (int64_t)g.k || k0 == 0; k0 += kMaxDepth) {
    p.k0 = k0;
    p.k = std::min((int64_t)g.k, k0 + kMaxDepth);
    if (k0 > 0) p.beta_zero = 0;
    int e;
    switch (g.kind) {
    case R8:
      e = tile == 2 ? launch_native<R8, 2>(q, s) : tile == 1 ? launch_native<R8, 1>(q, s) : launch_native<R8, 0>(q, s);
      break;
    case R4:
      e = tile == 2 ? launch_native<R4, 2>(q, s) : tile == 1 ? launch_native<R4, 1>(q, s) : launch_native<R4, 0>(q, s);
      break;
    case C8: e = tile == 1 ? launch_native<C8, 1>(q, s) : launch_native<C8, 0>(q, s); break;
    case C4: e = tile == 1 ? launch_native<C4, 1>(q, s) : launch_native<C4, 0>(q, s); break;
    default: return TALSH_INVALID_ARGS;
    }
    if (e) return e;
  }
  return 0;
}

// Exchanges A and B (the product of the transposes, C^T = B^T A^T).
void exchange(Product &q, GemmArgs &g)
{
  auto &p = q.p;
  std::swap(p.a, p.b);
  std::swap(p.m, p.n);
  std::swap(p.conj_a, p.conj_b);
  std::swap(p.a_row, p.b_row);
  std::swap(p.a_k, p.b_k);
  std::swap(p.c_row, p.c_col);
  std::swap(q.a_kfast, q.b_kfast);
  std::swap(g.m, g.n);
}

Product product_of(const GemmArgs &g)
{
  Product q;
  auto &p = q.p;
  p.a = g.a; p.b = g.b; p.c = g.c;
  p.m = (int64_t)g.m; p.n = (int64_t)g.n; p.k = (int64_t)g.k;
  p.alpha_re = g.alpha_re; p.alpha_im = g.alpha_im;
  p.beta_zero = g.beta_zero ? 1 : 0;
  p.conj_a = g.conj_a; p.conj_b = g.conj_b;
  q.a_kfast = g.a_kfast;
  q.b_kfast = g.b_kfast;
  return q;
}

// A matricized product. C is column-major, so A and B change places: the
// kernels write along the result's columns (16 lanes of a wave on consecutive
// columns), which then are C's contiguous index.
int launch_matrix(GemmArgs g, int tile, void *ws, size_t ws_bytes, hipStream_t s)
{
  Product q = product_of(g);
  auto &p = q.p;
  p.a_row = line_group(g.a_kfast ? p.k : 1);
  p.a_k = line_group(g.a_kfast ? 1 : p.m);
  p.b_row = line_group(g.b_kfast ? p.k : 1);
  p.b_k = line_group(g.b_kfast ? 1 : p.n);
  p.c_row = line_group(1);
  p.c_col = line_group(p.m);
  const int es = kind_size(g.kind);
  const bool off32 = lane_offsets_fit(p.a_row, p.a_k, p.m, es) && lane_offsets_fit(p.b_row, p.b_k, p.n, es);
  q.mode = !off32 ? kTab
           : gemm_vec_loads(es, g.a_kfast, g.m, g.k) && gemm_vec_loads(es, g.b_kfast, g.n, g.k) ? kVec : kUni;
  exchange(q, g);
  return launch_product(q, g, tile, ws, ws_bytes, s);
}

}  // namespace

int launch_gemm_ws(const GemmArgs &g, void *ws, size_t ws_bytes, hipStream_t s)
{
  if (g.m == 0 || g.n == 0) return 0;
  if (g.k == 0 && !g.beta_zero) return 0;  // empty contraction leaves C unchanged
  if (gemm_uses_split3(g)) {
    if (!ws || ws_bytes < gemm_workspace_bytes(g)) return TALSH_INVALID_ARGS;
    return launch_bf16x3(g, ws, s);
  }
  if (!ws) ws_bytes = 0;
  const int tile = resolved_tile(g);
  if (!complex_realified(g) || ws_bytes < realified_bytes(g)) return launch_matrix(g, tile, ws, ws_bytes, s);
  const bool dp = g.kind == C8;
  const size_t es = dp ? 8 : 4;
  const int64_t k2 = 2 * (int64_t)g.k;
  char *a2 = static_cast<char *>(ws);
  char *b2 = a2 + (2 * g.m * (size_t)k2 * es + 255) / 256 * 256;
  const bool real_alpha = g.alpha_im == 0.0;
  const double are = real_alpha ? 1.0 : g.alpha_re, aim = real_alpha ? 0.0 : g.alpha_im;
  const int64_t lda = g.a_kfast ? (int64_t)g.k : (int64_t)g.m, ldb = g.b_kfast ? (int64_t)g.k : (int64_t)g.n;
  const int ga = (int)std::min<int64_t>(((int64_t)g.m * (int64_t)g.k + 255) / 256, 65536);
  const int gb = (int)std::min<int64_t>(((int64_t)g.n * (int64_t)g.k + 255) / 256, 65536);
  GemmArgs r = g;
  r.kind = dp ? R8 : R4;
  r.m = 2 * g.m;
  r.k = (size_t)k2;
  r.a = a2;
  r.b = b2;
  r.a_kfast = r.b_kfast = true;
  r.conj_a = r.conj_b = false;
  r.alpha_re = real_alpha ? g.alpha_re : 1.0;
  r.alpha_im = 0.0;
  if (dp) {
    hipLaunchKernelGGL((k_realify<double, true>), dim3(ga), dim3(256), 0, s, static_cast<const double *>(g.a),
                       (int64_t)g.m, (int64_t)g.k, lda, g.a_kfast ? 1 : 0, g.conj_a ? 1 : 0, are, aim,
                       reinterpret_cast<double *>(a2));
    hipLaunchKernelGGL((k_realify<double, false>), dim3(gb), dim3(256), 0, s, static_cast<const double *>(g.b),
                       (int64_t)g.n, (int64_t)g.k, ldb, g.b_kfast ? 1 : 0, g.conj_b ? 1 : 0, 1.0, 0.0,
                       reinterpret_cast<double *>(b2));
  } else {
    hipLaunchKernelGGL((k_realify<float, true>), dim3(ga), dim3(256), 0, s, static_cast<const float *>(g.a),
                       (int64_t)g.m, (int64_t)g.k, lda, g.a_kfast ? 1 : 0, g.conj_a ? 1 : 0, are, aim,
                       reinterpret_cast<float *>(a2));
    hipLaunchKernelGGL((k_realify<float, false>), dim3(gb), dim3(256), 0, s, static_cast<const float *>(g.b),
                       (int64_t)g.n, (int64_t)g.k, ldb, g.b_kfast ? 1 : 0, g.conj_b ? 1 : 0, 1.0, 0.0,
                       reinterpret_cast<float *>(b2));
  }
  return launch_matrix(r, 0, nullptr, 0, s);
}

// Three-way split product of tensors read in place. Groups of at most
// kSmallDims dimensions and matrix indices below 2^31; rows along each
// operand's contiguous side need not be known (a_kfast, b_kfast say which).
bool split3_gather_ok(const GatherMaps &mp, size_t m, size_t n, size_t k)
{
  for (const GatherGroup *x : {&mp.a_row, &mp.a_k, &mp.b_row, &mp.b_k, &mp.c_row, &mp.c_col})
    if (x->nd > kSmallDims) return false;
  // runs of four elements on every side: with shorter ones the gathers and the
  // scatter move single elements (2574 x 2560 x 3072, L's and D's runs shortened:
  // 16 elements 267 us against 339 with transposes, 4 302 against 338, 2 357
  // against 334)
  auto run = [](const GatherGroup &x) { return x.nd > 0 && x.str[0] == 1 && x.ext[0] >= 4; };
  return (run(mp.a_row) || run(mp.a_k)) && (run(mp.b_row) || run(mp.b_k)) && run(mp.c_row) &&
         std::max({m, n, k}) < (size_t)1 << 24 && n <= (size_t)65535 * 64;
}

int launch_split3_gather(const GemmArgs &g, const GatherMaps &mp, void *ws, size_t ws_bytes, hipStream_t s)
{
  if (g.kind != R4 || !gemm_uses_split3(g) || !split3_gather_ok(mp, g.m, g.n, g.k)) return TALSH_INVALID_ARGS;
  if (!ws || ws_bytes < gemm_workspace_bytes(g)) return TALSH_INVALID_ARGS;
  const B3Geom G = b3_geom(g);
  unsigned short *a3 = static_cast<unsigned short *>(ws), *b3 = a3 + 3 * G.plane_a;
  auto shrink = [](const GatherGroup &x) {
    const FullGroup f = dev_group(x);
    DevGroup<kSmallDims> d{};
    d.nd = f.nd;
    for (int j = 0; j < kSmallDims; ++j) d.str[j] = f.str[j];
    for (int j = 0; j + 1 < kSmallDims; ++j) d.div[j] = f.div[j];
    return d;
  };
  auto split = [&](const void *x, const GatherGroup &row, const GatherGroup &kg, size_t rows, bool kfast,
                   unsigned short *out, int64_t rows_pad, int64_t plane) {
    const int64_t tiles = rows_pad / 64 * ((G.kp + 63) / 64);
    const dim3 grid((unsigned)std::min<int64_t>(tiles, 1 << 16));
    if (kfast)
      hipLaunchKernelGGL(k_split3_gather<false>, grid, dim3(256), 0, s, static_cast<const float *>(x), shrink(row),
                         shrink(kg), (int)rows, (int)g.k, out, (int)rows_pad, (int)G.kp, G.blk, plane);
    else
      hipLaunchKernelGGL(k_split3_gather<true>, grid, dim3(256), 0, s, static_cast<const float *>(x), shrink(row),
                         shrink(kg), (int)rows, (int)g.k, out, (int)rows_pad, (int)G.kp, G.blk, plane);
  };
  split(g.a, mp.a_row, mp.a_k, g.m, g.a_kfast, a3, G.mp, G.plane_a);
  split(g.b, mp.b_row, mp.b_k, g.n, g.b_kfast, b3, G.np, G.plane_b);
  const B3Params p = b3_product(g, G, a3, b3, s);
  hipLaunchKernelGGL(k_splitk_reduce_gather, dim3((unsigned)((g.m + 63) / 64), (unsigned)((g.n + 63) / 64)), dim3(256), 0,
                     s, p.part, (int)G.nz, (int)g.m, (int)g.n, shrink(mp.c_row), shrink(mp.c_col),
                     static_cast<float *>(g.c), g.alpha_re, g.beta_zero ? 1 : 0);
  return XT_HIP_OK(hipGetLastError()) ? 0 : TALSH_FAILURE;
}

int launch_gemm_gather(const GemmArgs &args, const GatherMaps &mp, void *ws, size_t ws_bytes, hipStream_t s)
{
  GemmArgs g = args;
  if (gemm_uses_split3(g)) return TALSH_NOT_IMPLEMENTED;
  if (g.m == 0 || g.n == 0) return 0;
  if (g.k == 0 && !g.beta_zero) return 0;  // empty contraction leaves C unchanged
  const GatherGroup *grp[6] = {&mp.a_row, &mp.a_k, &mp.b_row, &mp.b_k, &mp.c_row, &mp.c_col};
  const size_t want[6] = {g.m, g.k, g.n, g.k, g.m, g.n};
  for (int t = 0; t < 6; ++t) {
    if (grp[t]->nd < 0 || grp[t]->nd > kGatherMaxDims) return TALSH_INVALID_ARGS;
    size_t count = 1;
    for (int j = 0; j < grp[t]->nd; ++j) {
      if (grp[t]->ext[j] < 1 || grp[t]->str[j] < 0) return TALSH_INVALID_ARGS;
      count *= (size_t)grp[t]->ext[j];
    }
    if (count != want[t]) return TALSH_INVALID_ARGS;
    if (count > INT32_MAX && grp[t]->nd > 1) return TALSH_LIMIT_EXCEEDED;  // digits are taken in 32 bits
  }
  const int es = kind_size(g.kind);
  Product q = product_of(g);
  auto &p = q.p;
  p.a_row = dev_group(mp.a_row);
  p.a_k = dev_group(mp.a_k);
  p.b_row = dev_group(mp.b_row);
  p.b_k = dev_group(mp.b_k);
  p.c_row = dev_group(mp.c_row);
  p.c_col = dev_group(mp.c_col);
  for (const GatherGroup *x : grp)
    if (x->nd > kSmallDims) q.mode = kTabLong;
  if (lane_offsets_fit(p.a_row, p.a_k, p.m, es) && lane_offsets_fit(p.b_row, p.b_k, p.n, es) &&
      gather_uniform_k(g.kind, mp))
    q.mode = gather_vec_loads(es, g.a_kfast, mp.a_row, mp.a_k, g.k) && gather_vec_loads(es, g.b_kfast, mp.b_row, mp.b_k, g.k)
                 ? kVec : kUni;
  const int tile = resolved_tile(g);
  // write along the columns: they should hold C's stride-1 index
  if (mp.c_row.nd > 0 && mp.c_row.str[0] == 1 && !(mp.c_col.nd > 0 && mp.c_col.str[0] == 1)) exchange(q, g);
  return launch_product(q, g, tile, ws, ws_bytes, s);
}

}  // namespace xt
