// Multi-panel f32 chain GEMM on the matrix cores, C = A B (alpha 1, beta 0), with the
// matrixmultiply 0.3.8 order of the reference (src/linalg.rs:56-184): per C element a fused chain
// over each KC = 256 panel of k, started from 0, and the panels folded in order,
// C = fma(1, chain_p, C) with C = 0 before the first panel. It serves the three GEMMs of the
// asymmetric calibration target W* = ((W M') U^T) U (src/engine.rs:737-755), where k = n and the
// output is as wide as k, so the output tiles alone fill the GPU and no panel runs apart from the
// others: each workgroup folds the panels of its tile in registers and writes C once. The evaluation's
// products (proxy loss, held-out error) take the same tiles and reduce them where they are.
//
// Chains: v_mfma_f32_32x32x1_2b_f32 (K = 1, one rounding per product, bit-identical to fmaf), as in
// the repair gradient and the lazy update. Tile 128 x 128, 8 waves (wave w: rows 32 (w & 3) .. +31,
// columns 64 (w >> 2) .. +63); 32-k stages filled with global_load_lds_dwordx4 into a ring of three
// (two stages in flight behind the one being multiplied), the stage layout and load plan of the
// lazy update's 128 x 128 tile.
//
// Triangular B (the factor U is upper triangular):
//   TRI_UPPER (B = U, B[k][j] = 0 for k > j): every product past column j of the tile is
//   fma(a, 0, c) = c exactly, so the tile stops at k = its last column + 1; the panels it skips are
//   all-zero chains (+0), and C + (+0) = C.
//   TRI_LOWER (B = U^T, B[k][j] = 0 for k < j): panels that end before the tile's first column hold
//   only zero products; their chains are +0 and fold into C = +0, so the tile starts at the panel
//   holding its first column, where the leading zero products leave the chain at +0.
// Both are exact for finite A; an infinite or NaN entry of A inside a skipped zero block would
// make the reference's chain NaN there and not this one.
#include <algorithm>

#include "cdclq_dev.h"
#include "kernels.h"

namespace cdclq {
namespace {

typedef float v32f __attribute__((ext_vector_type(32)));

constexpr int TM = 128, TN = 128, SK = 32, NBUF = 3;
constexpr int STAGE = SK * TM + SK * TN;  // floats per stage: A [128 rows][8 slots][4], B [32 k][128 cols]
constexpr int LPW = STAGE / 512 / 4;      // 1 KB loads per wave and stage (4: two of A, two of B)
// tiles per XCD block: 4 row tiles x 8 column tiles run together on one XCD and share their A and B
// stages through its L2
constexpr int XB_R = 4, XB_C = 8, XB = XB_R * XB_C;

__device__ __forceinline__ v32f mfma32(float a, float b, v32f c) {
  return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, c, 0, 0, 0);
}

// The 128 x 128 tile at (r0, cb): c = the chains of A B over the panels of [kbeg, kend), folded in
// panel order (kend > kbeg, whole 32-k stages). The wave's register r holds row r0 + 32 (wv & 3) +
// tile_row(r) and column cb + 64 (wv >> 2) + tile_col(r). BT: B is given transposed (n rows of k,
// row stride ldb); its stage then has the layout of A's and a lane reads 4 k of its column at once.
__device__ __forceinline__ int tile_row(int r, int lane) { return (r & 3) + 8 * ((r & 15) >> 2) + 4 * (lane >> 5); }
__device__ __forceinline__ int tile_col(int r, int lane) { return 32 * (r >> 4) + (lane & 31); }

template <bool BT>
__device__ __forceinline__ void chain_tile(float (&R)[NBUF][STAGE], int m, int n, int kbeg, int kend,
                                           const float* __restrict__ A, long lda, const float* __restrict__ B,
                                           long ldb, int r0, int cb, float (&c)[32]) {
  const int nst = (kend - kbeg) / SK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wv & 3, wc = wv >> 2;
  // per-lane source offsets (relative to A + r0 * lda + ks and B + ks * ldb, BT: B + cb * ldb + ks):
  // loads 0..15 fill the A stage (8 rows each, k-quad (lane & 7) ^ (row & 7) into slot lane & 7),
  // loads 16..31 the B stage (2 k rows each, BT: 8 columns each like A's rows); rows past m and
  // columns past n read clamped addresses whose values only reach outputs that are never used
  long off[LPW];
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int ins = wv + 8 * q, rl = 8 * (ins & 15) + (lane >> 3);
    if (q < 2)
      off[q] = (min(r0 + rl, m - 1) - r0) * lda + 4 * ((lane & 7) ^ (rl & 7));
    else if (BT)
      off[q] = (min(cb + rl, n - 1) - cb) * ldb + 4 * ((lane & 7) ^ (rl & 7));
    else
      off[q] = (2 * (ins - 16) + (lane >> 5)) * ldb + min(cb + 4 * (lane & 31), n - 4);
  }
  const uint32_t lds0 = lds_offset(&R[0][0]);
  const float* a_base = A + (long)r0 * lda;
  const float* b_base = BT ? B + (long)cb * ldb : B;
  int fi = 0;  // stages issued
  auto issue = [&]() {
    if (fi >= nst) return;
    const uint32_t buf = lds0 + (uint32_t)((fi % NBUF) * STAGE * 4);
    const int ks = kbeg + fi * SK;
    const float* ea = a_base + ks;
    const float* hb = BT ? b_base + ks : b_base + (long)ks * ldb;
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
      const int ins = wv + 8 * q;
      dma16_untracked((q < 2 ? ea : hb) + off[q], buf + 1024u * (uint32_t)ins);
    }
    ++fi;
  };
  issue();
  issue();
  const int er = 32 * wr + (lane & 31), cl = 64 * wc + lane;
  v32f acc = {};
#pragma unroll
  for (int r = 0; r < 32; ++r) c[r] = 0.0f;
  for (int fc = 0; fc < nst; ++fc) {
    // this wave's part of stage fc has landed once at most the next stage's loads are outstanding
    if (fi - fc >= 2)
      wait_vmcnt<LPW>();
    else
      wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();  // all parts of stage fc visible; every read of stage fc - 1 done
    issue();                       // stage fc + 2, into the slot of stage fc - 1
    const float* buf = &R[fc % NBUF][0];
    const float* es = buf + 32 * er;
    const float* hs = buf + SK * TM + (BT ? 32 * cl : cl);
#pragma unroll
    for (int q = 0; q < SK / 4; ++q) {
      const float4 a = *reinterpret_cast<const float4*>(es + 4 * (q ^ (er & 7)));
      float4 b;
      if (BT) {
        b = *reinterpret_cast<const float4*>(hs + 4 * (q ^ (cl & 7)));
      } else {
        b.x = hs[(4 * q + 0) * TN];
        b.y = hs[(4 * q + 1) * TN];
        b.z = hs[(4 * q + 2) * TN];
        b.w = hs[(4 * q + 3) * TN];
      }
      acc = mfma32(a.x, b.x, acc);
      acc = mfma32(a.y, b.y, acc);
      acc = mfma32(a.z, b.z, acc);
      acc = mfma32(a.w, b.w, acc);
    }
    const int knext = kbeg + (fc + 1) * SK;
    if (knext % CDCLQ_KC == 0 || knext == kend) {  // a panel (or the tile's k range) ends here
#pragma unroll
      for (int r = 0; r < 32; ++r) c[r] = __builtin_fmaf(1.0f, acc[r], c[r]);
      acc = v32f{};
    }
  }
}

// Tile of workgroup b: it runs on XCD b % 8. Slot i = b / 8 of an XCD belongs to block (i / 32) * 8 +
// xcd; a block is 4 x 8 tiles, row tiles outer. False for an empty slot.
__device__ __forceinline__ bool tile_of(int m, int n, int* r0, int* cb) {
  const int ntr = (m + TM - 1) / TM, ntc = (n + TN - 1) / TN;
  const int nbc = (ntc + XB_C - 1) / XB_C;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int blk = (slot / XB) * 8 + xcd, pos = slot % XB;
  const int tr = (blk / nbc) * XB_R + pos / XB_C, tc = (blk % nbc) * XB_C + pos % XB_C;
  *r0 = tr * TM;
  *cb = tc * TN;
  return tr < ntr && tc < ntc;
}

template <int TRI>
__global__ __launch_bounds__(512) void k_chain_gemm_tiles(int m, int n, int k, const float* __restrict__ A, long lda,
                                                          const float* __restrict__ B, long ldb, float* __restrict__ C,
                                                          long ldc) {
  __shared__ float R[NBUF][STAGE];
  int r0, cb;
  if (!tile_of(m, n, &r0, &cb)) return;
  int kbeg = 0, kend = k;
  if (TRI == 1) kend = min(k, cb + TN);
  if (TRI == 2) kbeg = (cb / CDCLQ_KC) * CDCLQ_KC;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (kend - kbeg < SK) {  // no nonzero product reaches this tile (only possible with TRI): C = +0
    for (int e = tid; e < TM * TN; e += 512) {
      const int row = r0 + e / TN, col = cb + e % TN;
      if (row < m && col < n) C[(long)row * ldc + col] = 0.0f;
    }
    return;
  }
  float c[32];
  chain_tile<false>(R, m, n, kbeg, kend, A, lda, B, ldb, r0, cb, c);
#pragma unroll
  for (int r = 0; r < 32; ++r) {
    const int row = r0 + 32 * (wv & 3) + tile_row(r, lane), col = cb + 64 * (wv >> 2) + tile_col(r, lane);
    if (row < m && col < n) C[(long)row * ldc + col] = c[r];
  }
}

// The evaluation's error sums (f64), without their products going through memory. Each workgroup
// reduces its tile's two sums into partial[2 b], partial[2 b + 1] (zero for an empty slot);
// k_sum_pairs adds the workgroups' in a fixed order.
__device__ __forceinline__ void reduce_pair(double s0, double s1, double* red, double* __restrict__ partial) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s0 += __shfl_xor(s0, o, 64);
    s1 += __shfl_xor(s1, o, 64);
  }
  if ((tid & 63) == 0) {
    red[2 * (tid >> 6)] = s0;
    red[2 * (tid >> 6) + 1] = s1;
  }
  __syncthreads();
  if (tid < 2) {
    double s = 0.0;
    for (int w = 0; w < 8; ++w) s += red[2 * w + tid];
    partial[2 * blockIdx.x + tid] = s;
  }
}

// bench::rel_err (src/bench.rs:106-121): sums of (o1 - o2)^2 and o1^2 over o1 = W X^T, o2 = W_hat
// X~^T, both k wide and row-major: two transposed-B tiles one after the other in the same registers'
// layout. 2048 x 2048 over 4096 tokens: this and the proxy loss's product took 1743 us as VALU chains
// whose results went to memory and back, and take 696 and 191 us here (99 and 90 TFLOP/s).
__global__ __launch_bounds__(512) void k_rel_err_tiles(int m, int n, int k, const float* __restrict__ W,
                                                       const float* __restrict__ W_hat, long ldw,
                                                       const float* __restrict__ X, const float* __restrict__ Xt,
                                                       long ldx, double* __restrict__ partial) {
  __shared__ float R[NBUF][STAGE];
  __shared__ double red[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int r0, cb;
  double num = 0.0, den = 0.0;
  if (tile_of(m, n, &r0, &cb)) {
    float o1[32], o2[32];
    chain_tile<true>(R, m, n, 0, k, W, ldw, X, ldx, r0, cb, o1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the ring is free again
    chain_tile<true>(R, m, n, 0, k, W_hat, ldw, Xt, ldx, r0, cb, o2);
#pragma unroll
    for (int r = 0; r < 32; ++r) {
      const int row = r0 + 32 * (wv & 3) + tile_row(r, lane), col = cb + 64 * (wv >> 2) + tile_col(r, lane);
      if (row < m && col < n) {
        const double d = (double)(o1[r] - o2[r]);
        num += d * d;
        den += (double)o1[r] * (double)o1[r];
      }
    }
  }
  reduce_pair(num, den, red, partial);
}

// engine::proxy_loss (src/engine.rs:808-815): the sum of e (e H) in f64; E m x k (row stride lde, its
// first n columns the residual).
__global__ __launch_bounds__(512) void k_proxy_tiles(int m, int n, int k, const float* __restrict__ E, long lde,
                                                     const float* __restrict__ H, long ldh,
                                                     double* __restrict__ partial) {
  __shared__ float R[NBUF][STAGE];
  __shared__ double red[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int r0, cb;
  double s = 0.0;
  if (tile_of(m, n, &r0, &cb)) {
    float c[32];
    chain_tile<false>(R, m, n, 0, k, E, lde, H, ldh, r0, cb, c);
#pragma unroll
    for (int r = 0; r < 32; ++r) {
      const int row = r0 + 32 * (wv & 3) + tile_row(r, lane), col = cb + 64 * (wv >> 2) + tile_col(r, lane);
      if (row < m && col < n) s += (double)E[(long)row * lde + col] * (double)c[r];
    }
  }
  reduce_pair(s, 0.0, red, partial);
}

__global__ __launch_bounds__(256) void k_sum_pairs(int count, const double* __restrict__ partial,
                                                   double* __restrict__ out) {
  __shared__ double red[2][256];
  const int tid = threadIdx.x;
  double s0 = 0.0, s1 = 0.0;
  for (int i = tid; i < count; i += 256) {
    s0 += partial[2 * (long)i];
    s1 += partial[2 * (long)i + 1];
  }
  red[0][tid] = s0;
  red[1][tid] = s1;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (tid < o) {
      red[0][tid] += red[0][tid + o];
      red[1][tid] += red[1][tid + o];
    }
    __syncthreads();
  }
  if (tid < 2) out[tid] = red[tid][0];
}

// rows x n with stride n into rows_out rows of ld floats, zero elsewhere
__global__ __launch_bounds__(256) void k_pad_rows(long rows, int n, long rows_out, int ld,
                                                  const float* __restrict__ src, float* __restrict__ dst) {
  const long count = rows_out * ld;
  for (long idx = (long)blockIdx.x * 256 + threadIdx.x; idx < count; idx += (long)gridDim.x * 256) {
    const long r = idx / ld;
    const int c = (int)(idx % ld);
    dst[idx] = r < rows && c < n ? src[r * n + c] : 0.0f;
  }
}

// dst = src^T for an n x n matrix: 64 x 64 tiles through LDS (padded rows), coalesced both ways.
__global__ __launch_bounds__(256) void k_transpose(int n, const float* __restrict__ src, float* __restrict__ dst) {
  __shared__ float t[64][65];
  const int bi = blockIdx.y * 64, bj = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int i = bi + r, j = bj + tx;
    if (i < n && j < n) t[r][tx] = src[(long)i * n + j];
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int i = bj + r, j = bi + tx;  // dst[i][j] = src[j][i]
    if (i < n && j < n) dst[(long)i * n + j] = t[tx][r];
  }
}

}  // namespace

hipError_t transpose_f32(hipStream_t st, int n, const float* src, float* dst) {
  if (n <= 0) return hipSuccess;
  const unsigned nb = (unsigned)((n + 63) / 64);
  hipLaunchKernelGGL(k_transpose, dim3(nb, nb), dim3(256), 0, st, n, src, dst);
  return hipGetLastError();
}

bool chain_gemm_tiles_ok(int m, int n, int k, const float* A, long lda, const float* B, long ldb, const float* C,
                         long ldc) {
  return m > 0 && n >= 4 && k > 0 && k % SK == 0 && n % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && lda >= k &&
         ldb >= n && ldc >= n && (uintptr_t)A % 16 == 0 && (uintptr_t)B % 16 == 0 && (uintptr_t)C % 4 == 0 &&
         (long)m * lda < (1L << 31) && (long)k * ldb < (1L << 31);
}

// workgroups over an m x n output: every XCD gets the same number of block slots
static long tile_grid(long m, long n) {
  const long ntr = (m + TM - 1) / TM, ntc = (n + TN - 1) / TN;
  const long nblk = ((ntr + XB_R - 1) / XB_R) * ((ntc + XB_C - 1) / XB_C);
  return (nblk + 7) / 8 * 8 * XB;
}

size_t eval_partials(size_t m, size_t n) { return 2 * (size_t)tile_grid((long)m, (long)n); }

bool eval_operand_ok(size_t n, const float* p) { return n % SK == 0 && (uintptr_t)p % 16 == 0; }

hipError_t pad_rows(hipStream_t st, long rows, int n, long rows_out, int ld, const float* src, float* dst) {
  const long count = rows_out * ld;
  if (count <= 0) return hipSuccess;
  const unsigned grid = (unsigned)std::min<long>((count + 255) / 256, 1L << 20);
  hipLaunchKernelGGL(k_pad_rows, dim3(grid), dim3(256), 0, st, rows, n, rows_out, ld, src, dst);
  return hipGetLastError();
}

hipError_t rel_err_sums(hipStream_t st, int m, int n, int k, const float* W, const float* W_hat, long ldw,
                        const float* X, const float* Xt, long ldx, double* partial, double* out) {
  const long grid = tile_grid(m, n);
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rel_err_tiles, dim3((unsigned)grid), dim3(512), 0, st, m, n, k, W, W_hat, ldw, X, Xt, ldx,
                     partial);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(256), 0, st, (int)grid, partial, out);
  return hipGetLastError();
}

hipError_t proxy_sum(hipStream_t st, int m, int n, int k, const float* E, long lde, const float* H, long ldh,
                     double* partial, double* out) {
  const long grid = tile_grid(m, n);
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_proxy_tiles, dim3((unsigned)grid), dim3(512), 0, st, m, n, k, E, lde, H, ldh, partial);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(256), 0, st, (int)grid, partial, out);
  return hipGetLastError();
}

hipError_t chain_gemm_tiles(hipStream_t st, int m, int n, int k, const float* A, long lda, const float* B, long ldb,
                            float* C, long ldc, int tri) {
  const long grid = tile_grid(m, n);
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  if (tri == 1)
    hipLaunchKernelGGL(k_chain_gemm_tiles<1>, dim3((unsigned)grid), dim3(512), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  else if (tri == 2)
    hipLaunchKernelGGL(k_chain_gemm_tiles<2>, dim3((unsigned)grid), dim3(512), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  else
    hipLaunchKernelGGL(k_chain_gemm_tiles<0>, dim3((unsigned)grid), dim3(512), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  return hipGetLastError();
}

}  // namespace cdclq
