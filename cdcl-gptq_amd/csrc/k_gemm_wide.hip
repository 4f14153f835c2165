// Multi-panel f32 chain GEMM on the matrix cores, C = A B (alpha 1, beta 0), with the
// matrixmultiply 0.3.8 order of the reference (src/linalg.rs:56-184): per C element a fused chain
// over each KC = 256 panel of k, started from 0, and the panels folded in order,
// C = fma(1, chain_p, C) with C = 0 before the first panel. It serves the three GEMMs of the
// asymmetric calibration target W* = ((W M') U^T) U (src/engine.rs:737-755), where k = n and the
// output is as wide as k, so the output tiles alone fill the GPU and no panel runs apart from the
// others: each workgroup folds the panels of its tile in registers and writes C once. The evaluation's
// products (proxy loss, held-out error) take the same tiles and reduce them where they are.
//
// Chains: the 128 x 128 tiles of mfma_tile.h, 4 waves of 32 rows x 128 columns, 32-k stages filled with
// global_load_lds_dwordx4 into a ring of two (64 KB, two workgroups per CU), an operand group read
// while the one before it is multiplied and each stage's barrier before the last of its groups.
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
#include "mfma_tile.h"

namespace cdclq {
namespace {

constexpr int TM = 128, TN = 128, SK = TILE_SK;
// tiles per XCD block: 4 row tiles x 8 column tiles run together on one XCD and share their A and B
// stages through its L2
constexpr int XB_R = 4, XB_C = 8, XB = XB_R * XB_C;

typedef MfmaTile<4, 1, 1, 4> Dense;         // B k x n
typedef MfmaTile<4, 1, 1, 2, true> DenseT;  // B given as n x k: 128 x 64, two results' registers at once

// The tile at (r0, cb): c[b][r] = the chains of A B over the panels of [kbeg, kend), folded in panel
// order (kend > kbeg, whole stages), at row r0 + T::row(0, r), column cb + T::col(b). BT: B is n x k. The
// ring may be used again once every wave has returned.
template <class T, bool BT>
__device__ __forceinline__ void chain_tile(float (&R)[2][T::STAGE], int m, int n, int kbeg, int kend,
                                           const float* __restrict__ A, long lda, const float* __restrict__ B,
                                           long ldb, int r0, int cb, tile_v16f (&c)[T::FC]) {
  static_assert(T::FR == 1 && T::WC == 1 && T::ROWS == TM, "a row block and every column per wave");
  const int nst = (kend - kbeg) / SK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  long off[T::NL];
  T::offsets(wv, lane, m - r0, lda, n - cb, ldb, off);
  const uint32_t lds0 = lds_offset(&R[0][0]);
  const float* a = A + (long)r0 * lda + kbeg;
  const float* b = BT ? B + (long)cb * ldb + kbeg : B + (long)kbeg * ldb + cb;
  const long bstep = BT ? SK : (long)SK * ldb;
  int fi = 0;  // stages issued
  auto issue = [&]() {
    if (fi >= nst) return;
    T::load_stage(a + (long)fi * SK, b + fi * bstep, off, lds0 + (uint32_t)((fi & 1) * T::STAGE * 4), wv);
    ++fi;
  };
  issue();
  issue();
  typename T::Acc acc;
  T::clear(acc);
#pragma unroll
  for (int q = 0; q < T::FC; ++q) c[q] = tile_v16f{};
  wait_vmcnt<0>();
  asm volatile("s_barrier" ::: "memory");
  typename T::Ops cur = T::read(&R[0][0], 0, wv, 0, lane);
  for (int fc = 0; fc < nst; ++fc) {
#pragma unroll
    for (int g = 0; g < TILE_G - 1; ++g) {
      const typename T::Ops nxt = T::read(&R[fc & 1][0], g + 1, wv, 0, lane);
      __builtin_amdgcn_sched_barrier(0);  // the next group's reads are issued before this group's products
      T::arrange(cur);
      T::mul(cur, acc);
      cur = nxt;
    }
    __builtin_amdgcn_sched_barrier(0);
    // this wave's part of the next stage has landed and its reads of this one have returned; the
    // barrier publishes the one and frees the other for the stage after next
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue();
    const typename T::Ops nxt = T::read(&R[(fc + 1) & 1][0], 0, wv, 0, lane);  // (after the last stage: not used)
    __builtin_amdgcn_sched_barrier(0);
    T::arrange(cur);
    T::mul(cur, acc);
    cur = nxt;
    const int knext = kbeg + (fc + 1) * SK;
    if (knext % CDCLQ_KC == 0 || knext == kend) {  // a panel (or the tile's k range) ends here
#pragma unroll
      for (int q = 0; q < T::FC; ++q) {
#pragma unroll
        for (int r = 0; r < 16; ++r) c[q][r] = __builtin_fmaf(1.0f, acc.c[0][q][r], c[q][r]);
      }
      T::clear(acc);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// Tile of workgroup b: it runs on XCD b % 8. Slot i = b / 8 of an XCD belongs to block (i / 32) * 8 +
// xcd; a block is 4 x 8 tiles, the row blocks of a column block following one another, and the
// column blocks go from the last to the first with `rev`: the longest tiles of a triangular B start
// first, in every XCD (row blocks outermost left the long tiles for the end: 1.08 ms against 0.71 for
// 4096 x 4096 x 4096). False for an empty slot.
template <class T>
__device__ __forceinline__ bool tile_of(int m, int n, int* r0, int* cb, bool rev = false) {
  const int ntr = (m + TM - 1) / TM, ntc = (n + T::COLS - 1) / T::COLS;
  const int nbr = (ntr + XB_R - 1) / XB_R, nbc = (ntc + XB_C - 1) / XB_C;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int blk = (slot / XB) * 8 + xcd, pos = slot % XB;
  const int bc = blk / nbr;
  if (bc >= nbc) return false;
  const int tr = (blk % nbr) * XB_R + pos / XB_C, tc = (rev ? nbc - 1 - bc : bc) * XB_C + pos % XB_C;
  *r0 = tr * TM;
  *cb = tc * T::COLS;
  return tr < ntr && tc < ntc;
}

template <int TRI>
__global__ __launch_bounds__(256) void k_chain_gemm_tiles(int m, int n, int k, const float* __restrict__ A, long lda,
                                                          const float* __restrict__ B, long ldb, float* __restrict__ C,
                                                          long ldc) {
  __shared__ __align__(16) float R[2][Dense::STAGE];
  int r0, cb;
  if (!tile_of<Dense>(m, n, &r0, &cb, TRI == 1)) return;
  int kbeg = 0, kend = k;
  if (TRI == 1) kend = min(k, cb + TN);
  if (TRI == 2) kbeg = (cb / CDCLQ_KC) * CDCLQ_KC;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (kend - kbeg < SK) {  // no nonzero product reaches this tile (only possible with TRI): C = +0
    for (int e = tid; e < TM * TN; e += 256) {
      const int row = r0 + e / TN, col = cb + e % TN;
      if (row < m && col < n) C[(long)row * ldc + col] = 0.0f;
    }
    return;
  }
  tile_v16f c[4];
  chain_tile<Dense, false>(R, m, n, kbeg, kend, A, lda, B, ldb, r0, cb, c);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = r0 + Dense::row(0, r, wv, lane), col = cb + Dense::col(0, lane);
    if (row < m && col < n) {  // (n % 4 == 0: the lane's four columns are all in or all out)
#pragma unroll
      for (int b = 0; b < 4; ++b) C[(long)row * ldc + col + b] = c[b][r];
    }
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
    for (int w = 0; w < 4; ++w) s += red[2 * w + tid];
    partial[2 * blockIdx.x + tid] = s;
  }
}

// bench::rel_err (src/bench.rs:106-121): sums of (o1 - o2)^2 and o1^2 over o1 = W X^T, o2 = W_hat
// X~^T, both k wide and row-major: two transposed-B tiles one after the other in the same registers'
// layout. 2048 x 2048 over 4096 tokens: this and the proxy loss's product took 1743 us as VALU chains
// whose results went to memory and back, and take 669 and 160 us here (103 and 107 TFLOP/s).
__global__ __launch_bounds__(256, 2) void k_rel_err_tiles(int m, int n, int k, const float* __restrict__ W,
                                                       const float* __restrict__ W_hat, long ldw,
                                                       const float* __restrict__ X, const float* __restrict__ Xt,
                                                       long ldx, double* __restrict__ partial) {
  __shared__ __align__(16) float R[2][DenseT::STAGE];
  __shared__ double red[8];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int r0, cb;
  double num = 0.0, den = 0.0;
  if (tile_of<DenseT>(m, n, &r0, &cb)) {
    tile_v16f o1[DenseT::FC], o2[DenseT::FC];
    chain_tile<DenseT, true>(R, m, n, 0, k, W, ldw, X, ldx, r0, cb, o1);
    asm volatile("s_barrier" ::: "memory");  // the ring is free again
    chain_tile<DenseT, true>(R, m, n, 0, k, W_hat, ldw, Xt, ldx, r0, cb, o2);
#pragma unroll
    for (int b = 0; b < DenseT::FC; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = r0 + DenseT::row(0, r, wv, lane), col = cb + DenseT::col(0, lane, b);
        if (row < m && col < n) {
          const double d = (double)(o1[b][r] - o2[b][r]);
          num += d * d;
          den += (double)o1[b][r] * (double)o1[b][r];
        }
      }
  }
  reduce_pair(num, den, red, partial);
}

// engine::proxy_loss (src/engine.rs:808-815): the sum of e (e H) in f64 over the residual's n columns; E
// m x k (row stride lde) and H k x ldh are zero past them. Padding columns stay out of the sum: an infinite
// residual times their zeros is NaN.
__global__ __launch_bounds__(256, 2) void k_proxy_tiles(int m, int n, int k, const float* __restrict__ E, long lde,
                                                     const float* __restrict__ H, long ldh,
                                                     double* __restrict__ partial) {
  __shared__ __align__(16) float R[2][Dense::STAGE];
  __shared__ double red[8];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int r0, cb;
  double s = 0.0;
  if (tile_of<Dense>(m, n, &r0, &cb)) {
    tile_v16f c[4];
    chain_tile<Dense, false>(R, m, (int)ldh, 0, k, E, lde, H, ldh, r0, cb, c);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = r0 + Dense::row(0, r, wv, lane), col = cb + Dense::col(0, lane);
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (row < m && col + b < n) s += (double)E[(long)row * lde + col + b] * (double)c[b][r];
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

// The most workgroups of 256 a launch may have: 2^32 work-items wrap to a smaller launch without an error.
constexpr long MAX_GRID = (1L << 24) - 1;

// workgroups over an m x n output: every XCD gets the same number of block slots
template <class T>
static long tile_grid(long m, long n) {
  const long ntr = (m + TM - 1) / TM, ntc = (n + T::COLS - 1) / T::COLS;
  const long nblk = ((ntr + XB_R - 1) / XB_R) * ((ntc + XB_C - 1) / XB_C);
  return (nblk + 7) / 8 * 8 * XB;
}

size_t eval_partials(size_t m, size_t n) { return 2 * (size_t)tile_grid<DenseT>((long)m, (long)n); }  // (the finer grid)

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
  const long grid = tile_grid<DenseT>(m, n);
  if (grid > MAX_GRID) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rel_err_tiles, dim3((unsigned)grid), dim3(256), 0, st, m, n, k, W, W_hat, ldw, X, Xt, ldx,
                     partial);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(256), 0, st, (int)grid, partial, out);
  return hipGetLastError();
}

hipError_t proxy_sum(hipStream_t st, int m, int n, int k, const float* E, long lde, const float* H, long ldh,
                     double* partial, double* out) {
  const long grid = tile_grid<Dense>(m, n);
  if (grid > MAX_GRID) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_proxy_tiles, dim3((unsigned)grid), dim3(256), 0, st, m, n, k, E, lde, H, ldh, partial);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(256), 0, st, (int)grid, partial, out);
  return hipGetLastError();
}

hipError_t chain_gemm_tiles(hipStream_t st, int m, int n, int k, const float* A, long lda, const float* B, long ldb,
                            float* C, long ldc, int tri) {
  const long grid = tile_grid<Dense>(m, n);
  if (grid > MAX_GRID) return hipErrorInvalidValue;
  if (tri == 1)
    hipLaunchKernelGGL(k_chain_gemm_tiles<1>, dim3((unsigned)grid), dim3(256), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  else if (tri == 2)
    hipLaunchKernelGGL(k_chain_gemm_tiles<2>, dim3((unsigned)grid), dim3(256), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  else
    hipLaunchKernelGGL(k_chain_gemm_tiles<0>, dim3((unsigned)grid), dim3(256), 0, st, m, n, k, A, lda, B, ldb, C, ldc);
  return hipGetLastError();
}

}  // namespace cdclq
