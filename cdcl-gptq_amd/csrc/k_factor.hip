// f64 factorisation kernels: U with H^-1 = U^T U (src/linalg.rs:200-375, src/engine.rs:320-342).
//
// Blocking follows the reference's NB = 96 block columns because the block boundaries fix the
// floating-point operation sequence of every element:
//   * diagonal block: unblocked left-looking Cholesky with separate multiply/subtract roundings;
//   * panel solve below it: for each column j of the block, s = a_ij - sum_t x_t l_jt in t order;
//   * trailing update: a_ij = fma(-1, chain_t(p_it p_jt), a_ij) per block (k_gemm.hip, lower tiles);
//   * inverse of every diagonal block by columns (mul/add roundings), then per block row two
//     chained GEMMs (k_gemm.hip).
// The panel solve and the blocks' inverse give a row several lanes (its columns interleaved over
// them): column t is finalised at step t and immediately subtracted from every later column, which
// performs the reference's per-element subtraction sequence in the same order.
#include <algorithm>

#include "cdclq_dev.h"
#include "kernels.h"

namespace cdclq {
namespace {

constexpr int NBC = 96;  // src/linalg.rs:202, :285

// the wave's LDS accesses are done; its stores to memory stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// hp = perm(H) in f64, dead diagonal -> 1, + damp on the diagonal; h32 = (f32)hp; a = flip(hp).
// h32 is ld x ld, zero past n. Grid-stride: the padded matrix of n = 65535 has 2^32 elements, one
// more than a launch may have work-items.
__global__ __launch_bounds__(256) void k_build_flipped(int n, int ld, const float* __restrict__ h,
                                                       const uint32_t* __restrict__ perm, double damp_val,
                                                       double* __restrict__ a, float* __restrict__ h32) {
  const long count = (long)ld * ld;
  for (long idx = (long)blockIdx.x * 256 + threadIdx.x; idx < count; idx += (long)gridDim.x * 256) {
    const int p = (int)(idx / ld), q = (int)(idx % ld);
    if (p >= n || q >= n) {
      h32[idx] = 0.0f;
      continue;
    }
    double v = (double)h[(long)perm[p] * n + perm[q]];
    if (p == q) {
      if (v == 0.0) v = 1.0;
      v = v + damp_val;
    }
    h32[idx] = (float)v;
    a[(long)(n - 1 - p) * n + (n - 1 - q)] = v;
  }
}

__global__ __launch_bounds__(256) void k_build_flipped_f64(int n, const double* __restrict__ h, double* __restrict__ a) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  const long nn = (long)n * n;
  if (idx >= nn) return;
  a[idx] = h[nn - 1 - idx];
}

// Unblocked factorisation of the diagonal block (src/linalg.rs:209-229). The reference works by
// columns (left-looking): d = a_jj - sum_{t<j} l_jt l_jt, l_jj = sqrt(d), then
// l_ij = (a_ij - sum_{t<j} l_it l_jt) / l_jj, every term a separate multiply and subtract in t
// order. Applying the subtraction of column t to the whole trailing triangle as soon as column t
// is final (right-looking) performs exactly the same operations on every element in the same
// order, with the trailing triangle updated in parallel.
//
// The block lies in LDS and is taken 8 columns at a time. A chain of square root, division and
// broadcast per column sets the time, so these run without LDS: wavefronts 0 and 1 hold a row of the
// open 8 columns per lane (lanes 0-7 of both the 8 diagonal rows, so that each has the pivots and the
// factors of the later columns in its own lanes), and a column's pivot and factors are lane reads.
// While they apply the last 8 columns of L to the next 8 and factor those, wavefronts 2, 3, 6 and 7
// (the SIMDs without 0 and 1) apply the last 8 to the columns beyond, a 4 x 4 tile per lane: one barrier
// per 8 columns. A failing pivot is recorded (the first one) and reported at the end; the remaining
// steps run on with values that are discarded with the error. Rows and columns past kb are those of
// the unit matrix.
// 96 columns: 26 us (one wavefront with the block in its registers and every column through LDS
// twice: 49 us).
constexpr int DW = 8;            // columns taken at a time
constexpr int DS = NBC + 2;      // row stride of the block (16-byte aligned, rows on different banks)
constexpr int DLS = NBC + 8;     // stride of a column of L

__device__ __forceinline__ double readlane_f64(double v, int l) {  // l uniform
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__global__ __launch_bounds__(512) void k_chol_diag(int n, double* __restrict__ a, int k, int kb, int* status,
                                                   double* pivot) {
  __shared__ __attribute__((aligned(16))) double A[NBC * DS];
  __shared__ __attribute__((aligned(16))) double L[2][DW * DLS];  // the last 8 columns of L
  if (*status) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  {
    constexpr int PER = NBC * NBC / 512;
    double v[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = tid + 512 * e, i = x / NBC, j = x % NBC;
      v[e] = a[(long)(k + min(i, kb - 1)) * n + k + min(j, kb - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = tid + 512 * e, i = x / NBC, j = x % NBC;
      A[i * DS + j] = (i < kb && j < kb) ? v[e] : (i == j ? 1.0 : 0.0);
    }
  }
  __syncthreads();
  const int np = (kb + DW - 1) / DW;
  int fail_t = -1;
  double fail_d = 0.0;
  for (int p = 0; p < np; ++p) {  // factors columns 8 p .. 8 p + 7
    const int c0 = DW * p;
    const double* lq = L[(p + 1) & 1];  // columns c0 - 8 .. c0 - 1
    if (wv < 2) {
      const int row = lane < DW ? c0 + lane : c0 + DW + (64 - DW) * wv + lane - DW;
      const int rr = min(row, NBC - 1);  // rows past the block: computed, never stored
      double x[DW];
#pragma unroll
      for (int j = 0; j < DW; ++j) x[j] = A[rr * DS + c0 + j];
      if (p > 0) {
#pragma unroll
        for (int t = 0; t < DW; ++t) {
          const double li = lq[t * DLS + rr];
#pragma unroll
          for (int j = 0; j < DW; ++j) x[j] = x[j] - li * lq[t * DLS + c0 + j];
        }
      }
      double* ln = L[p & 1];
      const bool own = row < NBC && (wv == 0 || lane >= DW);
#pragma unroll
      for (int t = 0; t < DW; ++t) {
        const double d = readlane_f64(x[t], t);
        const bool rec = (!(d > 0.0) || !isfinite(d)) && fail_t < 0;
        fail_d = rec ? d : fail_d;
        fail_t = rec ? c0 + t : fail_t;
        const double ltt = sqrt(d);
        x[t] = lane == t ? ltt : x[t] / ltt;
#pragma unroll
        for (int j = t + 1; j < DW; ++j) x[j] = x[j] - x[t] * readlane_f64(x[t], j);
      }
#pragma unroll
      for (int t = 0; t < DW; ++t)
        if (own) {
          ln[t * DLS + row] = x[t];
          if (row >= c0 + t && row < kb && c0 + t < kb) a[(long)(k + row) * n + k + c0 + t] = x[t];
        }
    } else if ((wv & 2) && p > 0) {  // columns c0 + 8 and later, lower 4 x 4 tiles
      const int o = c0 + DW, nt = (NBC - o) / 4;
      const int w = (wv & 1) + ((wv & 4) >> 1);
      for (int e = w * 64 + lane; e < nt / 2 * (nt + 1); e += 256) {
        const int u = e / (nt + 1), v = e % (nt + 1);  // rows u and nt - 1 - u of the triangle share a line
        const int i0 = o + 4 * (v <= u ? u : nt - 1 - u), j0 = o + 4 * (v <= u ? v : v - u - 1);
        double s[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) s[i][j] = A[(i0 + i) * DS + j0 + j];
#pragma unroll
        for (int t = 0; t < DW; ++t) {
          double li[4], lj[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            li[q] = lq[t * DLS + i0 + q];
            lj[q] = lq[t * DLS + j0 + q];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) s[i][j] = s[i][j] - li[i] * lj[j];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) A[(i0 + i) * DS + j0 + j] = s[i][j];
      }
    }
    lds_barrier();
  }
  if (tid == 0 && fail_t >= 0) {
    *status = k + fail_t + 1;
    *pivot = fail_d;
  }
}

// Triangular solves against the transposed diagonal block, a row x at a time: x_j = (a_j - sum_{t<j}
// x_t l_jt) / l_jj, every product and difference rounded separately, t ascending.
//   * k_chol_panel: the rows of A below the block (src/linalg.rs:233-241);
//   * k_trinv_diag: the inverse y of every diagonal block (src/linalg.rs:291-306), whose column c is the
//     row of x for the unit row c: y_cc = 1 / l_cc, y_ic = -(sum_{t=c}^{i-1} l_it y_tc) / l_ii. Its sums
//     are kept as they are added there (from +0, negated at the division, so that zeros keep their
//     signs); the terms t < c are zeros.
// G = 16 lanes per row: lane g of them holds columns j = 16 q + g (q < 6), so the columns still open at any
// step are spread evenly over the row's lanes. Step t: the lane holding column t divides it by l_tt
// (all lanes run the division; the others' quotients are discarded), a DPP broadcast hands the quotient
// to the row's lanes, and each lane subtracts x_t l_jt from its columns j > t. Column j thus receives
// the reference's subtractions in the reference's order (right-looking instead of a dot product per
// column), and finished columns are never touched again. The lower part of L_kk is staged in LDS
// as LP[t][g][q] = l_{G q + g, t} (zero on and above the diagonal and past the block), so a lane reads
// the factors of its columns for step t as consecutive pairs; the diagonal is staged separately.
// The step's chain (broadcast, update, division) bounds it: 20 us for a panel below a block of 96 at
// n = 4096, against 24 with four lanes per row, where the reads of 24 factors per lane and step did.
constexpr int G = 16, PQ = NBC / G;
constexpr int TRS_WAVES = 4;

template <int C>
__device__ __forceinline__ double row_bcast(double v) {  // lane C's value of every 16 lanes to the 16 lanes
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), 0x150 + C, 0xf, 0xf, false);  // row_newbcast
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x150 + C, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Step T of the solve for one lane; templated on T so that every index into the lane's columns is a
// constant. On entry `xo` is column T divided by its pivot (valid in the lanes holding column T),
// `cur` this step's factors l_{Gq+g, T} (q >= T / G) and `dn` the next pivot l_{T+1, T+1}, read from LDS
// a step ahead so that their latency hides behind the previous step. The step finalises column T,
// updates column T + 1 first and starts its division, so that the division's latency overlaps the
// step's other updates (a division started for a column past the block, T + 1 = kb, divides by the
// pivot 1 staged there and is never used).
template <bool INV, int T>
__device__ __forceinline__ void trs_step(double (&s)[PQ], const double (&cur)[PQ], double xo, double dn,
                                         int g, int kb, const double* lp0, const double* dg) {
  constexpr int qt = T / G, gt = T % G, T1 = T + 1, q1 = T1 / G;
  if (T >= kb) return;  // uniform; a real branch, which also bounds the scheduler's reach
  double nxt[PQ], dn2 = 1.0;
  if constexpr (T1 < NBC) {
    const double* lp = lp0 + (T1 * G + g) * PQ;  // LP[T + 1][g][.]
#pragma unroll
    for (int q = q1; q < PQ; ++q) nxt[q] = lp[q];
    if constexpr (T1 + 1 < NBC) dn2 = dg[T1 + 1];
  }
  const double x = row_bcast<gt>(xo);
  double up = INV ? s[qt] + x * cur[qt] : s[qt] - x * cur[qt];
  asm volatile("" : "+v"(up));  // computed in every lane, so that the select below is no branch
  const double keep = s[qt];
  const double upd = g > gt ? up : keep;
  s[qt] = g == gt ? xo : upd;
  if constexpr (T1 < NBC) {
    if constexpr (q1 != qt) s[q1] = INV ? s[q1] + x * cur[q1] : s[q1] - x * cur[q1];
    double xo1 = (INV ? -s[q1] : s[q1]) / dn;
    asm volatile("" : "+v"(xo1));  // the division starts here, before the step's other updates
#pragma unroll
    for (int q = q1 + 1; q < PQ; ++q) s[q] = INV ? s[q] + x * cur[q] : s[q] - x * cur[q];
    trs_step<INV, T1>(s, nxt, xo1, dn2, g, kb, lp0, dg);
  }
}

// stages the block of L at `l` (row stride n, kb columns) and runs the steps on s
template <bool INV>
__device__ __forceinline__ void trs_rows(const double* __restrict__ l, long n, int kb, double (&s)[PQ], double* LP,
                                         double* dg) {
  const int tid = threadIdx.x;
  {  // stage the block with all of a thread's loads in flight at once (clamped addresses)
    constexpr int PER = NBC * NBC / (64 * TRS_WAVES);
    double v[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = tid + 64 * TRS_WAVES * e, j = x / NBC, t = x % NBC;
      v[e] = l[(long)min(j, kb - 1) * n + min(t, kb - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = tid + 64 * TRS_WAVES * e, j = x / NBC, t = x % NBC;
      LP[(t * G + j % G) * PQ + j / G] = (t < j && j < kb) ? v[e] : 0.0;
      if (t == j) dg[t] = t < kb ? v[e] : 1.0;
    }
  }
  __syncthreads();
  const int g = tid & (G - 1);
  double f0[PQ];
#pragma unroll
  for (int q = 0; q < PQ; ++q) f0[q] = LP[g * PQ + q];
  trs_step<INV, 0>(s, f0, (INV ? -s[0] : s[0]) / dg[0], dg[1], g, kb, LP, dg);
}

__global__ __launch_bounds__(64 * TRS_WAVES) void k_chol_panel(int n, double* __restrict__ a, int k, int kb,
                                                               const int* status) {
  __shared__ __attribute__((aligned(16))) double LP[NBC * NBC];
  __shared__ double dg[NBC];
  if (*status) return;
  const int g = threadIdx.x & (G - 1);
  const int row = k + kb + blockIdx.x * (64 * TRS_WAVES / G) + (int)threadIdx.x / G;
  const double* src = a + (long)min(row, n - 1) * n + k;  // rows past the end: computed, never stored
  double s[PQ];
#pragma unroll
  for (int q = 0; q < PQ; ++q) s[q] = src[min(G * q + g, kb - 1)];
  trs_rows<false>(a + (long)k * n + k, n, kb, s, LP, dg);
  if (row < n) {
    double* dst = a + (long)row * n + k;
#pragma unroll
    for (int q = 0; q < PQ; ++q)
      if (G * q + g < kb) dst[G * q + g] = s[q];
  }
}

// Workgroup (x, y): columns 16 y .. 16 y + 15 of block x's inverse. 16 us for any n whose blocks fit
// the device at once (a thread per column reading L from memory at every step: 124 us).
__global__ __launch_bounds__(64 * TRS_WAVES) void k_trinv_diag(int n, const double* __restrict__ l, double* __restrict__ y,
                                                               const int* status) {
  __shared__ __attribute__((aligned(16))) double LP[NBC * NBC];
  __shared__ double dg[NBC];
  if (*status) return;
  const int s0 = blockIdx.x * NBC, w = min(NBC, n - s0);
  const int g = threadIdx.x & (G - 1), c = blockIdx.y * (64 * TRS_WAVES / G) + (int)threadIdx.x / G;
  if ((int)blockIdx.y * (64 * TRS_WAVES / G) >= w) return;
  double s[PQ];
#pragma unroll
  for (int q = 0; q < PQ; ++q) s[q] = G * q + g == c ? -1.0 : 0.0;
  trs_rows<true>(l + (long)s0 * n + s0, n, w, s, LP, dg);
  if (c < w) {
#pragma unroll
    for (int q = 0; q < PQ; ++q) {
      const int i = G * q + g;
      if (i >= c && i < w) y[(long)(s0 + i) * n + s0 + c] = s[q];
    }
  }
}

// U_ij = (f32) y[n-1-i][n-1-j] for j >= i, 0 below (src/linalg.rs:368-373).
__global__ __launch_bounds__(256) void k_scatter_u(int n, const double* __restrict__ y, float* __restrict__ u) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)n * n) return;
  const int i = (int)(idx / n), j = (int)(idx % n);
  u[idx] = (j >= i) ? (float)y[(long)(n - 1 - i) * n + (n - 1 - j)] : 0.0f;
}

__global__ __launch_bounds__(256) void k_fill_zero_f64(double* p, long count) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx < count) p[idx] = 0.0;
}

inline unsigned nblk(long count) { return (unsigned)((count + 255) / 256); }

}  // namespace

hipError_t build_flipped(hipStream_t st, int n, int ld, const float* h, const uint32_t* perm, double damp_val,
                         double* a, float* h32) {
  const unsigned grid = (unsigned)std::min<long>(((long)ld * ld + 255) / 256, 1L << 20);
  hipLaunchKernelGGL(k_build_flipped, dim3(grid), dim3(256), 0, st, n, ld, h, perm, damp_val, a, h32);
  return hipGetLastError();
}

hipError_t build_flipped_f64(hipStream_t st, int n, const double* h, double* a) {
  hipLaunchKernelGGL(k_build_flipped_f64, dim3(nblk((long)n * n)), dim3(256), 0, st, n, h, a);
  return hipGetLastError();
}

hipError_t chol_diag(hipStream_t st, int n, double* a, int k, int kb, int* status, double* pivot) {
  hipLaunchKernelGGL(k_chol_diag, dim3(1), dim3(512), 0, st, n, a, k, kb, status, pivot);
  return hipGetLastError();
}

hipError_t chol_panel(hipStream_t st, int n, double* a, int k, int kb, const int* status) {
  const int rows = n - (k + kb);
  if (rows <= 0) return hipSuccess;
  const int per_wg = 64 * TRS_WAVES / G;
  hipLaunchKernelGGL(k_chol_panel, dim3((rows + per_wg - 1) / per_wg), dim3(64 * TRS_WAVES), 0, st, n, a, k, kb, status);
  return hipGetLastError();
}

hipError_t trinv_diag(hipStream_t st, int n, const double* l, double* y, const int* status) {
  hipLaunchKernelGGL(k_trinv_diag, dim3((n + NBC - 1) / NBC, NBC * G / (64 * TRS_WAVES)), dim3(64 * TRS_WAVES), 0, st, n, l, y, status);
  return hipGetLastError();
}

hipError_t scatter_u(hipStream_t st, int n, const double* y, float* u) {
  hipLaunchKernelGGL(k_scatter_u, dim3(nblk((long)n * n)), dim3(256), 0, st, n, y, u);
  return hipGetLastError();
}

hipError_t fill_zero_f64(hipStream_t st, double* p, size_t count) {
  if (!count) return hipSuccess;
  hipLaunchKernelGGL(k_fill_zero_f64, dim3(nblk((long)count)), dim3(256), 0, st, p, (long)count);
  return hipGetLastError();
}

}  // namespace cdclq
