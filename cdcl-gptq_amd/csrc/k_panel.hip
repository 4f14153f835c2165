// Phase-2 sweeps of one KC panel (256 columns) per launch (src/engine.rs:543-658).
//
// The repair's gradient g = E H[:, c0 .. c0 + wd] is, per element, one fused chain per KC panel of
// k, the panels' chains folded in order. A step on columns of panel q changes E only there, so the
// chains of every other panel are the same for all of panel q's refit groups (or descent
// sub-blocks): one GEMM over the panel's 256 columns computes them (panel_gemm with skip = q), and
// the kernels here run the panel's steps one after another, computing panel q's own chain from the
// E that the previous step left and folding it into its place. Per panel that is two launches
// instead of two per step, and a GEMM of 256 columns instead of 64 or 128.
//
// A workgroup takes R rows, a wavefront per row, and keeps the rows' E over the panel in LDS. The
// columns of H that a step needs (256 x 64 floats, 64 KB a piece) are loaded directly to LDS, two
// pieces at a time. Latency bounds these kernels: R is the smallest of 4, 8 and 16 whose workgroups
// fit the device at once. In cycles, one piece of a descent with 8 rows: the own chains 2600 (64
// v_mfma_f32_16x16x4_f32 of 32 cycles, four steps of k in ascending order each as in mfma_tile.h, beside the
// next piece's loads), the fold 250, issuing the next chains' and columns' loads behind the piece's
// 1300, the visits 700 to 2000 (the row with the most moves), barriers 200. One group of a refit with 8
// rows: the own chains and U H_CC side by side 6900, the fold 800, the sums 1600, the update 400, the
// next pieces' loads 3000 from the sums on.
//
// Repair of one matrix, a launch pair per step against a launch pair per panel: 256 x 256 3.9 ->
// 1.6 ms, 1001 x 1350 11.5 -> 5.1 ms, 2048 x 2048 12.9 -> 8.2 ms, 2048 x 5632 (groups of 64) 68.7 ->
// 41.8 ms, 4096 x 14336 397 -> 360 ms.
#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "cdclq_dev.h"
#include "kernels.h"

namespace cdclq {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int KC = CDCLQ_KC;
constexpr int PW = 64;             // columns of a piece of H
constexpr int PIECE = KC * PW;     // floats of a piece
constexpr size_t LDS_BYTES = 160 * 1024;
constexpr int ES = KC + 4;         // row stride of the staged E (16-byte aligned, rows on different banks)

// LDS-only barrier: the wave's LDS writes are visible to the workgroup after it; vector loads and
// direct-to-LDS loads stay in flight (wait_vmcnt where their data is needed).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Rows [0, kr) of panel row c0 .. and columns col .. col + 63 of H into the piece at LDS offset
// `dst`: load i covers rows 4 i .. 4 i + 3 (lane l: row 4 i + (l >> 4)). Column c of row k lies at position
// c ^ 16 (k & 3) (at()), so that the four rows that one MFMA step reads side by side start on
// different banks. kr is a multiple of 16 and c0 + kr <= ld, col + 64 <= ld (ld is a multiple of 64).
__device__ __forceinline__ int at(int k, int c) { return k * PW + (c ^ ((k & 3) << 4)); }

template <int W>
__device__ __forceinline__ void load_piece(const float* __restrict__ h32, int ld, int c0, int kr, int col,
                                           uint32_t dst, int wv, int lane) {
  const int q = lane >> 4;
  const float* src = h32 + (long)(c0 + q) * ld + col + 4 * ((lane & 15) ^ (4 * q));
  for (int i = wv; i < kr / 4; i += W) dma16_untracked(src + (long)(4 * i) * ld, dst + 1024u * (uint32_t)i);
}

// kr steps (a multiple of 16) of the chains of 16 rows and 16 columns: a = the lane's first A element
// (row lane & 15, step lane >> 4, the row's steps following one another), b = its first B element (step
// lane >> 4 of the piece, column lane & 15 of the 16). Register r of the result is row 4 (lane >> 4) + r,
// column lane & 15. Every instruction waits for the one before it (32 cycles), so the operands are
// read eight instructions ahead and the reads issued between the instructions.
__device__ __forceinline__ v4f chain16(const float* ap, const float* bp, int kr) {
  // LDS addresses in a register each: the reads' offsets then fit the instructions
  typedef const __attribute__((address_space(3))) float* lds_t;
  lds_t a = (lds_t)ap, b = (lds_t)bp;
  asm volatile("" : "+v"(a), "+v"(b));
  v4f acc = {};
  int k = 0;
  for (; k + 128 <= kr; k += 128) {
    float x[32], y[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      x[u] = a[k + 4 * u];
      y[u] = b[(k + 4 * u) * PW];
    }
#pragma unroll
    for (int u = 0; u < 32; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], y[u], acc, 0, 0, 0);
    // (a read brings the operands of two instructions)
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
    for (int u = 0; u < 12; ++u) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
  }
  for (; k < kr; k += 16) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k + 4 * u], b[(k + 4 * u) * PW], acc, 0, 0, 0);
  }
  return acc;
}

// The chains of 4 rows and 64 columns on v_mfma_f32_4x4x1_16b_f32, its 16 blocks side by side: piece =
// the steps' first row of H (a multiple of 4 of the panel's rows), lane l column l. Register i of the
// result is row i, column l. a(k) = the lane's A element of step k + (lane >> 2) and row lane & 3; the
// instruction broadcasts the block of its step to the 16 blocks (cbsz 4, abid the block), so that one
// register serves 16 steps.
typedef const __attribute__((address_space(3))) float* lds_f;

struct Cols4 {  // a lane's column of a piece: row k at h[k & 3][(k & ~3) * PW]
  lds_f h[4];
  __device__ __forceinline__ Cols4(const float* piece, int lane) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = (lds_f)(piece + at(j, lane));
      asm volatile("" : "+v"(h[j]));
    }
  }
};

#define CHAIN4_STEP(B) \
  acc = __builtin_amdgcn_mfma_f32_4x4x1f32(x, c.h[(B) & 3][(k + ((B) & ~3)) * PW], acc, 4, B, 0)
#define CHAIN4_QUAD(B) CHAIN4_STEP(B), CHAIN4_STEP(B + 1), CHAIN4_STEP(B + 2), CHAIN4_STEP(B + 3)

// kr steps (and on to a multiple of 4) of one chain. Groups start at multiples of 16, so the rows read
// stay inside the piece.
template <class FA>
__device__ __forceinline__ void chain4(FA a, const Cols4& c, int kr, v4f& acc) {
  float x = a(0);
  int k = 0;
  for (; k + 16 <= kr; k += 16) {
    const float xn = a(min(k + 16, (kr - 1) & ~15));
    CHAIN4_QUAD(0), CHAIN4_QUAD(4), CHAIN4_QUAD(8), CHAIN4_QUAD(12);
    x = xn;
  }
  if (k < kr) CHAIN4_QUAD(0);
  if (k + 4 < kr) CHAIN4_QUAD(4);
  if (k + 8 < kr) CHAIN4_QUAD(8);
  if (k + 12 < kr) CHAIN4_QUAD(12);
}
#undef CHAIN4_QUAD
#undef CHAIN4_STEP

// The loads into v have arrived from here on. The compiler counts the loads it knows of; without this,
// the wait before their first use would also wait for the direct-to-LDS loads issued since.
template <int NB>
__device__ __forceinline__ void arrived(float (&v)[NB]) {
#pragma unroll
  for (int u = 0; u < NB; ++u) asm volatile("" : "+v"(v[u]));
}

// NB of a row's other-panel chains in flight: slots u0 .. u0 + NB - 1 of P (those past nf repeat the
// last), src the row's first element in slot 0 (uniform), lo the lane's element. The running offset
// and the bounds are opaque, so that the addresses and tests are formed one after another instead
// of being kept (and spilled) across the steps.
template <int NB>
__device__ __forceinline__ void load_chains(const float* __restrict__ src, uint32_t lo, long pstride, int u0, int nf,
                                            float (&v)[NB]) {
  long off = (long)u0 * pstride;
  asm volatile("" : "+s"(off), "+s"(nf));
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    v[u] = __builtin_nontemporal_load(src + off + lo);
    off += u0 + u + 1 < nf ? pstride : 0;
  }
  __builtin_amdgcn_sched_barrier(0);  // issued here, not sunk to the adds
}

// The element's ordered fold C = C + P_p over every panel, the own chain at position q; v holds the
// first NB of the nf other panels' chains, the rest is loaded here.
template <int NB>
__device__ __forceinline__ float fold_with_own(const float* __restrict__ src, uint32_t lo, long pstride, int q, int nf,
                                               float own, float (&v)[NB]) {
  float acc = 0.0f;
  asm volatile("" : "+s"(q), "+s"(nf));
  for (int u0 = 0; u0 < nf; u0 += NB) {
    if (u0) load_chains<NB>(src, lo, pstride, u0, nf, v);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (u0 + u < nf) {  // uniform
        if (u0 + u == q) acc = acc + own;
        acc = acc + v[u];
      }
    }
  }
  return q == nf ? acc + own : acc;
}

// ---- Coordinate descent over the panel's 64-column sub-blocks (src/engine.rs:600-658), decisions
// and accounting as in k_cd: every lane evaluates its own column with the current gradient, and the
// lowest column at or after the cursor whose code changes is the next move of the sequential visit.
// Wavefronts: the first R have a row; 0 to 3 run the own chains while the others (at least four) load
// the next piece.
template <int R, int NB>
__global__ __launch_bounds__(64 * (R < 8 ? 8 : R)) void k_cd_panel(CdPanelArgs a) {
  constexpr int W = R < 8 ? 8 : R;
  __shared__ __align__(16) float Hs[2][PIECE];
  __shared__ __align__(16) float Es[R * ES];
  __shared__ float Gs[R * PW];
  __shared__ uint32_t need;
  static_assert(sizeof(Hs) + sizeof(Es) + sizeof(Gs) + sizeof(need) <= LDS_BYTES, "a CU's LDS");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = a.n, ld = a.ld, q = a.q, c0 = q * KC;
  const int kc = min(KC, n - c0), npc = (kc + PW - 1) / PW, kr = (kc + 15) & ~15;
  const bool roww = wv < R;
  const int wvr = min(wv, R - 1);
  const int r = blockIdx.x * R + wvr, rr = min(r, a.rows - 1), chunk = rr / a.rc;
  const int sb0 = q * (KC / PW);
  // pieces (= sub-blocks) that this row, and the workgroup, work on
  if (tid == 0) need = 0;
  __syncthreads();
  uint32_t act = a.active[chunk], chosen = a.sel[(long)chunk * a.nsb + sb0 + min(lane, npc - 1)];
  asm volatile("" : "+v"(act), "+v"(chosen));  // both loads issued before either is tested
  const uint32_t pick =
      roww && r < a.rows && __builtin_amdgcn_readfirstlane(act) ? (uint32_t)__ballot(chosen && lane < npc) : 0u;
  if (lane == 0 && pick) atomicOr(&need, pick);
  __syncthreads();
  uint32_t todo = __builtin_amdgcn_readfirstlane(need);
  if (!todo) return;

  const uint32_t hs0 = lds_offset(&Hs[0][0]);
  int j = __builtin_ctz(todo), buf = 0;
  todo &= todo - 1;
  const long pstride = (long)a.rows * a.wdp;
  const int nf = a.np - 1;  // the other panels, slot u of P: panel u + (u >= q)
  const float* prow = a.P + (long)rr * a.wdp;
  float v[NB];
  struct Col {  // a column's state and parameters, one column per lane
    float wq, sc, zz;
    int code, bits;
  };
  auto load_col = [&](int jj) {
    const int wd = min(PW, kc - PW * jj), col = c0 + PW * jj + min(lane, wd - 1), gi = col / a.g;
    Col c;
    c.wq = a.wq[(long)rr * n + col];
    c.code = (int)a.codes[(long)rr * n + col];
    c.sc = a.scales[(long)rr * a.ng + gi];
    c.zz = a.zeros[(long)rr * a.ng + gi];
    c.bits = a.gbits[gi];
    return c;
  };
  Col nxt;
  {
    // (the piece first: loads return in order, and it is the largest)
    load_piece<W>(a.h32, ld, c0, kr, c0 + PW * j, hs0, wv, lane);
    v4f ev = {};
    if (4 * lane < a.wdp) ev = *reinterpret_cast<const v4f*>(a.e + (long)rr * ld + c0 + 4 * lane);
    if (nf > 0) load_chains<NB>(prow + PW * j, lane, pstride, 0, nf, v);
    nxt = load_col(j);
    if (roww) *reinterpret_cast<v4f*>(&Es[wv * ES + 4 * lane]) = ev;
  }
  wait_vmcnt<0>();
  lds_barrier();
  // This wavefront's part of the next piece has landed once at most the chains' loads issued after
  // it are outstanding (a row's; the column's come on top, so this waits for a few of the chains too).
  auto wait_part = [&]() {
    if (roww && nf > 0)
      wait_vmcnt<(NB < 60 ? NB : 60)>();
    else
      wait_vmcnt<0>();
  };
  uint32_t nevals = 0, nnear = 0;
  while (true) {
    const int jn = todo ? __builtin_ctz(todo) : -1;
    if (jn >= 0) todo &= todo - 1;
    arrived(v);
    asm volatile("" : "+v"(nxt.wq), "+v"(nxt.sc), "+v"(nxt.zz), "+v"(nxt.bits), "+v"(nxt.code));
    if (jn >= 0 && wv >= 4)  // the next piece, into the buffer whose readers passed the last barrier
      load_piece<W - 4>(a.h32, ld, c0, kr, c0 + PW * jn, hs0 + (uint32_t)((buf ^ 1) * PIECE * 4), wv - 4, lane);
    if (wv < 4) {  // the own chains of columns 16 wv .. + 15
      const int q4 = lane >> 4, i = lane & 15;
      const float* ea = &Es[min(i, R - 1) * ES + q4];
      const float* hb = &Hs[buf][at(q4, 16 * wv + i)];
      const v4f g = chain16(ea, hb, kr);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (4 * q4 + u < R) Gs[(4 * q4 + u) * PW + 16 * wv + i] = g[u];
      }
    }
    lds_barrier();
    const int wd = min(PW, kc - PW * j);
    const float* hcc = &Hs[buf][PW * j * PW];  // the sub-block's rows and columns of H
    float gg = fold_with_own<NB>(prow + PW * j, lane, pstride, q, nf, Gs[wvr * PW + lane], v);
    const Col cur = nxt;
    if (jn >= 0 && roww) {
      if (nf > 0) load_chains<NB>(prow + PW * jn, lane, pstride, 0, nf, v);
      nxt = load_col(jn);
    }
    if ((pick >> j) & 1) {
      const bool in = lane < wd;
      const uint64_t inmask = __ballot(in);
      float mwq = cur.wq, me = Es[wv * ES + PW * j + lane];
      int mc = cur.code;
      const float hd = hcc[at(min(lane, wd - 1), min(lane, wd - 1))], sc = cur.sc, zz = cur.zz;
      const float mq = (float)((1u << cur.bits) - 1u);
      const long step = (long)(sb0 + j) * a.rows + r;
      double* dl = a.dlog + step * a.cap;
      uint32_t moves = 0;
      for (int sw = 0; sw < a.sweeps; ++sw) {
        bool changed = false;
        int start = 0;
        while (start < PW) {
          const float target = mwq + gg / hd;
          float qv;
          const float newdq = quant_dq(target, sc, zz, mq, &qv);
          const int qc = (int)code_of(qv);
          const uint64_t mask = __ballot(in && lane >= start && qc != mc);
          // the sequential visit evaluated columns start .. (the move, or the end) with this gradient
          const int last = mask ? (int)__builtin_ctzll(mask) : 63;
          const uint64_t seen = (~0ull << start) & (last == 63 ? ~0ull : ((1ull << (last + 1)) - 1ull)) & inmask;
          nevals += (uint32_t)__builtin_popcountll(seen);
          nnear += (uint32_t)__builtin_popcountll(__ballot(near_midpoint(target, sc, zz, mq)) & seen);
          if (mask == 0) break;
          const int jl = __builtin_amdgcn_readfirstlane(last);
          const float de = readlane(mwq, jl) - readlane(newdq, jl);
          const float gj = readlane(gg, jl), hjj = readlane(hd, jl);
          const float d32 = (2.0f * de) * gj + (de * de) * hjj;
          if (lane == 0) dl[moves] = (double)d32;
          ++moves;
          gg = gg + de * hcc[at(jl, lane)];  // lanes past wd take values that are never used
          if (lane == jl) {
            mwq = newdq;
            mc = qc;
            me = me + de;
          }
          changed = true;
          start = jl + 1;
        }
        if (!changed) break;
      }
      if (jn >= 0 && wv >= 4) wait_part();
      if (moves && in) {
        const int col = c0 + PW * j + lane;
        a.wq[(long)r * n + col] = mwq;
        a.codes[(long)r * n + col] = (uint8_t)mc;
        a.e[(long)r * ld + col] = me;
        Es[wv * ES + PW * j + lane] = me;
      }
      if (lane == 0) a.dcnt[step] = moves;
    }
    if (jn < 0) break;
    if (wv >= 4 && !((pick >> j) & 1)) wait_part();
    lds_barrier();
    j = jn;
    buf ^= 1;
  }
  if (pick && lane == 0) {
    a.evals[r] += nevals;  // one wave per row: no other writer in this launch
    if (nnear) atomicAdd(&a.mid[MID_CD_NEAR], (unsigned long long)nnear);
  }
}

// ---- Closed-form f16 scale refit of the panel's groups, one after another (src/engine.rs:543-587).
// Per group: hu = U H_CC (U = codes - zero) and the own chains run side by side on different
// wavefronts, the rows' wavefronts fold the gradient, and one lane per row sums num = sum u_k g_k
// and den = sum u_k hu_k in k order. NH: 64-column pieces a group takes (1: groups of at most 64
// columns that divide 64, the next piece loading meanwhile; 2: 128, or one group of all n <= 128
// columns: both buffers hold the group, whose products u hu use the second one once its chains are
// done, and the next group's first piece loads behind the sums).
template <int R, int NB, int NH>
__global__ __launch_bounds__(64 * R) void k_refit_panel(RefitPanelArgs a) {
  constexpr int PS = 64 * NH + 4;              // row stride of the products (16-byte aligned)
  constexpr int ZN = NH == 2 ? 2 : 16;         // groups of a panel
  constexpr int RG = R / 4, NT = RG * NH;      // row quads; chains of each kind
  // 16 rows of 128-column groups: the products u hu lie in the second piece's buffer; otherwise LDS
  // has room for them, and both pieces of the next group load as soon as the chains are done
  constexpr bool PHIN = R == 16 && NH == 2;
  static_assert(2 * NT <= R, "a wavefront per chain");
  __shared__ __align__(16) float Hs[2][PIECE];
  __shared__ __align__(16) float Es[R * ES];
  __shared__ uint32_t Cs[R * KC / 4];          // codes, one byte per column
  __shared__ __align__(16) float PG[R * PS];                 // the own chains, then the products u g
  __shared__ __align__(16) float PH1[PHIN ? 1 : R * PS];
  __shared__ float Zs[R * ZN], snew[R];
  __shared__ int lv[R], mv[R], nlive;
  static_assert(sizeof(Hs) + sizeof(Es) + sizeof(Cs) + sizeof(PG) + sizeof(PH1) + sizeof(Zs) + sizeof(snew) +
                        sizeof(lv) + sizeof(mv) + sizeof(nlive) <= LDS_BYTES, "a CU's LDS");
  float* PH = PHIN ? &Hs[1][0] : PH1;          // the products u hu
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = a.n, ld = a.ld, q = a.q, g = a.g, ng = a.ng, c0 = q * KC;
  const int kc = min(KC, n - c0), kr = (kc + 15) & ~15;
  const int g0 = c0 / g, gcnt = (kc + g - 1) / g;
  const int r0 = blockIdx.x * R, r = r0 + wv, rr = min(r, a.rows - 1);
  if (tid == 0) nlive = 0;
  __syncthreads();
  const bool live = r < a.rows && a.active[rr / a.rc];
  if (lane == 0) lv[wv] = live;
  if (lane == 0 && live) atomicAdd(&nlive, 1);
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(nlive) == 0) return;

  const uint32_t hs0 = lds_offset(&Hs[0][0]);
  uint8_t* cb = reinterpret_cast<uint8_t*>(Cs) + wv * KC;
  const long pstride = (long)a.rows * a.wdp;
  const int nf = a.np - 1;
  const float* prow = a.P + (long)rr * a.wdp;
  float v[NH][NB], wqn[NH], sold_n = 0.0f;
  // a group's column for this lane: panel column off + kcol, kcol = 64 h + lane - o (o: the group's
  // offset in its piece); off = t g
  auto prefetch = [&](int t) {
    const int off = t * g, o = NH == 2 ? 0 : off % PW, wd = min(g, kc - off);
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int col = off + min(max(64 * h + lane - o, 0), wd - 1);
      if (nf > 0) load_chains<NB>(prow, col, pstride, 0, nf, v[h]);
      wqn[h] = a.wq[(long)rr * n + c0 + col];
    }
    if (wv == 0) sold_n = a.scales[(long)min(r0 + min(lane, R - 1), a.rows - 1) * ng + g0 + t];
  };
  {
    // (the pieces first: loads return in order, and they are the largest)
    load_piece<R>(a.h32, ld, c0, kr, c0, hs0, wv, lane);
    if (NH == 2 && kc > PW) load_piece<R>(a.h32, ld, c0, kr, c0 + PW, hs0 + PIECE * 4, wv, lane);
    v4f ev = {};
    if (4 * lane < a.wdp) ev = *reinterpret_cast<const v4f*>(a.e + (long)rr * ld + c0 + 4 * lane);
    uint8_t cv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cv[i] = a.codes[(long)rr * n + c0 + min(64 * i + lane, kc - 1)];
    const float z = a.zeros[(long)rr * ng + g0 + min(lane, gcnt - 1)];
    prefetch(0);
    *reinterpret_cast<v4f*>(&Es[wv * ES + 4 * lane]) = ev;
#pragma unroll
    for (int i = 0; i < 4; ++i) cb[64 * i + lane] = cv[i];
    if (lane < ZN) Zs[wv * ZN + lane] = z;
  }
  wait_vmcnt<0>();
  lds_barrier();
  for (int t = 0; t < gcnt; ++t) {
    const int off = t * g, o = NH == 2 ? 0 : off % PW, wd = min(g, kc - off), gi = g0 + t;
    const int slot = NH == 2 ? 0 : (off / PW) & 1;  // NH == 2: pieces off / 64 and off / 64 + 1 in slots 0, 1
    const bool more = t + 1 < gcnt;
    const int offn = off + g;
    if (NH == 1 && o == 0 && off + PW < kc)  // the next piece, while this one's groups run
      load_piece<R>(a.h32, ld, c0, kr, c0 + off + PW, hs0 + (uint32_t)((slot ^ 1) * PIECE * 4), wv, lane);
    const int tk = wv % NT, rg = tk % RG, h = tk / RG;
    const bool own = wv < NT, hut = wv >= NT && wv < 2 * NT;
    const bool cols = 64 * h < wd;  // (wd <= 64: the second piece is not loaded)
    const int kcol = 64 * h + lane - o;
    const uint8_t* cbytes = reinterpret_cast<const uint8_t*>(Cs);
    v4f gv = {}, hu = {}, ph = {};
    if (cols && (own || hut)) {
      const float* ea = &Es[(4 * rg + (lane & 3)) * ES + (lane >> 2)];
      // hu: one chain of wd <= KC steps (sgemm at src/engine.rs:560); rows of H past n are zero, so a
      // step past wd (the last group's remainder up to a multiple of 4) adds a zero product
      const float za = Zs[(4 * rg + (lane & 3)) * ZN + t];
      const uint8_t* crow = cbytes + (4 * rg + (lane & 3)) * KC + off + (lane >> 2);
      auto ae = [&](int k) { return ea[k]; };
      auto au = [&](int k) { return (float)crow[k] - za; };
      const Cols4 he(&Hs[slot + h][0], lane), hc(&Hs[slot + h][off * PW], lane);
      if (own)
        chain4(ae, he, kr, gv);
      else
        chain4(au, hc, wd, hu);
      if (own && kcol >= 0 && kcol < wd) {
#pragma unroll
        for (int i = 0; i < 4; ++i) PG[(4 * rg + i) * PS + kcol] = gv[i];
      }
      if (hut) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // panel end C = fma(1, chain, 0), then u_k * hu_k
          const int row = 4 * rg + i;
          const float u = (float)cbytes[row * KC + min(max(off + kcol, 0), KC - 1)] - Zs[row * ZN + t];
          ph[i] = u * __builtin_fmaf(1.0f, hu[i], 0.0f);
        }
      }
      if (!PHIN && hut && kcol >= 0 && kcol < wd) {
#pragma unroll
        for (int i = 0; i < 4; ++i) PH[(4 * rg + i) * PS + kcol] = ph[i];
      }
    }
#pragma unroll
    for (int hh = 0; hh < NH; ++hh) arrived(v[hh]);
    arrived(wqn);
    asm volatile("" : "+v"(sold_n));
    lds_barrier();  // the chains are done: both buffers of a 128-column group are free
    if (PHIN && hut && cols && kcol < wd) {
#pragma unroll
      for (int i = 0; i < 4; ++i) PH[(4 * rg + i) * PS + kcol] = ph[i];
    }
    float wqv[NH], uu[NH];
    const float z = Zs[wv * ZN + t], sold = sold_n;
#pragma unroll
    for (int hh = 0; hh < NH; ++hh) {
      const int kl = 64 * hh + lane - o, kq = min(max(kl, 0), wd - 1);
      const float gg = fold_with_own<NB>(prow, off + kq, pstride, q, nf, PG[wv * PS + kq], v[hh]);
      uu[hh] = (float)cb[off + kq] - z;
      wqv[hh] = wqn[hh];
      if (kl >= 0 && kl < wd) PG[wv * PS + kl] = uu[hh] * gg;
    }
    lds_barrier();
    if (NH == 2 && more && wv > 0) {  // the next group's pieces, while wavefront 0 adds
      load_piece<R - 1>(a.h32, ld, c0, kr, c0 + offn, hs0, wv - 1, lane);
      if (!PHIN && offn + PW < kc) load_piece<R - 1>(a.h32, ld, c0, kr, c0 + offn + PW, hs0 + PIECE * 4, wv - 1, lane);
    }
    float num = 0.0f, den = 0.0f;
    if (wv == 0) {
      // num, den: separate multiply and add, sequential in k (src/engine.rs:562-566), num on lane
      // `row`, den on lane 32 + row; 16 columns are read while the 16 before them are added
      const float* ps = (lane < 32 ? PG : PH) + min(lane & 31, R - 1) * PS;
      v4f x[4], y[4];
      auto rd = [&](int c, v4f (&v)[4]) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) v[jj] = *reinterpret_cast<const v4f*>(ps + c + 4 * jj);
      };
      auto add = [&](const v4f (&v)[4]) {
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) num = num + v[jj >> 2][jj & 3];
      };
      int k = 0;
      if (wd >= 32) {
        rd(0, x);
        for (; k + 32 <= wd; k += 32) {
          rd(k + 16, y);
          __builtin_amdgcn_sched_barrier(0);
          add(x);
          rd(min(k + 32, wd - 16) & ~3, x);  // (after the last pair: read and not used)
          __builtin_amdgcn_sched_barrier(0);
          add(y);
        }
      }
      for (; k < wd; ++k) num = num + ps[k];
      den = __shfl(num, (lane & 31) + 32, 64);
    }
    if (wv == 0 && lane < R) {
      // the closed-form f16 scale and its acceptance test (:567-587)
      const int row = r0 + lane;
      int moved = 0;
      float s_new = 0.0f;
      if (lv[lane]) {
        if (den > 1e-30f) {
          s_new = rs_maxf(round_f16(sold + num / den), CDCLQ_F16_MIN_NORMAL);
          const float d = s_new - sold;
          const float dl32 = (-2.0f * d) * num + (d * d) * den;
          if ((double)dl32 < 0.0) {
            a.scales[(long)row * ng + gi] = s_new;
            a.dlog[(long)gi * a.rows + row] = (double)dl32;
            moved = 1;
          }
        }
        a.dcnt[(long)gi * a.rows + row] = moved;
      }
      mv[lane] = moved;
      snew[lane] = s_new;
    }
    if (more) {
      if (!PHIN) wait_vmcnt<0>();  // the next pieces' loads, issued at the latest after the chains
      __builtin_amdgcn_sched_barrier(0);
      prefetch(t + 1);
    }
    lds_barrier();
    if (PHIN && more && offn + PW < kc)
      load_piece<R>(a.h32, ld, c0, kr, c0 + offn + PW, hs0 + PIECE * 4, wv, lane);
    if (mv[wv]) {  // e += W_hat - ndq, W_hat = ndq
      const float s_new = snew[wv];
#pragma unroll
      for (int hh = 0; hh < NH; ++hh) {
        const int kl = 64 * hh + lane - o;
        if (kl >= 0 && kl < wd) {
          const int pc = off + kl;
          const float ndq = s_new * uu[hh];
          const float ne = Es[wv * ES + pc] + (wqv[hh] - ndq);
          Es[wv * ES + pc] = ne;
          a.e[(long)r * ld + c0 + pc] = ne;
          a.wq[(long)r * n + c0 + pc] = ndq;
        }
      }
    }
    if (!more) break;
    if (PHIN) wait_vmcnt<0>();
    lds_barrier();
  }
}

// rows per workgroup: the smallest whose workgroups (one per CU) fit at once
int panel_rows(int rows, int cus) { return rows <= 4 * cus ? 4 : (rows <= 8 * cus ? 8 : 16); }

}  // namespace

hipError_t refit_panel(hipStream_t st, const RefitPanelArgs& a) {
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const int R = panel_rows(a.rows, cus);
  const dim3 grid((a.rows + R - 1) / R), blk(64 * R);
  const bool two = a.g > PW;
// (24 chains of two columns in flight is what 16 wavefronts' registers hold)
#define REFIT_PANEL(RR, NB)                                                          \
  do {                                                                               \
    if (two)                                                                         \
      hipLaunchKernelGGL((k_refit_panel<RR, (NB > 24 ? 24 : NB), 2>), grid, blk, 0, st, a); \
    else                                                                             \
      hipLaunchKernelGGL((k_refit_panel<RR, NB, 1>), grid, blk, 0, st, a);           \
  } while (0)
#define REFIT_PANEL_R(RR)                                                            \
  do {                                                                               \
    if (a.np <= 9)                                                                   \
      REFIT_PANEL(RR, 8);                                                            \
    else if (a.np <= 17)                                                             \
      REFIT_PANEL(RR, 16);                                                           \
    else                                                                             \
      REFIT_PANEL(RR, 32);                                                           \
  } while (0)
  if (R == 4)
    REFIT_PANEL_R(4);
  else if (R == 8)
    REFIT_PANEL_R(8);
  else
    REFIT_PANEL_R(16);
#undef REFIT_PANEL_R
#undef REFIT_PANEL
  return hipGetLastError();
}

hipError_t cd_panel(hipStream_t st, const CdPanelArgs& a) {
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const int R = panel_rows(a.rows, cus);
  const dim3 grid((a.rows + R - 1) / R), blk(64 * std::max(R, 8));
#define CD_PANEL_R(RR)                                                               \
  do {                                                                               \
    if (a.np <= 9)                                                                   \
      hipLaunchKernelGGL((k_cd_panel<RR, 8>), grid, blk, 0, st, a);                  \
    else if (a.np <= 17)                                                             \
      hipLaunchKernelGGL((k_cd_panel<RR, 16>), grid, blk, 0, st, a);                 \
    else if (a.np <= 33)                                                             \
      hipLaunchKernelGGL((k_cd_panel<RR, 32>), grid, blk, 0, st, a);                 \
    else                                                                             \
      hipLaunchKernelGGL((k_cd_panel<RR, 60>), grid, blk, 0, st, a);                 \
  } while (0)
  if (R == 4)
    CD_PANEL_R(4);
  else if (R == 8)
    CD_PANEL_R(8);
  else
    CD_PANEL_R(16);
#undef CD_PANEL_R
  return hipGetLastError();
}

}  // namespace cdclq
