// Tiles of fused multiply-add chains on the matrix cores (gfx950), shared by the f32 GEMM kernels.
//
// v_mfma_f32_32x32x2_f32 advances each of its 32 x 32 elements by two steps of the chain, k = 2 s then
// 2 s + 1, each product added with one rounding: bit for bit two fmaf in ascending k (checked on the
// device over 2e7 outputs with operands spread over 2^+-72, denormal products included). Lane l
// supplies A[l & 31][2 s + (l >> 5)] and B[2 s + (l >> 5)][l & 31]; register r of the result is row
// (r & 3) + 8 (r >> 2) + 4 (l >> 5), column l & 31.
//
// A workgroup of WR x WC wavefronts owns a tile of 32 FR WR rows x 32 FC WC columns, a wavefront FR x
// FC of the 32 x 32 blocks. Stages of 32 k live in LDS: A as [rows][8 quads of k], the quad at
// position p of row r being p ^ (r / 2 & 7): even and odd rows start on different halves of the banks,
// and this spreads the 16 rows that a 16-byte read serves at once over each half (with p ^ (r & 7)
// every such read took 4 cycles more); B as [32 k][columns]. An operand group is 8 k:
//   A: one 16-byte read per 32 rows gives lane (i, h) the quad 2 g + h of its row; two
//      v_permlane32_swap turn the four registers into the operands of the group's four steps.
//   B: one read per step gives lane (j, h) FC neighbouring columns of row 2 s + h: block b's column j
//      is column FC j + b of the wavefront, so that the blocks need no reads of their own and a row of
//      results is FC consecutive floats per lane. With BT, B is given transposed (a row of k per
//      column): it is staged and read as A is, and block b's column j is column 32 b + j.
// With FR x FC = 2 x 4 blocks that is 6 LDS reads per 32 MFMAs.
#pragma once

#include "cdclq_dev.h"

namespace cdclq {

typedef float tile_v4f __attribute__((ext_vector_type(4)));
typedef float tile_v16f __attribute__((ext_vector_type(16)));

constexpr int TILE_SK = 32;  // k per stage
constexpr int TILE_G = TILE_SK / 8;  // operand groups per stage

template <int WR_, int WC_, int FR_, int FC_, bool BT = false>
struct MfmaTile {
  static constexpr int WR = WR_, WC = WC_, FR = FR_, FC = FC_;
  static constexpr int W = WR * WC, THREADS = 64 * W;
  static constexpr int ROWS = 32 * FR * WR, COLS = 32 * FC * WC;
  static constexpr int STAGE = TILE_SK * (ROWS + COLS);  // floats
  static constexpr int LA = TILE_SK * ROWS / 256 / W;    // 1 KB loads per wave and stage: of A,
  static constexpr int LB = TILE_SK * COLS / 256 / W;    // of B
  static constexpr int NL = LA + LB;
  static constexpr int KR = 256 / COLS;                  // k rows per load of B
  static_assert(LA >= 1 && LB >= 1 && COLS <= 256 && 256 % COLS == 0, "stage too small for the workgroup");

  struct Ops {  // one operand group: step s (0..3) of row block f: a[f][s]; of column block b: b[s][b]
    float a[FR][4];
    float b[4][FC];
  };
  struct Acc {
    tile_v16f c[FR][FC];
  };

  // The lane's offsets from the tile's first A element / B row (BT: B element): off[q] of load q of
  // this wave. Rows from m_left on and columns from n_left on (from the tile's first; without BT n_left
  // is a multiple of 4) repeat the last ones.
  template <class I>
  static __device__ __forceinline__ void offsets(int wv, int lane, int m_left, long lda, int n_left, long ldb,
                                                 I (&off)[NL]) {
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      if (q < LA || BT) {
        const int rl = 8 * (wv + W * (q < LA ? q : q - LA)) + (lane >> 3);
        off[q] = min(rl, (q < LA ? m_left : n_left) - 1) * (I)(q < LA ? lda : ldb) + 4 * ((lane & 7) ^ ((rl >> 1) & 7));
      } else {
        const int kr = KR * (wv + W * (q - LA)) + lane / (COLS / 4);
        off[q] = kr * (I)ldb + min(4 * (lane % (COLS / 4)), n_left - 4);
      }
    }
  }
  // Loads one stage into LDS at byte offset `dst`: a = the tile's A at the stage's first k, b = the
  // stage's first row of B at the tile's first column (BT: the tile's B at the stage's first k).
  template <class I>
  static __device__ __forceinline__ void load_stage(const float* a, const float* b, const I (&off)[NL], uint32_t dst,
                                                    int wv) {
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const uint32_t at = q < LA ? (uint32_t)(wv + W * q) : (uint32_t)(ROWS * TILE_SK / 256 + wv + W * (q - LA));
      dma16_untracked((q < LA ? a : b) + off[q], dst + 1024u * at);
    }
  }
  // Operand group g (0..3) of the stage at `st`.
  static __device__ __forceinline__ Ops read(const float* st, int g, int wr, int wc, int lane) {
    const int i = lane & 31, h = lane >> 5;
    Ops o;
    const float* as = st + TILE_SK * (32 * FR * wr + i) + 4 * ((2 * g + h) ^ ((i >> 1) & 7));
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      const tile_v4f x = *reinterpret_cast<const tile_v4f*>(as + f * 32 * TILE_SK);
#pragma unroll
      for (int s = 0; s < 4; ++s) o.a[f][s] = x[s];  // k 8 g + 4 h + s; put in step order by arrange()
    }
    if constexpr (BT) {
      const float* bs = st + TILE_SK * (ROWS + 32 * FC * wc + i) + 4 * ((2 * g + h) ^ ((i >> 1) & 7));
#pragma unroll
      for (int b = 0; b < FC; ++b) {
        const tile_v4f x = *reinterpret_cast<const tile_v4f*>(bs + b * 32 * TILE_SK);
#pragma unroll
        for (int s = 0; s < 4; ++s) o.b[s][b] = x[s];
      }
      return o;
    }
    const float* bs = st + TILE_SK * ROWS + (8 * g + h) * COLS + 32 * FC * wc + FC * i;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float* p = bs + 2 * s * COLS;
      if constexpr (FC == 4) {
        const tile_v4f x = *reinterpret_cast<const tile_v4f*>(p);
#pragma unroll
        for (int b = 0; b < 4; ++b) o.b[s][b] = x[b];
      } else if constexpr (FC == 2) {
        const float2 x = *reinterpret_cast<const float2*>(p);
        o.b[s][0] = x.x;
        o.b[s][1] = x.y;
      } else {
#pragma unroll
        for (int b = 0; b < FC; ++b) o.b[s][b] = p[b];
      }
    }
    return o;
  }
  // A's registers from (lane half h: k 4 h + s) to step order (step s: k 2 s + h): with x_s = the
  // register of k {s, 4 + s}, swapping the upper half of one with the lower half of the next gives
  // {0, 1} and {4, 5} from x_0, x_1, {2, 3} and {6, 7} from x_2, x_3.
  static __device__ __forceinline__ void to_steps(float& x0, float& x1, float& x2, float& x3) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x0), __float_as_uint(x1), false, false);
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(x2), __float_as_uint(x3), false, false);
    x0 = __uint_as_float(p[0]);
    x1 = __uint_as_float(q[0]);
    x2 = __uint_as_float(p[1]);
    x3 = __uint_as_float(q[1]);
  }
  static __device__ __forceinline__ void arrange(Ops& o) {
#pragma unroll
    for (int f = 0; f < FR; ++f) to_steps(o.a[f][0], o.a[f][1], o.a[f][2], o.a[f][3]);
    if constexpr (BT) {
#pragma unroll
      for (int b = 0; b < FC; ++b) to_steps(o.b[0][b], o.b[1][b], o.b[2][b], o.b[3][b]);
    }
  }
  static __device__ __forceinline__ void mul(const Ops& o, Acc& acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int f = 0; f < FR; ++f)
#pragma unroll
        for (int b = 0; b < FC; ++b)
          acc.c[f][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[f][s], o.b[s][b], acc.c[f][b], 0, 0, 0);
  }
  static __device__ __forceinline__ void clear(Acc& acc) {
#pragma unroll
    for (int f = 0; f < FR; ++f)
#pragma unroll
      for (int b = 0; b < FC; ++b) acc.c[f][b] = tile_v16f{};
  }
  // Tile row of register r of row block f, and the lane's tile column of column block b (without BT
  // the FC blocks' columns are consecutive).
  static __device__ __forceinline__ int row(int f, int r, int wr, int lane) {
    return 32 * (FR * wr + f) + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
  }
  static __device__ __forceinline__ int col(int wc, int lane, int b = 0) {
    return 32 * FC * wc + (BT ? 32 * b + (lane & 31) : FC * (lane & 31) + b);
  }
};

}  // namespace cdclq
