// Which kernels phase 2 takes (src/engine.rs:534-670), by the sizes of the work alone: plain host rules,
// without HIP, so that they can be tested anywhere.
#pragma once

namespace cdclq {

// Tile of the repair gradient's direct-to-LDS GEMM (k_repair.hip, k_grad).
enum GradTile { GRAD_128x128, GRAD_128x64, GRAD_64x64, GRAD_128x32 };

// units = 128-row tiles times panels, wd columns on a device of `cus` CUs. 128 x 128 tiles from 2.5 a CU (2048 x
// 5632, 2.6 a CU: 58.1 us against 61.4 on 128 x 64; 5632 x 2048, 2.4 a CU: 57.4 against 52.0) and only where
// they compute at most a twentieth more columns than the 64-column ones, which is what their rate is ahead; 64
// x 64 ones where 128 x 64 tiles would leave CUs without one (1001 x 1350: 14.2 against 14.8 us); 128 x 32 ones
// for 32 columns and fewer while 64 x 64 ones would be more than a CU each (the descent of 8192 x 4096 in
// sub-blocks of 32, two passes: 10.3 ms against 14.1; the refit of 1920 x 3552 in groups of 8 20.0 against 23.5, of
// 64 x 3552 18.0 and 17.9).
inline GradTile grad_tile(long units, int wd, int cus) {
  const long t128 = (wd + 127) / 128, t64 = (wd + 63) / 64;
  if (2 * units * t128 >= 5L * cus && 19 * 2 * t128 <= 20 * t64) return GRAD_128x128;
  if (wd <= 32) return 2 * units > cus ? GRAD_128x32 : GRAD_64x64;
  return units * t64 >= cus ? GRAD_128x64 : GRAD_64x64;
}

// The units of an XCD: its workgroups, `stride` of the `grid` (workgroup w runs on XCD w % nx), take units first,
// first + 1, .. end - 1 in turn. In proportion to the workgroups, not an nx-th each: with a workgroup per unit
// and a grid that nx does not divide, an XCD would have had more units than workgroups and the launch taken two
// units' time (64 x 3552 in groups of 8, 28 units: 16.7 us a launch, 9.6 so; the refit of 640 x 1536's descent in
// sub-blocks of 48 2.38 -> 1.62 ms).
struct GradShare {
  int first, end, stride;
};
#ifdef __HIP__
__host__ __device__
#endif
inline GradShare grad_share(int xcd, int grid, int nx, int units) {
  const int per = grid / nx, more = grid % nx;
  const int w0 = xcd * per + (xcd < more ? xcd : more), n = per + (xcd < more);
  return {(int)((long)w0 * units / grid), (int)((long)(w0 + n) * units / grid), n};
}

// Whether the refit of `rows` rows in groups of g runs a KC panel of groups per launch (k_panel.hip,
// k_refit_panel) and not a launch pair per group. The groups have to lie inside the panels: 16, 32, 64 or 128
// columns, or one group of all n <= 128. A panel launch keeps one workgroup of at most 16 rows a CU where the
// per-group refit keeps two of up to 64, so what it saves in launches it loses again in rounds: groups of
// two 64-column pieces from the third round on (refit of one pass and the last, groups of 128: 8192 x
// 2048 3.11 against 3.15 ms, 12288 x 2048 4.46 and 4.10, 14336 x 4096 17.5 and 15.5, 131072 x 512 6.67 and 4.53),
// in wide layers, where the gradient leaves the launches little, from the second (7000 x 6000 17.9 and 19.3,
// 5000 x 8192 25.0 and 22.9, 4096 x 8192 18.7 and 19.0),
// one group alone, which saves a single launch, from the fifth (131072 x 64 0.58 and 0.51; 16384 x 64 0.157 and
// 0.161); several groups of 64 and less to a panel never (131072 x 256, groups of 16, 7.31 and 7.44).
inline bool refit_panel_ok(int n, int g, int rows, int cus) {
  if (!(g <= 128 && (g >= n || g == 128 || (g >= 16 && 64 % g == 0)))) return false;
  if (g > 64) return rows <= (n <= 6144 ? 32L : 16L) * cus;
  return g < n || rows <= 64L * cus;
}

// Whether the descent may run a KC panel of sub-blocks per launch (k_panel.hip, k_cd_panel) and not a launch
// pair per sub-block: sub-blocks of 64, or one of all n <= 64. Narrow layers save few launches, and from
// many rows on lose more in rounds of 16 rows a CU (repair of three passes with the refit: 16384 x 64
// 0.399 against 0.374 ms a sub-block at a time, 12288 x 64 0.350 and 0.356, 16384 x 128 0.579 and 0.559, 32768 x
// 256 1.320 and 1.314, 65536 x 256 2.28 and 2.20, 65536 x 512 5.29 and 5.24; 131072 x 1024 27.6 and 28.9).
inline bool cd_panel_ok(int n, int sbw, int rows, int cus) {
  if (!(sbw == 64 || (sbw >= n && n <= 64))) return false;
  return n > 512 || rows <= (n <= 128 ? 48L : 96L) * cus;
}

// Which of the two a panel takes in one pass: tiles[i] 128-row tiles take part in its i-th of nsub sub-blocks,
// `both` of them in any, out of np panels. The panel form computes all of its columns' gradient for every
// such tile, so a sparse selection (refine_frac < 1, chunks that have converged) pays for columns that
// no row uses; a sub-block at a time computes those alone. In tiles of 128 x 64 times panels (36 ns of the
// whole device, an eighth more in 64-column launches; a launch takes at least half a device of them): the panel form does best while p < q, with
// what j selected sub-blocks save in sweeps and launches, less what a round of 16-row workgroups adds, and
// from the second round on adds again where further sweeps of a sub-block make its rows differ more.
// Descent alone, two passes, in panels / a sub-block at a time / by this rule: 14336 x 4096, three
// quarters selected 9.43 / 9.52 / 8.95 ms, a tenth 2.31 / 1.77 / 1.75, 3% 1.51 / 0.85 / 0.86; 4096 x 4096, a quarter
// 1.36 / 1.40 / 1.20; 1024 x 2048, a tenth 0.237 / 0.296 / 0.224. Two sweeps, repair of one pass, in panels / a
// sub-block at a time: 45528 x 960 5.91 / 5.41, 14336 x 4096 18.9 / 18.5 (ten passes 118.7 / 120.2), 4096 x 1024
// 1.03 / 1.18.
inline bool cd_panel_pays(const int* tiles, int nsub, int both, int np, int rows, int sweeps, int cus) {
  if (np == 1) return true;  // no gradient of other panels
  const long least = cus / 2;
  long j = 0, q = 0;
  for (int i = 0; i < nsub; ++i) {
    if (tiles[i] == 0) continue;
    const long t = (long)tiles[i] * np;
    q += t > least ? t + t / 8 : least;
    ++j;
  }
  long p = (long)nsub * both * (np - 1);
  if (p < least) p = least;
  const long rounds = (rows + 16L * cus - 1) / (16L * cus);
  const long again = sweeps > 1 ? cus * j * (rounds - 1) / 4 : 0;
  return p < q + cus * (2 * j - 3) / 2 - cus * j * rounds / 25 - again;
}

}  // namespace cdclq
