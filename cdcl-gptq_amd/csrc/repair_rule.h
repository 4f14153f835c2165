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
// for 32 columns and fewer (the descent of 8192 x 4096 in sub-blocks of 32, two passes: 10.3 ms against 14.1; of
// 1024 x 4096, where 64 x 64 tiles are taken: 4.15 ms with either).
inline GradTile grad_tile(long units, int wd, int cus) {
  const long t128 = (wd + 127) / 128, t64 = (wd + 63) / 64;
  if (2 * units * t128 >= 5L * cus && 19 * 2 * t128 <= 20 * t64) return GRAD_128x128;
  if (units * t64 < cus) return GRAD_64x64;
  return wd <= 32 ? GRAD_128x32 : GRAD_128x64;
}

// Whether the refit of `rows` rows in groups of g runs a KC panel of groups per launch (k_panel.hip,
// k_refit_panel) and not a launch pair per group. The groups have to lie inside the panels: 16, 32, 64 or 128
// columns, or one group of all n <= 128. A panel launch keeps one workgroup of at most 16 rows a CU where the
// per-group refit keeps two of up to 64, so what it saves in launches it loses again in rounds: groups of
// two 64-column pieces from the third round on (refit of one pass and the last, groups of 128: 8192 x
// 2048 3.11 against 3.15 ms, 12288 x 2048 4.46 and 4.10, 14336 x 4096 17.5 and 15.5, 131072 x 512 6.67 and 4.53),
// one group alone, which saves a single launch, from the fifth (131072 x 64 0.58 and 0.51; 16384 x 64 0.157 and
// 0.161); several groups of 64 and less to a panel never (131072 x 256, groups of 16, 7.31 and 7.44).
inline bool refit_panel_ok(int n, int g, int rows, int cus) {
  if (!(g <= 128 && (g >= n || g == 128 || (g >= 16 && 64 % g == 0)))) return false;
  if (g > 64) return rows <= 32L * cus;
  return g < n || rows <= 64L * cus;
}

}  // namespace cdclq
