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

}  // namespace cdclq
