// How the kernel gradient of the product on the sphere (s2_mm_real.hip) cuts a row of features.  Plain C++: the rule is checked on the host.
#pragma once

namespace s2cnn {

constexpr int GRADY_KC = 8;       // input features per register pass

// Lanes of a slice: up to 64, the tiles of a row as even as they come, and narrower ones (9 to 16 lanes, or wider where that suffices) while
// there are fewer than four workgroups for each CU.  The passes over the input features are workgroups too: 16 degrees, batch 32, 6 -> 100
// takes 59 us with 256 workgroups of 25 lanes and 40 with 512 of 13; 32 -> 100, 4 passes, 63 with 1024 of 25 and 77 with 2048 of 13.
// At least 4 lanes, so at most 64 slices: with 256 of one lane 13 degrees, batch 7, 8 -> 4 took 14 us, with 64 of 4 it takes 9.
inline int grady_lanes(int nl, int f_in, int fov) {
  const long workgroups = (long)nl * nl * ((f_in + GRADY_KC - 1) / GRADY_KC);
  int tiles = (fov + 63) / 64;
  while (workgroups * tiles < 1024 && fov > 16 * tiles) tiles *= 2;
  const int even = (fov + tiles - 1) / tiles;
  return even < 4 ? 4 : even;
}

}  // namespace s2cnn
