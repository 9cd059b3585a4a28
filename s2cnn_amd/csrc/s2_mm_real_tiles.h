// How the kernel gradient of the product on the sphere (s2_mm_real.hip) cuts a row of features and its sums.  Plain C++: the rule is checked on the host.
#pragma once

namespace s2cnn {

constexpr int GRADY_KC = 8;       // input features per register pass
struct GradySplit { int lanes, slices; };      // a workgroup of 256: slices of so many lanes, and how many of them

// Lanes: up to 64, the tiles of a row as even as they come, and narrower ones (9 to 16 lanes, or wider where that suffices) while there are fewer
// than four workgroups for each CU and a slice still gets five (row, batch item) pairs of the largest degree, or while there are CUs without any.
// The passes over the input features are workgroups too: 16 degrees, batch 32, 6 -> 100 takes 32 us with 256 workgroups of 25 lanes and 23 with
// 512 of 13; 32 -> 100, 4 passes, 40 with 1024 of 25 and 52 with 2048 of 13.  Few pairs: 22 degrees, batch 2, 4 -> 46: 4.9 with 23 lanes, 5.4 with
// 12; 18 degrees, batch 2, 7 -> 148: 5.8 with 19, 8.3 with 10; 16 degrees, batch 4, 6 -> 100: 5.9 with 25, 5.5 with 13.  CUs without work: 3 degrees,
// batch 7, 5 -> 224: 5.6 with 9 workgroups of 56 lanes, 4.5 with 36 of 14; 5 degrees, batch 3, 60 -> 204: 5.3 with 200 of 51, 4.8 with 400 of 26.
// At least 4 lanes, so at most 64 slices: 13 degrees, batch 64, 8 -> 4 takes 18 us with 256 of one lane, 14 with 64 of 4.
// Slices: no more than give each four pairs, which a lane loads together: 10 degrees, batch 4, 1 -> 20: 5.6 us with 51 slices, 4.7 with 19;
// 14 degrees, batch 4, 49 -> 4: 11.2 with 64, 8.6 with 27.
inline GradySplit grady_split(int nl, int nbatch, int f_in, int fov) {
  const long workgroups = (long)nl * nl * ((f_in + GRADY_KC - 1) / GRADY_KC), pairs = (2L * nl - 1) * nbatch;
  int tiles = (fov + 63) / 64;
  while (workgroups * tiles < 1024 && fov > 16 * tiles && (workgroups * tiles < 256 || pairs * ((fov + 2 * tiles - 1) / (2 * tiles)) >= 5 * 256)) tiles *= 2;
  const int even = (fov + tiles - 1) / tiles, lanes = even < 4 ? 4 : even;
  const long share = (pairs + 3) / 4;
  return {lanes, share < 256 / lanes ? (int)share : 256 / lanes};
}

}  // namespace s2cnn
