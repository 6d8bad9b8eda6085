// Height of the two-fluid stage kernel's strips, chosen from the sizes of a batch's members (host code).
#pragma once

namespace spruce {

// Rows per strip for n domains of rows[k] rows and tiles[k] 60-column tiles.  `resident` blocks run at once: a
// block has two wavefronts, of which a SIMD holds two where a member has the curl terms (217 registers),
// else three (167).  A strip costs its rows plus about three (the halo rows it reads, one face and the start
// of the pipeline): the height with the least rounds x cost, the taller of equals.  Measured, RK2 steps with
// curl terms, us, against the height for 1536 blocks: 256x256 46 against 52, 512x512 82 against 107, eight
// 160x200 domains 78 against 103, sixteen domains of 1.64 million cells 426 against 501; strips of 4 rows take 58,
// 105, 102 and 484 there, of 8 rows 73, 98, 93 and 445.
inline int tf_strip_rows_default(const int* rows, const int* tiles, int n, bool curl) {
  const long resident = curl ? 1024 : 1536;
  int best = 1;
  long least = 0;
  for (int R = 1; R <= 64; ++R) {
    long blocks = 0;
    for (int k = 0; k < n; ++k) blocks += (long)tiles[k] * ((rows[k] + R - 1) / R);
    const long cost = (blocks + resident - 1) / resident * (R + 3);
    if (R == 1 || cost <= least) { best = R; least = cost; }
  }
  return best;
}

}  // namespace spruce
