// An expert's units of 16 rows cut into even tiles (moe_rows_kernel).  No product of units and tiles: both grow with the rows, and past three million rows of one
// expert 32 bits do not hold it.
#pragma once

namespace sgl_amd {

struct RowTile {
  int from, units;
};

// tile k of `tiles` over `all` units: the first all % tiles tiles have one unit more
__host__ __device__ inline RowTile even_tile(int all, int tiles, int k) {
  const int each = all / tiles, over = all - each * tiles;
  return RowTile{k * each + (k < over ? k : over), each + (k < over ? 1 : 0)};
}

}  // namespace sgl_amd
