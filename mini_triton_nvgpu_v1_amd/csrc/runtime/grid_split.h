// How a planned problem is spread over the chip: the choice of builds and
// sub-problems one launch of a plan runs.
#pragma once

#include "tb_gfx950.h"

#include <cstdint>
#include <vector>

namespace tbrt {

// A rectangle of C computed by one kernel launch: rows row0 .. row0+m-1 and
// columns col0 .. col0+n-1 of the problem, on the configuration `cfg` (whose
// m and n are the rectangle's).
struct GridPart {
  tb_gemm_config cfg;
  int64_t row0 = 0, col0 = 0;
};

// Predicted time in us of an m x n rectangle of the problem on the planned
// tile (0: no estimate for that tile), `share` of the part that depends on
// the tile.
double planned_us(const tb_gemm_config &c, int64_t m, int64_t n, double share = 1);

// The rectangles a planned configuration runs as. Empty: as planned.
std::vector<GridPart> split_grid(const tb_gemm_config &c);

} // namespace tbrt
