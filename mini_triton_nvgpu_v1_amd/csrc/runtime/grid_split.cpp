// The builds and rectangles a plan's launch runs (grid_split.h).
//
// A plan names one macro tile. Run as such, a grid of fewer tiles than CUs
// leaves CUs idle, and a grid of a few more tiles than a multiple of 256 runs
// a last round that is nearly empty: 24 tiles of 256x256 (1000 x 1496 x 712)
// kept 24 of 256 CUs busy for 30 us, and 320 of them (5000 x 4096 x 4104)
// took two rounds, the second a quarter full, 178 us. C does not depend on
// the tile: every build adds the products of an element in the same k order
// in f32 (bit-identical for f16 and plain f32 results; for f32 C += A*B see
// adds_c_early). So the launch of a plan may run the same problem on another
// tile, or cut it in two rectangles: the rows (or columns) that fill whole
// rounds on the planned tile, and the rest on a tile that spreads it over the
// chip.
//
// The choice is by time, from two measured constants per tile: a grid's
// round of up to 256 tiles takes c0 + (K / 64) * c1(fill) us, where c1 rises
// from `lo` (up to half the CUs: the clock is high) to `hi` (all of them:
// the part is power-limited). Measured back to back, f16 C, K = 128 .. 4096:
//   tile     c0    lo     hi     e.g. K = 4096, 32 / 128 / 256 tiles
//   256x256  7.3   0.955  1.37   68.1 / 68.6 / 95.1 us
//   256x128  4.6   0.53   0.79   38.3 / 38.8 / 56.0
//   128x128  4.1   0.333  0.455  25.4 / 25.8 / 33.1
//    64x128  3.7   0.305  0.355  23.2 / 23.5 / 26.6
//    64x64   3.25  0.255  0.262  19.6 / 19.7 / 20.1
// The 64-row tiles fit a CU two or three times, so their further rounds
// overlap: each costs 2.2 and 0.92 us and the K part 0.3 and 0.195 us per 64
// of K and round (1024 tiles, K = 64 / 1024 / 4096: 12.0 / 27.0 / 88.2 us on
// 64x128, 7.0 / 17.6 / 55.3 on 64x64).
// A choice has to save 10% of the planned grid's time by these constants, which
// reproduce the measured times to about 8%.
#include "grid_split.h"

#include <algorithm>
#include <bitset>

namespace tbrt {
namespace {

constexpr int64_t kCus = 256, kXcds = 8;

// A tile the launch may choose: its build, and its cost per round.
struct Build {
  int64_t bm, bn, wgm, wgn, stages;
  int32_t mfma;
  double c0, lo, hi;
  // overlapping rounds: us per round after the first, and per 64 of K and
  // round (0: rounds do not overlap)
  double more, more_k;
};
const Build kBuilds[] = {
    {256, 256, 2, 2, 2, TB_MFMA_16X16X32, 7.3, 0.955, 1.37, 0, 0},
    {256, 128, 4, 2, 3, TB_MFMA_16X16X32, 4.6, 0.53, 0.79, 0, 0},
    {128, 128, 2, 2, 3, TB_MFMA_16X16X32, 4.1, 0.333, 0.455, 0, 0},
    {64, 128, 2, 4, 3, TB_MFMA_32X32X16, 3.7, 0.305, 0.355, 2.2, 0.3},
    {64, 64, 2, 2, 3, TB_MFMA_32X32X16, 3.25, 0.255, 0.262, 0.92, 0.195},
};

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

double round_us(const Build &b, int64_t tiles, double nk) {
  const double fill = (double)tiles / kCus;
  const double rise = std::clamp(2 * fill - 1, 0.0, 1.0);
  return b.c0 + nk * (b.lo + rise * (b.hi - b.lo));
}

int64_t tiles_of(int64_t m, int64_t n, int64_t bm, int64_t bn) {
  return ceil_div(m, bm) * ceil_div(n, bn);
}

// A grid of `tiles` tiles that cost what b's do.
double tiles_us(const Build &b, int64_t tiles, int64_t k) {
  const double nk = (double)ceil_div(k, 64);
  if (b.more > 0 && tiles > kCus) {
    const double rounds = (double)ceil_div(tiles, kCus);
    return b.c0 + (rounds - 1) * b.more + nk * std::max(b.hi, rounds * b.more_k);
  }
  const int64_t full = tiles / kCus, rest = tiles % kCus;
  return (double)full * round_us(b, kCus, nk) + (rest ? round_us(b, rest, nk) : 0);
}

// An m x n problem on build b.
double grid_us(const Build &b, int64_t m, int64_t n, int64_t k) {
  return tiles_us(b, tiles_of(m, n, b.bm, b.bn), k);
}

// The build of the planned tile's shape or of its transpose, which costs the
// same per tile; null: neither.
const Build *build_of(const tb_gemm_config &c) {
  for (const Build &b : kBuilds)
    if ((b.bm == c.block_m && b.bn == c.block_n) ||
        (b.bm == c.block_n && b.bn == c.block_m))
      return &b;
  return nullptr;
}

bool is_build(const tb_gemm_config &c, const Build &b) {
  return c.block_m == b.bm && c.block_n == b.bn && c.block_k == 64 && c.stages == b.stages &&
         c.wave_grid_m == b.wgm && c.wave_grid_n == b.wgn && c.mfma == b.mfma;
}

// The time of the planned grid over its shape's build. A workgroup alone on
// its CU waits for its loads on 2 stages, or issues them too slowly on 1 or 2
// waves, once the k-loop is long (64x64, 256 tiles, K = 2048: 26.9 us on
// 32-deep 2-stage k-tiles, 16.9 on 64-deep ones, 14.6 on 2 waves, 12.7 on
// the build; K = 512: 6.6, 6.4, 7.0, 6.5). With several workgroups per CU
// the stages and waves make little difference. The 256x256 tile is fastest
// on its own build for any K from 512 (256 tiles, K = 512: 19.9 us, the
// other builds 22.5-48).
double over_build(const tb_gemm_config &c, const Build &b) {
  if (is_build(c, b))
    return 1;
  if (b.bm == 256 && b.bn == 256)
    return c.k >= 512 ? 1.15 : 1;
  const int64_t tiles = tiles_of(c.m, c.n, c.block_m, c.block_n);
  return tiles <= kCus && c.k >= 1024 && (c.stages == 2 || c.num_waves < 4) ? 1.2 : 1;
}

// f32 C += A*B: the 256x256 build adds the prior C inside its first 16
// k-tiles (whole k-tiles only, at least 18 of them), the other builds after
// the last one. Every sum after the addition rounds at the larger magnitude:
// at K = 4096 the error against f64 is 1.6 times that of adding C last. So a
// plan on another tile, whose kernel adds C last (or, on small wave tiles not
// staged through LDS, first), never moves there.
bool adds_c_early(const Build &b, const tb_gemm_config &c) {
  return c.acc_init == TB_ACC_INIT_LOAD_C && b.bm == 256 && b.bn == 256 && c.k % 64 == 0 &&
         c.k >= 18 * 64;
}

// What the constants (f16 C, no fused steps) leave out of a grid, in us: the
// prior C of C += A*B and its wider result, 6 bytes per element more at the
// 4.9 TB/s of a copy, and an activation, 5.9 us per round of 256x256 tiles
// (ReLU 1.6), twice that in a C += A*B, which dispatches it per 16-row block.
// Overlapped rounds hide some of it. Without this, 3609 x 4400 x 192, C += A*B
// on 64x128, moved to 256x128: 25.4 -> 34.0 us.
double extra_us(const tb_gemm_config &c, const Build &b, int64_t m, int64_t n, int64_t tiles) {
  const bool accumulate = c.acc_init == TB_ACC_INIT_LOAD_C;
  double us = 0;
  if (accumulate)
    us += 6 * (double)m * (double)n / 4.9e6;
  if (c.epi_activation != TB_ACT_NONE)
    us += (double)ceil_div(tiles, kCus) * (double)(b.bm * b.bn) *
          (c.epi_activation == TB_ACT_RELU ? 2.5e-5 : 9e-5) * (accumulate ? 2 : 1);
  return b.more > 0 && tiles > kCus ? 0.6 * us : us;
}

// From a tile of which several fit a CU, a coarser one has to be predicted 25%
// faster, not 10%: the constants know such grids to about 20% (231 x 7480 x
// 552 on 64x64 in 2 stages: 7.7 us predicted and 8.0 measured, 6.8 and 10.8 on
// 64x128). Of 424 random plans moved to a coarser tile with 10% for all and
// no extra_us, 42 ran more than 5% longer than as planned, up to 1.35x.
double margin(const tb_gemm_config &c, const Build &b) {
  return b.bm * b.bn > c.block_m * c.block_n && build_of(c)->more > 0 ? 0.9 / 0.75 : 1;
}

// An m x n rectangle of plan c's problem on build b, as a candidate.
double build_us(const tb_gemm_config &c, const Build &b, int64_t m, int64_t n) {
  return grid_us(b, m, n, c.k) * margin(c, b) +
         extra_us(c, b, m, n, tiles_of(m, n, b.bm, b.bn));
}

// The finest build within 5% of the fastest: what the constants leave out is
// per element and spreads over more CUs (1000 x 1496 x 712: 8.1 us predicted
// on 128x128, 7.7 on 64x128; 9.9 and 8.3 measured). `c`: the plan, whose K it
// is and whose C += A*B rounding the build may not worsen.
const Build &fastest(const tb_gemm_config &c, int64_t m, int64_t n) {
  auto us = [&](const Build &b) { return build_us(c, b, m, n); };
  auto allowed = [&](const Build &b) {
    return !adds_c_early(b, c) || is_build(c, b);
  };
  const Build *best = nullptr;
  for (const Build &b : kBuilds)
    if (allowed(b) && (!best || us(b) < us(*best)))
      best = &b;
  const double least = us(*best);
  for (const Build &b : kBuilds) // coarse to fine
    if (allowed(b) && us(b) <= 1.05 * least)
      best = &b;
  return *best;
}

// Rows and columns of C (as rows of A, columns of B) that the XCDs of a grid
// of at most 256 tiles read together, in grouped order by eights: blocks are
// dealt to the XCDs in turn, and with `remap` each XCD takes a contiguous run
// of programs (program_of_block and map_program of the kernels).
int64_t xcd_lines(int64_t tm, int64_t tn, int64_t bm, int64_t bn, bool remap) {
  const int64_t nprog = tm * tn, gm = tm > 1 && tn > 1 ? 8 : 1;
  int64_t lines = 0;
  for (int64_t x = 0; x < kXcds; ++x) {
    std::bitset<kCus> rows, cols;
    for (int64_t block = x; block < nprog; block += kXcds) {
      const int64_t pid =
          remap ? x * (nprog / kXcds) + std::min(x, nprog % kXcds) + block / kXcds : block;
      const int64_t first = pid / (gm * tn) * gm, in_group = pid % (gm * tn);
      const int64_t gsz = std::min(tm - first, gm);
      rows.set((size_t)(first + in_group % gsz));
      cols.set((size_t)(in_group / gsz));
    }
    lines += (int64_t)rows.count() * bm + (int64_t)cols.count() * bn;
  }
  return lines;
}

// Whether neighbours of a grid run on one XCD: where that order has the XCDs
// read a quarter less of A and B from memory (218 x 2968 x 2456 on 64x64: 19.8 ->
// 16.2 us; 314 x 3032 x 568: 8.7 -> 7.8; from 80% on the other order was as
// fast or up to 4% faster), or where a single row of tiles shares the cache
// lines of B's rows (41 x 12904 x 1464 on 64x64: 15.1 -> 9.5). A short K (272 to
// 470) gained nothing, a full chip always does.
bool neighbours_on_one_xcd(int64_t tm, int64_t tn, int64_t k, int64_t bm, int64_t bn) {
  if (tm * tn >= kCus)
    return true;
  if (tm * tn < 32 || k < 512)
    return false;
  return tm == 1 ||
         4 * xcd_lines(tm, tn, bm, bn, true) <= 3 * xcd_lines(tm, tn, bm, bn, false);
}

// The configuration of an m x n rectangle of c on build b: a plain grid in
// grouped order.
tb_gemm_config on_build(const tb_gemm_config &c, const Build &b, int64_t m, int64_t n) {
  tb_gemm_config r = c;
  r.m = m;
  r.n = n;
  r.block_m = b.bm;
  r.block_n = b.bn;
  r.block_k = 64;
  r.num_waves = b.wgm * b.wgn;
  r.wave_grid_m = b.wgm;
  r.wave_grid_n = b.wgn;
  r.stages = b.stages;
  r.mfma = b.mfma;
  const int64_t tm = ceil_div(m, b.bm), tn = ceil_div(n, b.bn);
  r.mapping = tm > 1 && tn > 1 ? TB_MAP_GROUPED_TILE : TB_MAP_TILE;
  r.group_m = r.mapping == TB_MAP_GROUPED_TILE ? 8 : 1;
  r.num_programs = tm * tn;
  r.xcd_remap = neighbours_on_one_xcd(tm, tn, c.k, b.bm, b.bn) ? kXcds : 0;
  return r;
}

} // namespace

double planned_us(const tb_gemm_config &c, int64_t m, int64_t n, double share) {
  const Build *b = build_of(c);
  if (!b)
    return 0;
  const int64_t tiles = tiles_of(m, n, c.block_m, c.block_n);
  return share * over_build(c, *b) * tiles_us(*b, tiles, c.k) + extra_us(c, *b, m, n, tiles);
}

std::vector<GridPart> split_grid(const tb_gemm_config &c) {
  if (c.mapping == TB_MAP_SPLIT_K) {
    // The splits stay the plan's. Of workgroups alone on their CUs, 2 stages
    // wait for loads that 3 have in flight (1024^2 x 8200 in 4 atomic splits
    // of 128x128: 36.1 -> 34.5 us, with a workspace 32.0 -> 29.6; 300 x 520 x
    // 10000 in 12: 18.4 -> 16.8); short splits end before it matters. 128x128
    // tiles on 64-deep k-tiles run the 16x16x32 loop's build (34.1 -> 29.8
    // us for the first of these).
    const int64_t k_tiles = ceil_div(c.k, c.block_k) / c.split_k;
    if (c.num_programs > kCus || k_tiles < 8)
      return {};
    GridPart p{c};
    if (c.block_m == 128 && c.block_n == 128 && c.block_k == 64 && c.wave_grid_m == 2 &&
        c.wave_grid_n == 2) {
      p.cfg.mfma = TB_MFMA_16X16X32;
      p.cfg.stages = 3;
      return {p};
    }
    if (c.stages != 2)
      return {};
    p.cfg.stages = 3;
    return {p};
  }
  const bool persistent =
      c.mapping == TB_MAP_PERSISTENT_TILE || c.mapping == TB_MAP_PERSISTENT_GROUPED;
  const int64_t tm = ceil_div(c.m, c.block_m), tn = ceil_div(c.n, c.block_n);
  const int64_t tiles = tm * tn;
  // a persistent plan of fewer programs than CUs asks for a part of the chip
  if (persistent && c.num_programs < kCus)
    return {};
  if (!build_of(c))
    return {};
  double best_us = planned_us(c, c.m, c.n, 0.9);
  std::vector<GridPart> best;

  // the whole problem on another tile, or on the build of the planned one
  const Build &whole = fastest(c, c.m, c.n);
  const double whole_us = build_us(c, whole, c.m, c.n);
  if (!is_build(c, whole) && whole_us < best_us) {
    best_us = whole_us;
    best = {GridPart{on_build(c, whole, c.m, c.n)}};
  }
  // the rows, or columns, of whole rounds as planned and the rest on the
  // tile that is fastest for it
  const int64_t full = tiles / kCus * kCus;
  for (const bool rows : {true, false}) {
    const int64_t per_line = rows ? tn : tm, block = rows ? c.block_m : c.block_n;
    const int64_t cut = full / per_line * block; // rows or columns of the first part
    if (cut == 0 || cut >= (rows ? c.m : c.n))
      continue;
    const int64_t m0 = rows ? cut : c.m, n0 = rows ? c.n : cut;
    const int64_t m1 = rows ? c.m - cut : c.m, n1 = rows ? c.n : c.n - cut;
    const Build &rest = fastest(c, m1, n1);
    // 2 us for what a second launch leaves idle at its start and end
    const double us = planned_us(c, m0, n0) + build_us(c, rest, m1, n1) + 2;
    if (us >= best_us)
      continue;
    best_us = us;
    tb_gemm_config first = c;
    first.m = m0;
    first.n = n0;
    const int64_t programs = ceil_div(m0, c.block_m) * ceil_div(n0, c.block_n);
    first.num_programs = persistent ? std::min(c.num_programs, programs) : programs;
    best = {GridPart{first},
            GridPart{on_build(c, rest, m1, n1), rows ? cut : 0, rows ? 0 : cut}};
  }
  return best;
}

} // namespace tbrt
