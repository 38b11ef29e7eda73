// The rectangles a plan's launch runs (csrc/runtime/grid_split.h) tile C
// exactly, on whole planned tiles, for random plans of every shape and order;
// split-K plans keep their splits, persistent plans of fewer programs than CUs
// run as they are, a plan and its transpose are predicted the same time, and
// f32 C += A*B never moves to the kernel that adds the prior C in its loop;
// plans that measured slower on another tile stay as they are.
#include "runtime/grid_split.h"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <utility>

#define CHECK(x)                                                                            \
  do {                                                                                      \
    if (!(x)) {                                                                             \
      std::printf("FAILED: %s (%lld x %lld x %lld on %lld x %lld, mapping %d)\n", #x,      \
                  (long long)c.m, (long long)c.n, (long long)c.k, (long long)c.block_m,     \
                  (long long)c.block_n, c.mapping);                                         \
      std::exit(1);                                                                         \
    }                                                                                       \
  } while (0)

static int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// the hand-scheduled 256x256 kernel, where it adds the prior C in its loop
static bool early_c(const tb_gemm_config &c) {
  return c.block_m == 256 && c.block_n == 256 && c.block_k == 64 && c.wave_grid_m == 2 &&
         c.wave_grid_n == 2 && c.stages == 2 && c.mfma == TB_MFMA_16X16X32 &&
         c.k % 64 == 0 && c.k >= 18 * 64;
}

static bool other_kernel(const tb_gemm_config &a, const tb_gemm_config &b) {
  return a.block_m != b.block_m || a.block_n != b.block_n || a.block_k != b.block_k ||
         a.stages != b.stages || a.wave_grid_m != b.wave_grid_m ||
         a.wave_grid_n != b.wave_grid_n || a.mfma != b.mfma;
}

static tb_gemm_config plan(int64_t m, int64_t n, int64_t k, int64_t bm, int64_t bn,
                           int64_t waves, int64_t wgm, int64_t stages, int mfma,
                           bool accumulate, int act) {
  tb_gemm_config c{};
  c.m = m, c.n = n, c.k = k;
  c.block_m = bm, c.block_n = bn, c.block_k = 64;
  c.num_waves = waves, c.wave_grid_m = wgm, c.wave_grid_n = waves / wgm;
  c.stages = stages, c.mfma = mfma, c.split_k = 1, c.group_m = 8;
  c.mapping = TB_MAP_GROUPED_TILE;
  c.num_programs = ceil_div(m, bm) * ceil_div(n, bn);
  c.c_dtype = accumulate ? TB_DTYPE_F32 : TB_DTYPE_F16;
  c.acc_init = accumulate ? TB_ACC_INIT_LOAD_C : TB_ACC_INIT_ZERO;
  c.epi_activation = act;
  return c;
}

// Plans that measured 12 to 35% longer on the coarser tile they were moved to:
// several workgroups per CU, f32 C += A*B, an activation.
static void stays_as_planned(const tb_gemm_config &c) { CHECK(tbrt::split_grid(c).empty()); }

// The order of a moved grid of fewer tiles than CUs: neighbours on one XCD
// for a wide problem, dealt out where that order reads as little.
static void moves_in_order(const tb_gemm_config &c, int xcd_remap) {
  const std::vector<tbrt::GridPart> parts = tbrt::split_grid(c);
  CHECK(parts.size() == 1 && parts[0].cfg.num_programs < 256);
  CHECK(parts[0].cfg.xcd_remap == xcd_remap);
}

int main() {
  const int m32 = TB_MFMA_32X32X16, m16 = TB_MFMA_16X16X32, gelu = TB_ACT_GELU_TANH;
  stays_as_planned(plan(231, 7480, 552, 64, 64, 4, 2, 2, m32, false, 0));
  stays_as_planned(plan(3609, 4400, 192, 64, 128, 4, 1, 2, m32, true, 0));
  stays_as_planned(plan(146, 14728, 1984, 64, 64, 4, 2, 2, m32, true, gelu));
  moves_in_order(plan(218, 2968, 2456, 128, 128, 4, 2, 3, m16, false, gelu), 8);
  moves_in_order(plan(41, 12904, 1464, 128, 128, 4, 2, 3, m16, false, 0), 8);
  moves_in_order(plan(1795, 568, 1680, 256, 256, 4, 2, 2, m16, false, 0), 0);
  std::mt19937 rng(7);
  const int blocks[] = {64, 128, 192, 256};
  int whole = 0, cut = 0, moved = 0;
  for (int i = 0; i < 20000; ++i) {
    tb_gemm_config c{};
    c.m = 1 + rng() % (1u << (4 + rng() % 13));
    c.n = 8 * (1 + rng() % (1u << (1 + rng() % 13)));
    c.k = 8 * (1 + rng() % 1000);
    c.block_m = blocks[rng() % 4];
    c.block_n = blocks[rng() % 4];
    c.block_k = rng() % 2 ? 64 : 32;
    c.num_waves = 1 << rng() % 4;
    c.stages = 2 + rng() % 3;
    c.mapping = rng() % 5;
    c.group_m = 8;
    c.split_k = c.mapping == TB_MAP_SPLIT_K ? 4 : 1;
    const bool accumulate = rng() % 2; // f32 C += A*B
    c.c_dtype = accumulate ? TB_DTYPE_F32 : TB_DTYPE_F16;
    c.acc_init = accumulate ? TB_ACC_INIT_LOAD_C : TB_ACC_INIT_ZERO;
    if (rng() % 2)
      c.k = (c.k + 63) / 64 * 64;
    c.wave_grid_m = c.num_waves >= 4 ? 2 : 1;
    c.wave_grid_n = c.num_waves / c.wave_grid_m;
    c.mfma = c.mapping != TB_MAP_SPLIT_K && rng() % 2 ? TB_MFMA_16X16X32 : TB_MFMA_32X32X16;
    const int64_t tiles = ceil_div(c.m, c.block_m) * ceil_div(c.n, c.block_n);
    const bool persistent =
        c.mapping == TB_MAP_PERSISTENT_TILE || c.mapping == TB_MAP_PERSISTENT_GROUPED;
    c.num_programs = persistent ? std::min<int64_t>(tiles, 1 + rng() % 512) : tiles * c.split_k;
    const std::vector<tbrt::GridPart> parts = tbrt::split_grid(c);
    // the transposed problem on the transposed tile is the same grid
    tb_gemm_config t = c;
    std::swap(t.m, t.n);
    std::swap(t.block_m, t.block_n);
    std::swap(t.wave_grid_m, t.wave_grid_n);
    CHECK(c.block_m == c.block_n || tbrt::planned_us(c, c.m, c.n) == tbrt::planned_us(t, t.m, t.n));
    // one launch in place of the planned one is another kernel
    if (parts.size() == 1)
      CHECK(other_kernel(parts[0].cfg, c));
    if (persistent && c.num_programs < 256)
      CHECK(parts.empty());
    if (c.mapping == TB_MAP_SPLIT_K) { // as planned but for the stages
      for (const tbrt::GridPart &p : parts) {
        CHECK(p.row0 == 0 && p.col0 == 0 && p.cfg.stages == 3);
        CHECK(c.stages == 2 || p.cfg.mfma == TB_MFMA_16X16X32);
        CHECK(p.cfg.m == c.m && p.cfg.n == c.n && p.cfg.split_k == c.split_k &&
              p.cfg.reduction == c.reduction && p.cfg.num_programs == c.num_programs);
      }
      CHECK(parts.size() <= 1);
      continue;
    }
    CHECK(parts.size() <= 2);
    int64_t area = 0;
    for (const tbrt::GridPart &p : parts) {
      CHECK(p.row0 % c.block_m == 0 && p.col0 % c.block_n == 0);
      CHECK(p.cfg.m > 0 && p.cfg.n > 0 && p.row0 + p.cfg.m <= c.m && p.col0 + p.cfg.n <= c.n);
      CHECK(p.cfg.k == c.k && p.cfg.split_k == 1 && p.cfg.n % 8 == 0);
      CHECK(p.cfg.c_dtype == c.c_dtype && p.cfg.acc_init == c.acc_init);
      // the kernel that adds the prior C inside its first k-tiles serves only
      // plans that name it
      if (accumulate && early_c(p.cfg))
        CHECK(early_c(c));
      moved += accumulate && p.cfg.block_m != c.block_m;
      const int64_t t = ceil_div(p.cfg.m, p.cfg.block_m) * ceil_div(p.cfg.n, p.cfg.block_n);
      const bool pers = p.cfg.mapping == TB_MAP_PERSISTENT_TILE ||
                        p.cfg.mapping == TB_MAP_PERSISTENT_GROUPED;
      CHECK(pers ? p.cfg.num_programs <= t : p.cfg.num_programs == t);
      // a moved grid that fills the chip runs neighbours on one XCD
      if (t >= 256 && (parts.size() == 1 || &p == &parts[1]))
        CHECK(p.cfg.xcd_remap == 8);
      area += p.cfg.m * p.cfg.n;
    }
    if (parts.size() == 2) { // side by side: the second starts where the first ends
      const tbrt::GridPart &a = parts[0], &b = parts[1];
      CHECK(a.row0 == 0 && a.col0 == 0);
      CHECK((b.row0 == a.cfg.m && b.col0 == 0 && b.cfg.n == c.n) ||
            (b.col0 == a.cfg.n && b.row0 == 0 && b.cfg.m == c.m));
      CHECK(a.cfg.block_m == c.block_m && a.cfg.mapping == c.mapping);
    }
    CHECK(parts.empty() || area == c.m * c.n);
    whole += parts.size() == 1;
    cut += parts.size() == 2;
  }
  if (whole < 1000 || cut < 10 || moved < 500) {
    std::printf("FAILED: only %d whole, %d cut and %d moved C += A*B problems\n", whole, cut,
                moved);
    return 1;
  }
  std::printf("ok: %d whole, %d cut, %d moved\n", whole, cut, moved);
  return 0;
}
