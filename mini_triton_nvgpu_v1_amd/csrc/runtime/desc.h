// Internal definition of the opaque tb_gemm_desc (include/tb_gfx950.h).
#pragma once

#include "tb_gfx950.h"

#include <cstddef>
#include <memory>
#include <string>
#include <vector>

namespace tbk {
struct KernelEntry;
}
struct tb_gemm_desc;

// One kernel launch of a descriptor that runs as several rectangles of C: the
// rectangle's own descriptor and its first row and column.
struct tb_gemm_part {
  std::unique_ptr<tb_gemm_desc> desc;
  int64_t row0 = 0, col0 = 0;
};

struct tb_gemm_desc {
  tb_gemm_config cfg{};
  const tbk::KernelEntry *entry = nullptr;
  int out_mode = 0;
  int64_t tiles_m = 0, tiles_n = 0, tiles_k = 0;
  int64_t total_work = 0;
  int64_t lds_bytes = 0;
  size_t workspace_bytes = 0;
  // the launches this descriptor runs in place of its own (grid_split.h);
  // empty: one launch as configured
  std::vector<tb_gemm_part> parts;
};

namespace tbrt {
// Validates a flattened config and binds it to a compiled kernel instance
// (`part`: one of a plan's launches, choose_parts).
int create_desc(const tb_gemm_config &c, tb_gemm_desc **out, bool part);
// Gives a planned descriptor the launches its problem runs best as
// (grid_split.h); a descriptor made from a configuration runs that
// configuration's own kernel.
void choose_parts(tb_gemm_desc *d);
// Sets the thread-local message returned by tb_last_error().
void set_error(const std::string &msg);
// The s_waitcnt depths compiled into the descriptor's kernel instance:
// {vmcnt at the prologue, vmcnt at the per-k-tile barrier, lgkmcnt there}.
void desc_waits(const tb_gemm_desc *d, int64_t out[3]);
} // namespace tbrt
