// Split-K builds on the 16x16x32 loop. No plan names them: a launch of a
// 128x128 split-K plan runs on them (csrc/runtime/grid_split.h), with the
// general loop's results bit for bit (both add an element's products in the
// same k order).
#include "gemm_mfma16g.h"

namespace tbk {
#define TBK_M16_SPLIT(BM, BN, BK, WGM, WGN, ST, OUT)                                       \
  {{BM, BN, BK, WGM, WGN, OUT, ST, 0, 1},                                                 \
   reinterpret_cast<const void *>(&gemm_mfma16g_split<BM, BN, BK, WGM, WGN, ST, OUT>),    \
   "tb_gemm_gfx950_" #BM "x" #BN "x" #BK "_w" #WGM "x" #WGN "_s" #ST "_out" #OUT          \
   "_16x16x32_split",                                                                     \
   Mfma16GTile<BM, BN, BK, WGM, WGN, ST>::VM_PROLOGUE,                                    \
   Mfma16GTile<BM, BN, BK, WGM, WGN, ST>::VM_LOOP, 0, nullptr, 0}
static const KernelEntry kSplit[] = {TBK_M16_SPLIT(128, 128, 64, 2, 2, 3, 1),
                                     TBK_M16_SPLIT(128, 128, 64, 2, 2, 3, 3)};
#undef TBK_M16_SPLIT

const KernelEntry *find_split_kernel(const KernelKey &k) {
  for (const KernelEntry &e : kSplit)
    if (e.key.bm == k.bm && e.key.bn == k.bn && e.key.bk == k.bk && e.key.wgm == k.wgm &&
        e.key.wgn == k.wgn && e.key.out == k.out && e.key.stages == k.stages)
      return &e;
  return nullptr;
}
} // namespace tbk
