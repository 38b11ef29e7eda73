// 16x16x32 instances of one block shape of TBK_M16_SHAPES (gemm_tiles.h):
// TBK_SHAPE names the list, TBK_OUT the output mode (0: f16 C, 1: plain f32
// C, 2: f32 C += A*B), TBK_EPI=0 instantiates it plain and TBK_EPI=1 with the
// fused epilogue steps. The Makefile compiles this file once per shape, mode
// and flavour.
#include "gemm_mfma16g.h"
#include "gemm_tiles.h"

#if !defined(TBK_SHAPE) || !defined(TBK_OUT) || !defined(TBK_EPI)
#error "compile with -DTBK_SHAPE=<shape of TBK_M16_SHAPES> -DTBK_OUT=0|1|2 -DTBK_EPI=0|1"
#endif

#define TBK_CAT2(a, b) a##b
#define TBK_CAT(a, b) TBK_CAT2(a, b)
#define TBK_EPI_BOOL TBK_CAT(TBK_EPI_B, TBK_EPI)
#define TBK_EPI_B0 false
#define TBK_EPI_B1 true
#if TBK_EPI
#define TBK_M16_SUFFIX "_16x16x32_epi"
#define TBK_TABLE TBK_CAT(TBK_CAT(TBK_CAT(entries_m16_, TBK_SHAPE), _o), TBK_CAT(TBK_OUT, _epi))
#else
#define TBK_M16_SUFFIX "_16x16x32"
#define TBK_TABLE TBK_CAT(TBK_CAT(TBK_CAT(entries_m16_, TBK_SHAPE), _o), TBK_OUT)
#endif
#define TBK_STR2(x) #x
#define TBK_STR(x) TBK_STR2(x)

#define TBK_M16_ENTRY(BM, BN, BK, WGM, WGN, ST)                                            \
  {{BM, BN, BK, WGM, WGN, TBK_OUT, ST, TBK_EPI, 1},                                       \
   reinterpret_cast<const void *>(                                                        \
       &gemm_mfma16g<BM, BN, BK, WGM, WGN, ST, TBK_OUT, TBK_EPI_BOOL>),                   \
   "tb_gemm_gfx950_" #BM "x" #BN "x" #BK "_w" #WGM "x" #WGN "_s" #ST                      \
   "_out" TBK_STR(TBK_OUT) TBK_M16_SUFFIX,                                                \
   Mfma16GTile<BM, BN, BK, WGM, WGN, ST>::VM_PROLOGUE,                                    \
   Mfma16GTile<BM, BN, BK, WGM, WGN, ST>::VM_LOOP, 0, nullptr, 0}

namespace tbk {
static const KernelEntry kEntries[] = {TBK_CAT(TBK_M16_TILES_, TBK_SHAPE)(TBK_M16_ENTRY)};
const KernelEntry *TBK_TABLE(int *n) {
  *n = sizeof(kEntries) / sizeof(kEntries[0]);
  return kEntries;
}
} // namespace tbk
