// What the host decides about a launch of the one-pass kernel, shared by the translation unit that decides (gemv_wide.hip)
// and the ones that launch (gemv_wide_<format>.hip through lowbit_gemv_wide.h).  No kernel code in here.
#pragma once
#include "lowbit_formats.h"

namespace lowbit {

struct WideShape {
    int r, waves;       // tile rows per workgroup (0: another kernel), waves at most
    int mb = 0;         // 16-row blocks of x per workgroup; 0: all of up to 64 rows
};

// Whether the fused gate/up form with two tile rows of either weight has the registers for mb 16-row blocks of x: with four it
// spills in all but nf4 and fp16 sym_int4 (56 rows on [8192 x 4096], one tile row / two: sym_int8 27.5 / 57.7 us, asym_int4
// 27.6 / 43.3, fp8_e4m3 26.7 / 30.6; nf4 27.7 / 25.2), and it is not built for those.
constexpr bool wide_mlp_two_rows(int qtype, bool f16, int mb) { return mb < 4 || qtype == QT_NF4 || (qtype == QT_SYM_INT4 && f16); }

}  // namespace lowbit
