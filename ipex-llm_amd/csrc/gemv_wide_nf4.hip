// The one-pass kernel for 9 .. 64 rows of x, nf4 weights (see lowbit_gemv_wide.h).
#include "lowbit_gemv_wide.h"

namespace lowbit {
template int launch_wide_q<QT_NF4>(const void *, const void *, const void *, void *, int, int, int, int, int, const WideShape &, hipStream_t);
template int launch_wide_mlp_q<QT_NF4>(const void *, const void *, const void *, void *, int, int, int, int, int, const WideShape &,
                                    hipStream_t);
}  // namespace lowbit
