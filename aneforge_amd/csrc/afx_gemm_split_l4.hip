// The split GEMM's kernels for one weight format (afx_gemm_split.h).
#include "afx_gemm_split.h"

namespace afx {
template split_fn pick_split<FMT_L4>(int, int);
}
