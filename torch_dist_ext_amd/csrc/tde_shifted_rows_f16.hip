// f16 row kernels for rows that start anywhere in a line of memory.
#include "tde_rows.h"

namespace tde {

hipError_t launch_shifted_rows_f16(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    return launch_rows_e<ElemF16, true>(n, vpt, q, wn, a, g, s);
}

} // namespace tde
