// Instantiates the row kernels for one element type (f32) so the three types compile in parallel.
#include "tde_rows.h"

namespace tde {

hipError_t launch_rows_f32(int n, int vpt, int q, bool wn, const RowArgs &a, const Geometry &g, hipStream_t s) {
    return launch_rows_e<ElemF32, false>(n, vpt, q, wn, a, g, s);
}

hipError_t launch_reduce_f32(int n, const RowArgs &a, uint64_t table, int64_t row_bytes, int64_t first_row, int64_t row_step, int64_t rows,
                             hipStream_t s) {
    return launch_reduce_e<ElemF32>(n, a, table, row_bytes, first_row, row_step, rows, s);
}

} // namespace tde
