// Row-block linear layers with split inputs, transforms on load or a separate initial sum
// (rows_gemm.h, input mode 2).
#include "rows_gemm.h"

int face::launch_rows_op(const RowsCtx& c, int NW, int NB, int xcd_order) {
    return launch_rows_xm<2>(c, NW, NB, xcd_order);
}
