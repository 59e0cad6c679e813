// Row-block linear layers with transforms of the input on load (rows_gemm.h, input mode 3).
#include "rows_gemm.h"

int face::launch_rows_op(const RowsCtx& c, RowsShape S) { return launch_rows_xm<3>(c, S); }
