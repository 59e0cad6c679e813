// Row-block linear layers with a per-group input scale (rows_gemm.h, input mode 1).
#include "rows_gemm.h"

int face::launch_rows_xs(const RowsCtx& c, RowsShape S) { return launch_rows_xm<1>(c, S); }
