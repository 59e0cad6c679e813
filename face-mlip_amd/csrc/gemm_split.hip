// Row-block linear layers with split inputs or a separate initial sum (rows_gemm.h, input mode 2).
#include "rows_gemm.h"

int face::launch_rows_split(const RowsCtx& c, RowsShape S) { return launch_rows_xm<2>(c, S); }
