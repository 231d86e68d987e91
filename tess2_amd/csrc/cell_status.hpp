// cell_status.hpp -- per-cell outcome codes (TESS2_CELL_* of the C ABI).
#pragma once

namespace t2 {

enum { ST_SCAN = 0, ST_CIC = 1, ST_INCOMPLETE = 2, ST_OUTSIDE = 3, ST_DEGENERATE = 4 };

}  // namespace t2
