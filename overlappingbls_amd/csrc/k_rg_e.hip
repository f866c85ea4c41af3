// Line kernels of lengths 216, 256 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_216() { return rg_make<216>(); }
const RgTable* rg_table_256() { return rg_make<256>(); }
}  // namespace les
