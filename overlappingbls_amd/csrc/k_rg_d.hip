// Line kernels of lengths 144, 192 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_144() { return rg_make<144>(); }
const RgTable* rg_table_192() { return rg_make<192>(); }
}  // namespace les
