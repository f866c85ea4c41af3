// Line kernels of lengths 64, 72, 96 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_64() { return rg_make<64>(); }
const RgTable* rg_table_72() { return rg_make<72>(); }
const RgTable* rg_table_96() { return rg_make<96>(); }
}  // namespace les
