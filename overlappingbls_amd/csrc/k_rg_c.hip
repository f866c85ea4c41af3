// Line kernels of lengths 108, 128 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_108() { return rg_make<108>(); }
const RgTable* rg_table_128() { return rg_make<128>(); }
}  // namespace les
