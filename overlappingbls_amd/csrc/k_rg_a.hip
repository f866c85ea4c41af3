// Line kernels of lengths 16, 24, 32, 36, 48 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_16() { return rg_make<16>(); }
const RgTable* rg_table_24() { return rg_make<24>(); }
const RgTable* rg_table_32() { return rg_make<32>(); }
const RgTable* rg_table_36() { return rg_make<36>(); }
const RgTable* rg_table_48() { return rg_make<48>(); }
}  // namespace les
