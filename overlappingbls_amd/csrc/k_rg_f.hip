// Line kernels of lengths 288, 384 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_288() { return rg_make<288>(); }
const RgTable* rg_table_384() { return rg_make<384>(); }
}  // namespace les
