// Line kernels of lengths 512 (lines_rg.hpp).
#include "lines_rg.hpp"

namespace les {
const RgTable* rg_table_512() { return rg_make<512>(); }
}  // namespace les
