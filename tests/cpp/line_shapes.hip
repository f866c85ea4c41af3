// The launch shapes that the comments of lines_rg.hpp give measurements for.
#include "../../overlappingbls_amd/csrc/lines_rg.hpp"

using namespace les;

template <typename T, int M, int N>
constexpr bool cross_is(int levels, bool tables_in_lds, int threads) {
    using S = CrossShape<T, M, N>;
    return S::NLV == levels && S::TWL == tables_in_lds && S::NTH == threads;
}
static_assert(cross_is<double, 384, 256>(3, true, 256), "");
static_assert(cross_is<float, 384, 256>(3, true, 256), "");
static_assert(cross_is<double, 576, 384>(2, true, 448), "");
static_assert(cross_is<float, 576, 384>(2, true, 448), "");
static_assert(cross_is<double, 768, 512>(1, false, 320), "");
static_assert(cross_is<float, 768, 512>(1, true, 320), "");
