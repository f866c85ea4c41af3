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

// vorticity pads: half the lines, in FP32 twice the threads unless one line;
// advection unpads: twice the threads
template <typename T, int N, int M>
constexpr bool fused_is(int lines, int threads) {
    return fused_lines<T, N, M>() == lines && fused_threads<T, N, M>() == threads;
}
static_assert(fused_is<double, 256, 384>(2, 64), "");
static_assert(fused_is<float, 256, 384>(2, 128), "");
static_assert(fused_is<float, 384, 576>(1, 128), "");
static_assert(fused_is<float, 512, 768>(1, 128), "");
static_assert(fused_is<double, 512, 768>(1, 128), "");
static_assert(fused_is<double, 384, 256>(5, 256), "");
static_assert(fused_is<float, 768, 512>(1, 256), "");
