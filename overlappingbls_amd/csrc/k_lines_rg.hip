// Dispatch of the compile-time line lengths (lines_rg.hpp): a table of
// launchers per length, instantiated in k_rg_*.hip.  Lengths without a table
// run the runtime-length kernels of k_lines.hip.
#include "lines_rg.hpp"

namespace les {

// The domain sides with a table: 2^a 3^b, multiples of 4, up to 512, without
// 8, 12, 324 and 432.  A runtime-length kernel makes one LDS round trip per
// radix-4, -3 or -2 stage (five to six for these lengths) where a table's
// makes one or two.  ddx / ddy / pad of 144 x 96 x 98 points in FP64: 9.7 / 6.9 /
// 28.9 us against 26.7 / 27.8 / 70.2 us; of 288 x 288 x 98: 33 / 32 / 107 us
// against 91 / 100 / 266 us.
#define LES_RG_LENGTHS(X) \
    X(16) X(24) X(32) X(36) X(48) X(64) X(72) X(96) X(108) X(128) X(144) X(192) X(216) X(256) X(288) X(384) X(512)

#define RG_DECL(n) const RgTable* rg_table_##n();
LES_RG_LENGTHS(RG_DECL)
#undef RG_DECL

static const RgTable* rg_table(int n) {
    switch (n) {
#define RG_CASE(n) case n: return rg_table_##n();
        LES_RG_LENGTHS(RG_CASE)
#undef RG_CASE
        default: return nullptr;
    }
}

// the unpadded length of a line op, or 0 when the two lengths are not its pair
static int rg_length(const Twiddle& tin, const Twiddle& tout, LineOp op) {
    const int a = tin.n, b = tout.n;
    switch (op) {
        case OP_PAD: return (2 * b == 3 * a) ? a : 0;
        case OP_UNPAD: return (2 * a == 3 * b) ? b : 0;
        default: return (a == b) ? a : 0;
    }
}

template <typename T, typename TI>
static const RgIo<T, TI>& rg_io(const RgTable* t) {
    if constexpr (sizeof(T) == 8) return t->dd;
    else if constexpr (sizeof(TI) == 8) return t->fd;
    else return t->ff;
}
template <typename T>
static const RgOps<T>& rg_ops(const RgTable* t) {
    if constexpr (sizeof(T) == 8) return t->d;
    else return t->f;
}

// the y-kernels read column pairs as one aligned vector: even column count,
// row stride and plane stride
template <typename TI, typename T>
static bool pairs_aligned(const TI* in, const T* out, int ncols, int ld_in, int ld_out, long ps_in, long ps_out) {
    return ncols % 2 == 0 && ld_in % 2 == 0 && ld_out % 2 == 0 && ps_in % 2 == 0 && ps_out % 2 == 0 &&
           (uintptr_t)in % (2 * sizeof(TI)) == 0 && (uintptr_t)out % (2 * sizeof(T)) == 0;
}

template <typename T, typename TI>
bool xline_real_ct(hipStream_t s, const Batch<T, TI>& io, long nrows, int ld_in, int ld_out, const Twiddle& tin,
                   const Twiddle& tout, LineOp op, double kfac) {
    const RgTable* t = rg_table(rg_length(tin, tout, op));
    return t && rg_io<T, TI>(t).x(s, op, io, nrows, ld_in, ld_out, tin, tout, kfac);
}
template <typename T, typename TI>
bool yline_real_ct(hipStream_t s, const Batch<T, TI>& io, int nplanes, int ncols, int ld_in, int ld_out, long ps_in,
                   long ps_out, const Twiddle& tin, const Twiddle& tout, LineOp op, double kfac) {
    for (int f = 0; f < io.nf; ++f)
        if (!pairs_aligned(io.in[f], io.out[f], ncols, ld_in, ld_out, ps_in, ps_out)) return false;
    const RgTable* t = rg_table(rg_length(tin, tout, op));
    return t && rg_io<T, TI>(t).y(s, op, io, nplanes, ncols, ld_in, ld_out, ps_in, ps_out, tin, tout, kfac);
}
template <typename T, typename TI>
bool x_r2c_ct(hipStream_t s, const Batch<cx<T>, TI>& io, long nrows, int ld_in, int ldc, const Twiddle& tw,
              double scale, int kst) {
    const RgTable* t = rg_table(tw.n);
    if (!t) return false;
    rg_io<T, TI>(t).r2c(s, io, nrows, ld_in, ldc, tw, scale, kst);
    return true;
}
template <typename T>
bool x_c2r_ct(hipStream_t s, const cx<T>* in, T* out, long nrows, int ldc, int ld_out, const Twiddle& tw, int deriv,
              double kfac, int kst) {
    const RgTable* t = rg_table(tw.n);
    if (!t) return false;
    rg_ops<T>(t).c2r(s, in, out, nrows, ldc, ld_out, tw, deriv, kfac, kst);
    return true;
}
template <typename T>
bool yline_spec_ct(hipStream_t s, const Batch<cx<T>, cx<T>>& io, int nplanes, int ncols, long ps, const Twiddle& tw,
                   SpecOp op, const double* G, int ld, int ldG, int mc) {
    const RgTable* t = rg_table(tw.n);
    if (!t) return false;
    rg_ops<T>(t).spec(s, op, io, nplanes, ncols, ps, tw, G, ld, ldG, mc);
    return true;
}

bool press_x_available(const Twiddle& tw) { return g_use_ct && rg_table(tw.n) != nullptr; }
template <typename W>
void press_x(hipStream_t s, const PressIn<W>& a, bool filter, const Twiddle& tw) {
    // u, v, w read, three half spectra written, and with filter u, v, w written
    FamScope fs(s, FAM_XR2C,
                3.0 * (a.nz - 1) * a.ny * (8.0 * tw.n * (filter ? 2.0 : 1.0) + sizeof(W) * (tw.n + 2.0)));
    rg_ops<W>(rg_table(tw.n)).press(s, a, filter, tw);
}
template void press_x<double>(hipStream_t, const PressIn<double>&, bool, const Twiddle&);
template void press_x<float>(hipStream_t, const PressIn<float>&, bool, const Twiddle&);

template <typename T>
bool cross_unpad_x(hipStream_t s, const ConvIn<T>& a, int scalar, T* o0, T* o1, T* o2, int nz, int ny2,
                   const Twiddle& tin, const Twiddle& tout) {
    const RgTable* t = rg_table(rg_length(tin, tout, OP_UNPAD));
    if (!t || ny2 % 2 != 0) return false;
    // six padded inputs (levels 1..nz) read, one or three x-unpadded outputs
    // (levels 1..nz-1) written
    FamScope fs(s, scalar ? FAM_SCALAR_UNPAD_X : FAM_CROSS_UNPAD_X,
                sizeof(T) * (6.0 * nz * tin.n * ny2 + (scalar ? 1.0 : 3.0) * (nz - 1) * ny2 * (double)tout.n));
    rg_ops<T>(t).cross(s, a, scalar, o0, o1, o2, nz, ny2, tin, tout);
    return true;
}
template <typename T>
bool vort_pad_x(hipStream_t s, const VortIn<T>& g, T* o0, T* o1, T* o2, int nz, int ny, const Twiddle& tin,
                const Twiddle& tout) {
    const RgTable* t = rg_table(rg_length(tin, tout, OP_PAD));
    if (!t || ny % 2 != 0) return false;
    // six velocity gradients read, three x-padded vorticity components written
    FamScope fs(s, FAM_VORT_PAD_X, sizeof(T) * (6.0 * nz * tin.n * ny + 3.0 * nz * ny * (double)tout.n));
    rg_ops<T>(t).vort(s, g, o0, o1, o2, nz, ny, tin, tout);
    return true;
}
bool lag_contract_available(const Twiddle& tw) {
    const RgTable* t = rg_table(tw.n);
    return t && rg_ops<double>(t).lag && rg_ops<float>(t).lag;
}
template <typename T>
bool lag_contract_x(hipStream_t s, int scale, const cx<T>* spt, int ldc, int kst, int nz, int ny, double* lm,
                    double* mm, const LagUpdate& u, double cst, const Twiddle& tw) {
    const RgTable* t = rg_table(tw.n);
    if (!t || !rg_ops<T>(t).lag) return false;
    // the 21 filtered spectra read; L M, M M (2 delta) or the F_* update and
    // Cs_opt2 (4 delta) written, FP64
    FamScope fs(s, FAM_LAG_CONTRACT_X,
                21.0 * nz * ny * ldc * 2.0 * sizeof(T) + (scale == 2 ? 2.0 : 7.0) * nz * ny * (double)tw.n * 8.0);
    rg_ops<T>(t).lag(s, scale, spt, ldc, kst, nz, ny, lm, mm, u, cst, tw);
    return true;
}
template bool lag_contract_x<double>(hipStream_t, int, const cx<double>*, int, int, int, int, double*, double*,
                                     const LagUpdate&, double, const Twiddle&);
template bool lag_contract_x<float>(hipStream_t, int, const cx<float>*, int, int, int, int, double*, double*,
                                    const LagUpdate&, double, const Twiddle&);
template bool cross_unpad_x<double>(hipStream_t, const ConvIn<double>&, int, double*, double*, double*, int, int,
                                    const Twiddle&, const Twiddle&);
template bool cross_unpad_x<float>(hipStream_t, const ConvIn<float>&, int, float*, float*, float*, int, int,
                                   const Twiddle&, const Twiddle&);
template bool vort_pad_x<double>(hipStream_t, const VortIn<double>&, double*, double*, double*, int, int,
                                 const Twiddle&, const Twiddle&);
template bool vort_pad_x<float>(hipStream_t, const VortIn<float>&, float*, float*, float*, int, int, const Twiddle&,
                                const Twiddle&);

#define INST_IO(T, TI)                                                                                       \
    template bool xline_real_ct<T, TI>(hipStream_t, const Batch<T, TI>&, long, int, int, const Twiddle&, const Twiddle&, \
                                       LineOp, double);                                                          \
    template bool yline_real_ct<T, TI>(hipStream_t, const Batch<T, TI>&, int, int, int, int, long, long, const Twiddle&, \
                                       const Twiddle&, LineOp, double);                                          \
    template bool x_r2c_ct<T, TI>(hipStream_t, const Batch<cx<T>, TI>&, long, int, int, const Twiddle&, double, int);
INST_IO(double, double)
INST_IO(float, float)
INST_IO(float, double)
#undef INST_IO
template bool x_c2r_ct<double>(hipStream_t, const cx<double>*, double*, long, int, int, const Twiddle&, int, double,
                               int);
template bool x_c2r_ct<float>(hipStream_t, const cx<float>*, float*, long, int, int, const Twiddle&, int, double,
                              int);
template bool yline_spec_ct<double>(hipStream_t, const Batch<cx<double>, cx<double>>&, int, int, long, const Twiddle&,
                                    SpecOp, const double*, int, int, int);
template bool yline_spec_ct<float>(hipStream_t, const Batch<cx<float>, cx<float>>&, int, int, long, const Twiddle&,
                                   SpecOp, const double*, int, int, int);

}  // namespace les
