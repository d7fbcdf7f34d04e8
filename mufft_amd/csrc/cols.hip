// Column transforms of images: instantiations of the column kernel in plain
// mode and the launcher of every mode.
#include "cols_impl.h"

namespace mufft {

// The alternative tile widths of a column length (col_TX_alt), plain mode.
template <int L_, int DIR>
static const void *col_alt_kernel(int tx) {
    if (tx == col_TX_alt(L_)) return (const void *)&fft_cols_kernel<L_, DIR, COL_PLAIN, col_TX_alt(L_)>;
    if constexpr (col_TX_alt(L_, 1) != 0)
        if (tx == col_TX_alt(L_, 1)) return (const void *)&fft_cols_kernel<L_, DIR, COL_PLAIN, col_TX_alt(L_, 1)>;
    return nullptr;
}
template <int DIR>
static const void *col_alt_kernel_ptr(int logL, int tx) {
    switch (logL) {
    case 7: return col_alt_kernel<128, DIR>(tx);
    case 8: return col_alt_kernel<256, DIR>(tx);
    case 9: return col_alt_kernel<512, DIR>(tx);
    case 10: return col_alt_kernel<1024, DIR>(tx);
    case 11: return col_alt_kernel<2048, DIR>(tx);
    case 12: return col_alt_kernel<4096, DIR>(tx);
    case 13: return col_alt_kernel<8192, DIR>(tx);
    default: return nullptr;
    }
}

template <int DIR>
static const void *col_kernel_ptr(int logL) {
    switch (logL) {
    case 1: return (const void *)&fft_cols_kernel<2, DIR>;
    case 2: return (const void *)&fft_cols_kernel<4, DIR>;
    case 3: return (const void *)&fft_cols_kernel<8, DIR>;
    case 4: return (const void *)&fft_cols_kernel<16, DIR>;
    case 5: return (const void *)&fft_cols_kernel<32, DIR>;
    case 6: return (const void *)&fft_cols_kernel<64, DIR>;
    case 7: return (const void *)&fft_cols_kernel<128, DIR>;
    case 8: return (const void *)&fft_cols_kernel<256, DIR>;
    case 9: return (const void *)&fft_cols_kernel<512, DIR>;
    case 10: return (const void *)&fft_cols_kernel<1024, DIR>;
    case 11: return (const void *)&fft_cols_kernel<2048, DIR>;
    case 12: return (const void *)&fft_cols_kernel<4096, DIR>;
    case 13: return (const void *)&fft_cols_kernel<8192, DIR>;
    default: return nullptr;
    }
}

hipError_t launch_cols(int logL, int direction, const ColArgs &a, hipStream_t s, int mode, int tx) {
    const void *k = nullptr;
    const int L = 1 << logL;
    ColArgs args = a;
    if (mode == COL_PLAIN) {
        if (tx == 0) tx = col_TX(L);
        if (tx != col_TX(L) && (logL < 1 || logL > COL_MAX_LOG2 || !col_TX_valid(L, tx))) return hipErrorInvalidValue;
        if (tx != col_TX(L)) k = direction < 0 ? col_alt_kernel_ptr<-1>(logL, tx) : col_alt_kernel_ptr<1>(logL, tx);
        else k = direction < 0 ? col_kernel_ptr<-1>(logL) : col_kernel_ptr<1>(logL);
    } else {
        if (tx != 0) return hipErrorInvalidValue;
        tx = col_TX(L);
        const bool narrow = use_narrow(L, tx, a.ncols, a.batch);
        k = col_mode_kernel(logL, direction, mode, narrow);
        if (narrow) tx = narrow_TX(L, tx);
    }
    if (!k || a.ncols <= 0) return hipErrorInvalidValue;
    if (mode == COL_TWIDDLE && (!a.coarse || !a.fine)) return hipErrorInvalidValue;
    if (mode == COL_TWO_LEVEL && a.img_div <= 0) return hipErrorInvalidValue;
    args.ntiles = (a.ncols + tx - 1) / tx;
    const long long nblocks = (long long)args.ntiles * a.batch;
    if (nblocks <= 0) return hipSuccess;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidValue;
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3((unsigned)nblocks), dim3(col_T(L) * tx), params, 0, s);
}

}  // namespace mufft
