// Column launches of the four-step: its first launch and the column kernel's
// other modes.
#include "cols_impl.h"

namespace mufft {

// Four-step first half (FourStepArgs): the column transforms above plus the
// w_N^(dir*n2*k1) twiddle, stored transposed: each column of the tile leaves
// as one contiguous run of N1 points.  The input is read with lanes along the
// columns (row segments of TX points); from the last exchange on the threads
// are renumbered with lanes along the points of a column, so the transposed
// store is coalesced without a trip of its own through LDS.
// TXP: tile width (columns per workgroup); 0 = fs_TX(L).
template <int L_, int DIR, int TXP = 0>
__global__ void __launch_bounds__(L_ / fs_E(L_) * (TXP ? TXP : fs_TX(L_)),
                                  fs_waves_per_simd(L_, TXP ? TXP : fs_TX(L_))) fft_four_step_cols_kernel(FourStepArgs a) {
    constexpr int E = fs_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = L_ / E;
    constexpr int TX = TXP ? TXP : fs_TX(L_);
    constexpr int XM = fs_xm(L_, TX);
    constexpr int LP = fs_pitch(L_, TX);
    constexpr int ROWS = L_ + L_ / E;
    constexpr int SMEM = XM == XM_SPLIT ? (LP * TX + 1) / 2 : LP * TX;
    static_assert(LP >= ROWS, "a padded column fits its pitch");
    __shared__ float2 smem[SMEM];
    __shared__ float2 steps[E * TX];

    const int tid = threadIdx.x;
    const int x = tid & (TX - 1);
    const int t = tid / TX;
    const int t1 = tid & (T - 1);   // numbering of the last pass and the store
    const int x1 = tid / T;
    const unsigned bid = xcd_block(blockIdx.x, gridDim.x);
    const int img = (int)(bid / (unsigned)a.ntiles);
    const int tile = (int)(bid % (unsigned)a.ntiles);
    const int col = tile * TX + x;   // n2; the host launches whole tiles only
    const int col1 = tile * TX + x1;
    const bool zp = (a.flags & RF_ZERO_PAD) != 0;

    float2 v[E];
    {
        // A transform spans at most 2^26 points (512 MiB): 32-bit offsets,
        // one per lane, the row offset of each point in a scalar register.
        const __amdgpu_buffer_rsrc_t rin = make_rsrc(a.in + (long long)img * a.in_bs, (unsigned)a.n2 * (unsigned)L_ * 8u);
        const unsigned vo = ((unsigned)t * (unsigned)a.n2 + (unsigned)col) * 8u;
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            const unsigned so = (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(T * c) * (unsigned)a.n2 * 8u));
            if constexpr (TX >= 16) v[c] = (zp && c >= E / 2) ? make_float2(0.f, 0.f) : bload_nt(rin, vo, so);
            else v[c] = (zp && c >= E / 2) ? make_float2(0.f, 0.f) : bload(rin, vo, so);
        });
    }

    // The twiddle of point (n2, k1) = (col1, t1 + T*c) is w^(col1*t1) *
    // w^(col1*T*c): a factor per thread and E steps per column, the steps of
    // the tile's columns in LDS, one coarse*fine product each (every product
    // is within about 1.5 ulp; a point's twiddle within about 3.5).  Two table
    // gathers per point instead cost 10-16% of the whole transform.
    const int smask = (1 << a.log2s) - 1;
    for (int i = tid; i < E * TX; i += T * TX) {   // step i / TX of column i % TX
        const unsigned es = (unsigned)(tile * TX + (i & (TX - 1))) * (unsigned)(T * (i / TX));   // < N
        steps[i] = cmul(a.coarse[es >> a.log2s], a.fine[es & smask]);
    }
    const unsigned e0 = (unsigned)col1 * (unsigned)t1;
    const float2 w0 = cmul(a.coarse[e0 >> a.log2s], a.fine[e0 & smask]);

    // The passes' exchanges synchronise the workgroup: the steps are
    // visible to every thread after them.  Column-major LDS with a pitch that
    // spreads both numberings over the banks (fs_pitch).
    auto slot = [x](int o) { return x * LP + pad_slot<LOGE>(o); };
    auto slot1 = [x1](int o) { return x1 * LP + pad_slot<LOGE>(o); };
    stockham_passes_renumbered<L_, E, DIR, XM, fs_twm(L_), E, false, false>(
        v, t, TwGlobal{a.tw}, smem, reinterpret_cast<float *>(smem), slot, t, t1, slot, slot1);

    float2 *dst = a.out + (long long)img * a.out_bs + (long long)col1 * L_ + t1;
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        dst[T * c] = cmul(v[c], cmul(w0, steps[c * TX + x1]));
    });
}

template <int DIR>
static const void *four_step_kernel_ptr(int logL, bool narrow) {
    switch (logL) {
    case 6: return (const void *)&fft_four_step_cols_kernel<64, DIR>;
    case 7: return (const void *)&fft_four_step_cols_kernel<128, DIR>;
#define MUFFT_FS_CASE(l)                                                                             \
    case l:                                                                                          \
        return narrow ? (const void *)&fft_four_step_cols_kernel<(1 << l), DIR, narrow_TX(1 << l, fs_TX(1 << l))> \
                      : (const void *)&fft_four_step_cols_kernel<(1 << l), DIR>
    MUFFT_FS_CASE(8);
    MUFFT_FS_CASE(9);
    MUFFT_FS_CASE(10);
    MUFFT_FS_CASE(11);
    MUFFT_FS_CASE(12);
#undef MUFFT_FS_CASE
    case 13: return (const void *)&fft_four_step_cols_kernel<8192, DIR>;
    default: return nullptr;
    }
}

hipError_t launch_four_step_cols(int logN1, int direction, const FourStepArgs &a, hipStream_t s) {
    const int L = 1 << logN1;
    const bool narrow = use_narrow(L, fs_TX(L), a.n2, a.batch);
    const void *k = direction < 0 ? four_step_kernel_ptr<-1>(logN1, narrow) : four_step_kernel_ptr<1>(logN1, narrow);
    if (!k) return hipErrorInvalidValue;
    const int tx = narrow ? narrow_TX(L, fs_TX(L)) : fs_TX(L);
    if (a.n2 % tx != 0) return hipErrorInvalidValue;
    FourStepArgs args = a;
    args.ntiles = a.n2 / tx;
    const long long nblocks = (long long)args.ntiles * a.batch;
    if (nblocks <= 0) return hipSuccess;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidValue;
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3((unsigned)nblocks), dim3(L / fs_E(L) * tx), params, 0, s);
}

template <int DIR, int MODE>
static const void *col_mode_kernel_ptr(int logL, bool narrow) {
    switch (logL) {
    case 6: return (const void *)&fft_cols_kernel<64, DIR, MODE>;
    case 7: return (const void *)&fft_cols_kernel<128, DIR, MODE>;
#define MUFFT_COL_CASE(l)                                                                            \
    case l:                                                                                          \
        return narrow ? (const void *)&fft_cols_kernel<(1 << l), DIR, MODE, narrow_TX(1 << l, col_TX(1 << l))> \
                      : (const void *)&fft_cols_kernel<(1 << l), DIR, MODE>
    MUFFT_COL_CASE(8);
    MUFFT_COL_CASE(9);
    MUFFT_COL_CASE(10);
#undef MUFFT_COL_CASE
    default: return nullptr;
    }
}

const void *col_mode_kernel(int logL, int direction, int mode, bool narrow) {
    const bool f = direction < 0;
    switch (mode) {
    case COL_TWIDDLE:
        return f ? col_mode_kernel_ptr<-1, COL_TWIDDLE>(logL, narrow) : col_mode_kernel_ptr<1, COL_TWIDDLE>(logL, narrow);
    case COL_TWO_LEVEL:
        return f ? col_mode_kernel_ptr<-1, COL_TWO_LEVEL>(logL, narrow)
                 : col_mode_kernel_ptr<1, COL_TWO_LEVEL>(logL, narrow);
    case COL_STREAM:
        return f ? col_mode_kernel_ptr<-1, COL_STREAM>(logL, narrow) : col_mode_kernel_ptr<1, COL_STREAM>(logL, narrow);
    default: return nullptr;
    }
}

}  // namespace mufft
