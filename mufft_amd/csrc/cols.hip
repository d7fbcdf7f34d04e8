// Fused column (strided-axis) transforms: the 2D vertical passes.
//
// The reference runs each vertical radix pass as a separate sweep over the
// whole image (kernel.c:455-738, driven by fft.c:978-987).  Here one
// workgroup owns a tile of TX adjacent columns and runs every pass of the
// column transforms in registers/LDS: one HBM read and one HBM write per
// point, lanes along the unit-stride axis so each row segment of the tile is
// a single coalesced access.  Tiles are assigned XCD-aware so neighbouring
// tiles, which share cache lines, run under the same L2.  In place is safe:
// a workgroup reads its whole tile before it writes any of it.
#include "kernels.h"
#include "stockham.h"

namespace mufft {

// TXP: tile width (columns per workgroup); 0 = the default col_TX(L).
template <int L_, int DIR, int MODE = COL_PLAIN, int TXP = 0>
__global__ void __launch_bounds__(col_T(L_) * (TXP ? TXP : col_TX(L_)), col_waves_per_simd(L_)) fft_cols_kernel(ColArgs a) {
    constexpr int E = col_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = col_T(L_);
    constexpr int TX = TXP ? TXP : col_TX(L_);
    constexpr int ROWS = L_ + L_ / E;
    constexpr int XM = col_xm(L_);
    constexpr bool LDS = np_for(L_, E) > 1;
    __shared__ float2 smem[!LDS ? 1 : XM == XM_SPLIT ? (ROWS * TX + 1) / 2 : ROWS * TX];

    const int tid = threadIdx.x;
    const int x = tid & (TX - 1);
    const int t = tid / TX;
    // The partial tiles of all images come first (r2c and c2r images have one
    // column more than a multiple of TX): they move little and end early.  Last
    // in the grid they ran alone after the full tiles, whose number often just
    // fills the GPU (2D r2c 2048^2 x 4: 512 full and 4 partial tiles on 512
    // places).
    const bool partial = a.ncols % TX != 0;
    const unsigned nfirst = partial ? (unsigned)a.batch : 0u;
    int img, tile;
    if (blockIdx.x < nfirst) {
        img = (int)blockIdx.x;
        tile = a.ntiles - 1;
    } else {
        const unsigned full = (unsigned)a.ntiles - (partial ? 1u : 0u);
        const unsigned bid = xcd_block(blockIdx.x - nfirst, gridDim.x - nfirst);
        img = __builtin_amdgcn_readfirstlane((int)(bid / full));
        tile = __builtin_amdgcn_readfirstlane((int)(bid % full));
    }
    const int col = tile * TX + x;
    // Lanes past the last column read it again and store nothing.
    const bool active = col < a.ncols;
    const int colr = active ? col : a.ncols - 1;
    auto slot = [x](int o) { return pad_slot<LOGE>(o) * TX + x; };

    long long ib = (long long)img * a.in_bs, ob = (long long)img * a.out_bs;
    if constexpr (MODE == COL_TWO_LEVEL) {
        ib = (long long)(img / a.img_div) * a.in_bs2 + (long long)(img % a.img_div) * a.in_bs;
        ob = (long long)(img / a.img_div) * a.out_bs2 + (long long)(img % a.img_div) * a.out_bs;
    }

    // Row t + T*c of this lane's column.  ROW_ADDR: a scalar row address per c
    // plus one 32-bit offset per lane (T is at most 32 there and a row at most
    // 2^21 points, so the offset stays below 4 GiB); else a 64-bit address per
    // lane.  The first takes fewer registers, which the 1024-point kernel
    // needs (with 64-bit addresses it spills: 2D c2c 1024^2 x 16 88 -> 104
    // us) and streams better; the long 2D columns run better with the second,
    // which spaces the loads out (2D c2c 4096^2 x 2 244 -> 222 us, c2r
    // 512^2 x 32 44.5 -> 41.2 us).
    constexpr bool ROW_ADDR = MODE != COL_PLAIN || L_ == 1024;
    float2 v[E];
    const unsigned vin = ((unsigned)t * (unsigned)a.in_rs + (unsigned)colr) * 8u;
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if constexpr (ROW_ADDR) v[c] = gload<MODE == COL_STREAM>(a.in + ib + (long long)(T * c) * a.in_rs, vin);
        else v[c] = active ? (a.in + ib + col)[(long long)(t + T * c) * a.in_rs] : make_float2(0.f, 0.f);
    });

    // COL_TWIDDLE: the twiddle of point t + T*c of a column with factor b is
    // w^(b*t) * w^(b*T*c), a factor per thread and E steps per column in LDS
    // (as in the four-step column kernel below), where a workgroup has a
    // thread per step.
    constexpr bool STEPS = MODE == COL_TWIDDLE && E <= T;
    __shared__ float2 steps[STEPS ? E * TX : 1];
    float2 w0 = make_float2(1.f, 0.f);
    if constexpr (STEPS) {
        const unsigned smask = (1u << a.log2s) - 1u;
        if (tid < E * TX) {   // step tid / TX of this thread's own column (tid % TX == x)
            const unsigned es = ((unsigned)col >> a.log2div) * (unsigned)(T * (tid / TX));
            steps[tid] = col < a.ncols ? cmul(a.coarse[es >> a.log2s], a.fine[es & smask]) : make_float2(1.f, 0.f);
        }
        if (active) {
            const unsigned e0 = ((unsigned)col >> a.log2div) * (unsigned)t;
            w0 = cmul(a.coarse[e0 >> a.log2s], a.fine[e0 & smask]);
        }
    }

    // Remainder pass last (seq_radix): the lanes of one column thread share its
    // twiddles.  Its exchanges synchronise the workgroup (the steps are visible
    // after them).
    stockham_passes<L_, E, DIR, XM, col_twm(L_), E, false, false>(v, t, TwGlobal{a.tw}, smem,
                                                                  reinterpret_cast<float *>(smem), slot);

    if (active) {
        if constexpr (STEPS) {
            static_for<0, E>([&](auto C) {
                constexpr int c = decltype(C)::value;
                v[c] = cmul(v[c], cmul(w0, steps[c * TX + x]));
            });
        } else if constexpr (MODE == COL_TWIDDLE) {
            const unsigned b = (unsigned)col >> a.log2div;
            const unsigned smask = (1u << a.log2s) - 1u;
            static_for<0, E>([&](auto C) {
                constexpr int c = decltype(C)::value;
                const unsigned e = b * (unsigned)(t + T * c);
                v[c] = cmul(v[c], cmul(a.coarse[e >> a.log2s], a.fine[e & smask]));
            });
        }
        const unsigned vout = ((unsigned)t * (unsigned)a.out_rs + (unsigned)col) * 8u;
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            if constexpr (ROW_ADDR) gstore<MODE == COL_STREAM>(a.out + ob + (long long)(T * c) * a.out_rs, vout, v[c]);
            else (a.out + ob + col)[(long long)(t + T * c) * a.out_rs] = v[c];
        });
    }
}

// Four-step first half (FourStepArgs): the column transforms above plus the
// w_N^(dir*n2*k1) twiddle, stored transposed: each column of the tile leaves
// as one contiguous run of N1 points.  The input is read with lanes along the
// columns (row segments of TX points); from the last exchange on the threads
// are renumbered with lanes along the points of a column, so the transposed
// store is coalesced without a trip of its own through LDS.
template <int L_, int DIR>
__global__ void __launch_bounds__(fs_WG(L_), fs_waves_per_simd(L_)) fft_four_step_cols_kernel(FourStepArgs a) {
    constexpr int E = fs_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = L_ / E;
    constexpr int TX = fs_TX(L_);
    constexpr int XM = fs_xm(L_);
    constexpr int LP = fs_pitch(L_);
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
    for (int i = tid; i < E * TX; i += fs_WG(L_)) {   // step i / TX of column i % TX
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
static const void *four_step_kernel_ptr(int logL) {
    switch (logL) {
    case 6: return (const void *)&fft_four_step_cols_kernel<64, DIR>;
    case 7: return (const void *)&fft_four_step_cols_kernel<128, DIR>;
    case 8: return (const void *)&fft_four_step_cols_kernel<256, DIR>;
    case 9: return (const void *)&fft_four_step_cols_kernel<512, DIR>;
    case 10: return (const void *)&fft_four_step_cols_kernel<1024, DIR>;
    case 11: return (const void *)&fft_four_step_cols_kernel<2048, DIR>;
    case 12: return (const void *)&fft_four_step_cols_kernel<4096, DIR>;
    case 13: return (const void *)&fft_four_step_cols_kernel<8192, DIR>;
    default: return nullptr;
    }
}

hipError_t launch_four_step_cols(int logN1, int direction, const FourStepArgs &a, hipStream_t s) {
    const void *k = direction < 0 ? four_step_kernel_ptr<-1>(logN1) : four_step_kernel_ptr<1>(logN1);
    if (!k) return hipErrorInvalidValue;
    const int L = 1 << logN1;
    if (a.n2 % fs_TX(L) != 0 || a.ntiles != a.n2 / fs_TX(L)) return hipErrorInvalidValue;
    const long long nblocks = (long long)a.ntiles * a.batch;
    if (nblocks <= 0) return hipSuccess;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidValue;
    FourStepArgs args = a;
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3((unsigned)nblocks), dim3(fs_WG(L)), params, 0, s);
}

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

// The middle and last passes of the three-pass transform: columns of 64 to
// 1024 points.
template <int DIR, int MODE>
static const void *col_mode_kernel_ptr(int logL) {
    switch (logL) {
    case 6: return (const void *)&fft_cols_kernel<64, DIR, MODE>;
    case 7: return (const void *)&fft_cols_kernel<128, DIR, MODE>;
    case 8: return (const void *)&fft_cols_kernel<256, DIR, MODE>;
    case 9: return (const void *)&fft_cols_kernel<512, DIR, MODE>;
    case 10: return (const void *)&fft_cols_kernel<1024, DIR, MODE>;
    default: return nullptr;
    }
}

hipError_t launch_cols(int logL, int direction, const ColArgs &a, hipStream_t s, int mode, int tx) {
    const void *k = nullptr;
    const int L = 1 << logL;
    if (tx == 0) tx = col_TX(L);
    if (tx != col_TX(L) && (mode != COL_PLAIN || logL < 1 || logL > COL_MAX_LOG2 || !col_TX_valid(L, tx)))
        return hipErrorInvalidValue;
    if (a.ntiles <= 0 || (long long)a.ntiles * tx < a.ncols) return hipErrorInvalidValue;
    if (mode == COL_PLAIN && tx != col_TX(L))
        k = direction < 0 ? col_alt_kernel_ptr<-1>(logL, tx) : col_alt_kernel_ptr<1>(logL, tx);
    else if (mode == COL_PLAIN) k = direction < 0 ? col_kernel_ptr<-1>(logL) : col_kernel_ptr<1>(logL);
    else if (mode == COL_TWIDDLE)
        k = direction < 0 ? col_mode_kernel_ptr<-1, COL_TWIDDLE>(logL) : col_mode_kernel_ptr<1, COL_TWIDDLE>(logL);
    else if (mode == COL_TWO_LEVEL)
        k = direction < 0 ? col_mode_kernel_ptr<-1, COL_TWO_LEVEL>(logL) : col_mode_kernel_ptr<1, COL_TWO_LEVEL>(logL);
    else if (mode == COL_STREAM)
        k = direction < 0 ? col_mode_kernel_ptr<-1, COL_STREAM>(logL) : col_mode_kernel_ptr<1, COL_STREAM>(logL);
    if (!k) return hipErrorInvalidValue;
    if (mode == COL_TWIDDLE && (!a.coarse || !a.fine)) return hipErrorInvalidValue;
    if (mode == COL_TWO_LEVEL && a.img_div <= 0) return hipErrorInvalidValue;
    const long long nblocks = (long long)a.ntiles * a.batch;
    if (nblocks <= 0) return hipSuccess;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidValue;
    ColArgs args = a;
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3((unsigned)nblocks), dim3(col_T(L) * tx), params, 0, s);
}

}  // namespace mufft
