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
#pragma once

#include "kernels.h"
#include "stockham.h"

namespace mufft {

// TXP: tile width (columns per workgroup); 0 = the default col_TX(L).
template <int L_, int DIR, int MODE = COL_PLAIN, int TXP = 0>
__global__ void __launch_bounds__(col_T(L_) * (TXP ? TXP : col_TX(L_)), col_waves_per_simd(L_, TXP ? TXP : col_TX(L_))) fft_cols_kernel(ColArgs a) {
    constexpr int E = col_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = col_T(L_);
    constexpr int TX = TXP ? TXP : col_TX(L_);
    constexpr int ROWS = L_ + L_ / E;
    constexpr int XM = col_xm(L_, TX);
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
    // Streaming only where a tile's row segments are whole 128-byte lines.  The
    // last of three launches streams too: c2c 2^24 x 2 303 -> 281 us, 2^23 x 8
    // 630 -> 600, 2^26 663 -> 642; the middle one in place does not (2^24 x 2
    // 282 -> 318).
    constexpr bool NT = (MODE == COL_STREAM || MODE == COL_TWO_LEVEL) && TX >= 16;
    float2 v[E];
    const unsigned vin = ((unsigned)t * (unsigned)a.in_rs + (unsigned)colr) * 8u;
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if constexpr (ROW_ADDR) v[c] = gload<NT>(a.in + ib + (long long)(T * c) * a.in_rs, vin);
        // (Long columns: with the clamped column, 2D c2c 4096^2 x 2 takes 310 us.)
        else if constexpr (L_ >= 4096) v[c] = active ? (a.in + ib + col)[(long long)(t + T * c) * a.in_rs] : make_float2(0.f, 0.f);
        else v[c] = (a.in + ib + colr)[(long long)(t + T * c) * a.in_rs];
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
            if constexpr (ROW_ADDR) gstore<NT>(a.out + ob + (long long)(T * c) * a.out_rs, vout, v[c]);
            else (a.out + ob + col)[(long long)(t + T * c) * a.out_rs] = v[c];
        });
    }
}

// The kernel of a mode other than COL_PLAIN, 64 to 1024 points (four_step.hip);
// narrow: tiles of narrow_TX columns.
const void *col_mode_kernel(int logL, int direction, int mode, bool narrow);

}  // namespace mufft
