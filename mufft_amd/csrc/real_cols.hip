// Column launches of the large real transforms with the resolve pass fused in.
//
// A real transform of 2n points is an n-point complex one plus the resolve
// (kernel.c:36-82), which pairs bin k with bin n - k.  Seen as columns of
// length L at stride M (k = j + M*k2, n = M*L), the partner of row k2 of
// column j is row L-1-k2 of column M-j.  Each thread here runs its point of
// column j and of column M-j, the second under the mirrored thread numbering
// T-1-t: the partners of its points t + T*c of the first column are then its
// own points (T-1-t) + T*(E-1-c) of the second, so the resolve needs neither
// an exchange nor a pass over memory of its own.  r2c resolves after the last
// column launch, c2r before the first.
//
// Columns 0 and M/2 are their own partners; they run in a small launch of
// their own (a workgroup each), which keeps the edge cases (bins 0 and
// n, rows k2 and L-k2 in different threads) out of the main kernels.
#include "kernels.h"
#include "stockham.h"

namespace mufft {

// Column j of a real transform's column launch: j >> log_cols selects the
// image, the rest the column in it.
__device__ __forceinline__ unsigned real_col_offset(unsigned j, int log_cols, unsigned image_stride) {
    return (j >> log_cols) * image_stride + (j & ((1u << log_cols) - 1u));
}

// X[k] and X[n-k] from za = Z[k], zb = Z[n-k], w = W[k] (kernel.c:47-82).
__device__ __forceinline__ void resolve_pair(float2 za, float2 zb, float2 w, float2 &xk, float2 &xnk) {
    const float2 bc = cconj(zb);
    const float2 fe = cadd(za, bc);
    const float2 fo = cmul(w, csub(za, bc));
    xk = cscale(cadd(fe, fo), 0.5f);
    xnk = cscale(cconj(csub(fe, fo)), 0.5f);
}

// Last launch of a forward real transform: columns j in [1, M/2) with their
// partners M - j.  The tile is what two column sets of 32 points per thread
// leave room for: 128 registers of points, one 512-thread workgroup per CU.
template <int L_, int TX>
__global__ void __launch_bounds__(L_ / fs_E(L_) * TX, rc_waves_per_simd(L_)) fft_cols_r2c_kernel(RealColArgs a) {
    constexpr int E = col_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = col_T(L_);
    constexpr int XM = rc_xm(L_, TX);
    constexpr int ROWS = L_ + L_ / E;
    __shared__ float2 smem[XM == XM_SPLIT ? (ROWS * TX + 1) / 2 : ROWS * TX];

    const int tid = threadIdx.x;
    const int x = tid & (TX - 1);
    const int t = tid / TX;
    const unsigned bid = xcd_block(blockIdx.x, gridDim.x);
    const int img = __builtin_amdgcn_readfirstlane((int)(bid / (unsigned)a.ntiles));
    const int tile = __builtin_amdgcn_readfirstlane((int)(bid % (unsigned)a.ntiles));
    const unsigned ja = (unsigned)(tile * TX + x);
    const bool active = ja != 0;                           // column 0: fft_cols_r2c_self_kernel
    const unsigned jb = active ? (unsigned)a.m - ja : 0u;
    const int ta = t, tb = T - 1 - t;

    const float2 *src = a.in + (long long)img * a.in_bs;
    const unsigned va = (real_col_offset(ja, a.log_cols, (unsigned)a.image_stride) + (unsigned)ta * (unsigned)a.in_rs) * 8u;
    const unsigned vb = (real_col_offset(jb, a.log_cols, (unsigned)a.image_stride) + (unsigned)tb * (unsigned)a.in_rs) * 8u;
    float2 u[E], v[E];
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        u[c] = gload<false>(src + (long long)(T * c) * a.in_rs, va);
    });
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        v[c] = gload<false>(src + (long long)(T * c) * a.in_rs, vb);
    });
    const float2 wb = a.rtw[(long long)ja + (long long)a.m * t];   // W[k] of point c = 0

    auto slot = [x](int o) { return pad_slot<LOGE>(o) * TX + x; };
    stockham_passes<L_, E, -1, XM, rc_twm(L_), E, false, false>(u, ta, TwGlobal{a.tw}, smem,
                                                                reinterpret_cast<float *>(smem), slot);
    stockham_passes<L_, E, -1, XM, rc_twm(L_), E, false, false>(v, tb, TwGlobal{a.tw}, smem,
                                                                reinterpret_cast<float *>(smem), slot);
    if (active) {
        float2 *dst = a.out + (long long)img * a.out_bs;
        const unsigned oa = (ja + (unsigned)ta * (unsigned)a.m) * 8u;
        const unsigned ob = (jb + (unsigned)tb * (unsigned)a.m) * 8u;
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            float2 xk, xnk;
            // W[k + M*T*c] = W[k] * exp(-i pi c / E)
            resolve_pair(u[c], v[E - 1 - c], twc<c, 2 * E, -1>(wb), xk, xnk);
            gstore<false>(dst + (long long)(T * c) * a.m, oa, xk);
            gstore<false>(dst + (long long)(T * (E - 1 - c)) * a.m, ob, xnk);
        });
    }
}

// Columns 0 and M/2 of the same launch, one workgroup each.  Every row is a
// cache line of its own and little else runs, so the latency of the gathers
// and of the passes is the launch's time: 4 points per thread spread both over
// the most waves (two columns by one wave of 32 points per thread took 33 us
// at 1024 rows).
template <int L_>
__global__ void __launch_bounds__(rcs_T(L_)) fft_cols_r2c_self_kernel(RealColArgs a) {
    constexpr int E = rcs_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = rcs_T(L_);
    __shared__ float2 smem[L_ + L_ / E];
    const int t = threadIdx.x;
    const int img = (int)(blockIdx.x >> 1);
    const bool zero = (blockIdx.x & 1) == 0;
    const unsigned j = zero ? 0u : (unsigned)a.m / 2;
    const float2 *src = a.in + (long long)img * a.in_bs + real_col_offset(j, a.log_cols, (unsigned)a.image_stride);
    float2 v[E], w[E];
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        v[c] = src[(long long)(t + T * c) * a.in_rs];
        w[c] = a.rtw[(long long)j + (long long)a.m * (t + T * c)];
    });
    auto slot = [](int o) { return pad_slot<LOGE>(o); };
    stockham_passes<L_, E, -1, XM_PAD, TW_FULL, E, false, false>(v, t, TwGlobal{a.tw_self}, smem, nullptr, slot);
    static_for<0, E>([&](auto C) { smem[slot(t + T * decltype(C)::value)] = v[decltype(C)::value]; });
    __syncthreads();
    float2 *dst = a.out + (long long)img * a.out_bs;
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        const int k2 = t + T * c;
        const long long k = (long long)j + (long long)a.m * k2;
        if (k == 0) {   // bins 0 and n from Z[0]
            dst[0] = make_float2(v[c].x + v[c].y, 0.f);
            dst[(long long)a.m * L_] = make_float2(v[c].x - v[c].y, 0.f);
        } else {
            float2 xk, xnk;
            resolve_pair(v[c], smem[slot(zero ? L_ - k2 : L_ - 1 - k2)], w[c], xk, xnk);
            dst[k] = xk;
        }
    });
}

// First launch of an inverse real transform: the resolve (kernel.c:36-45) as
// the points are loaded, then the four-step first launch (cols.hip) on columns
// j in [1, N2/2) and N2 - j.
template <int L_, int TX>
__global__ void __launch_bounds__(L_ / fs_E(L_) * TX, rc_waves_per_simd(L_)) fft_four_step_c2r_kernel(RealFourStepArgs a) {
    constexpr int E = fs_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = L_ / E;
    constexpr int XM = rc_xm(L_, TX);
    constexpr int LP = tile_pitch(L_ + L_ / E, TX, XM);
    __shared__ float2 smem[XM == XM_SPLIT ? (LP * TX + 1) / 2 : LP * TX];
    __shared__ float2 steps[2 * E * TX];

    const int tid = threadIdx.x;
    const int x = tid & (TX - 1);
    const int t = tid / TX;
    const int t1 = tid & (T - 1);
    const int x1 = tid / T;
    const unsigned bid = xcd_block(blockIdx.x, gridDim.x);
    const int img = __builtin_amdgcn_readfirstlane((int)(bid / (unsigned)a.ntiles));
    const int tile = __builtin_amdgcn_readfirstlane((int)(bid % (unsigned)a.ntiles));
    const unsigned ja = (unsigned)(tile * TX + x);
    const unsigned jb = ja != 0 ? (unsigned)a.n2 - ja : 0u;
    const int ta = t, tb = T - 1 - t;

    const float2 *src = a.in + (long long)img * a.in_bs;
    const unsigned va = (ja + (unsigned)ta * (unsigned)a.n2) * 8u;
    const unsigned vb = (jb + (unsigned)tb * (unsigned)a.n2) * 8u;
    float2 u[E], v[E];
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        u[c] = gload<false>(src + (long long)(T * c) * a.n2, va);
    });
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        v[c] = gload<false>(src + (long long)(T * c) * a.n2, vb);
    });
    const float2 wb = a.rtw[(long long)ja + (long long)a.n2 * t];

    const int smask = (1 << a.log2s) - 1;
    for (int i = tid; i < 2 * E * TX; i += T * TX) {   // steps of column ja, then of N2 - ja
        const int h = i / (E * TX), r = i % (E * TX);
        const unsigned j0 = (unsigned)(tile * TX + (r & (TX - 1)));
        const unsigned j = h ? (j0 != 0 ? (unsigned)a.n2 - j0 : 0u) : j0;
        const unsigned es = j * (unsigned)(T * (r / TX));   // < n
        steps[i] = cmul(a.coarse[es >> a.log2s], a.fine[es & smask]);
    }
    const unsigned ja1 = (unsigned)(tile * TX + x1);
    const unsigned jb1 = ja1 != 0 ? (unsigned)a.n2 - ja1 : 0u;
    const unsigned e0 = ja1 * (unsigned)t1, e1 = jb1 * (unsigned)t1;
    const float2 wa0 = cmul(a.coarse[e0 >> a.log2s], a.fine[e0 & smask]);
    const float2 wb0 = cmul(a.coarse[e1 >> a.log2s], a.fine[e1 & smask]);

    // Z[k] and Z[n-k] of every pair of points.
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        const float2 xa = u[c], xb = v[E - 1 - c];
        const float2 ac = cconj(xa), bc = cconj(xb);
        const float2 w = twc<c, 2 * E, 1>(wb);
        u[c] = cadd(cadd(xa, bc), cmul(csub(xa, bc), w));
        v[E - 1 - c] = cadd(cadd(xb, ac), cmul(csub(xb, ac), cconj(w)));
    });

    auto slot = [x](int o) { return x * LP + pad_slot<LOGE>(o); };
    auto slot1 = [x1](int o) { return x1 * LP + pad_slot<LOGE>(o); };
    // Stores through a descriptor: an offset beyond it drops those of column 0.
    const __amdgpu_buffer_rsrc_t rout = make_rsrc(a.out + (long long)img * a.out_bs, (unsigned)a.n2 * (unsigned)L_ * 8u);
    const unsigned oa = ja1 != 0 ? (ja1 * (unsigned)L_ + (unsigned)t1) * 8u : 0x80000000u;
    const unsigned ob = ja1 != 0 ? (jb1 * (unsigned)L_ + (unsigned)t1) * 8u : 0x80000000u;
    stockham_passes_renumbered<L_, E, 1, XM, fs_twm(L_), E, false, false>(
        u, ta, TwGlobal{a.tw}, smem, reinterpret_cast<float *>(smem), slot, ta, t1, slot, slot1);
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        bstore(rout, oa, T * c * 8u, cmul(u[c], cmul(wa0, steps[c * TX + x1])));
    });
    // The last pass of both columns reads the same twiddles; t1b hides that, or
    // the compiler keeps the first one's twiddle products, up to 62 registers,
    // for the second.
    int t1b = t1;
    asm volatile("" : "+v"(t1b));
    stockham_passes_renumbered<L_, E, 1, XM, fs_twm(L_), E, false, false>(
        v, tb, TwGlobal{a.tw}, smem, reinterpret_cast<float *>(smem), slot, tb, t1b, slot, slot1);
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        bstore(rout, ob, T * c * 8u, cmul(v[c], cmul(wb0, steps[E * TX + c * TX + x1])));
    });
}

// Columns 0 and N2/2 of the same launch, as fft_cols_r2c_self_kernel; a
// point's partner is read directly.
template <int L_>
__global__ void __launch_bounds__(rcs_T(L_)) fft_four_step_c2r_self_kernel(RealFourStepArgs a) {
    constexpr int E = rcs_E(L_);
    constexpr int LOGE = ilog2(E);
    constexpr int T = rcs_T(L_);
    __shared__ float2 smem[L_ + L_ / E];
    const int t = threadIdx.x;
    const int img = (int)(blockIdx.x >> 1);
    const unsigned j = (blockIdx.x & 1) == 0 ? 0u : (unsigned)a.n2 / 2;
    const int smask = (1 << a.log2s) - 1;
    const float2 *src = a.in + (long long)img * a.in_bs;
    const long long n = (long long)a.n2 * L_;
    float2 v[E], w[E];
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        const long long k = (long long)j + (long long)a.n2 * (t + T * c);
        const float2 xa = src[k], bc = cconj(src[n - k]);
        v[c] = cadd(cadd(xa, bc), cmul(csub(xa, bc), a.rtw[k]));
        const unsigned e = j * (unsigned)(t + T * c);   // < n
        w[c] = cmul(a.coarse[e >> a.log2s], a.fine[e & smask]);
    });
    auto slot = [](int o) { return pad_slot<LOGE>(o); };
    stockham_passes<L_, E, 1, XM_PAD, TW_FULL, E, false, false>(v, t, TwGlobal{a.tw_self}, smem, nullptr, slot);
    float2 *dst = a.out + (long long)img * a.out_bs + (long long)j * L_ + t;
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        dst[T * c] = cmul(v[c], w[c]);
    });
}

namespace {

struct RealKernels {
    const void *pairs, *narrow, *self;
};
template <int L_>
RealKernels r2c_kernels() {
    constexpr int tx = rc_TX(L_), nt = narrow_TX(L_, tx) ? narrow_TX(L_, tx) : tx;
    return {(const void *)&fft_cols_r2c_kernel<L_, tx>, (const void *)&fft_cols_r2c_kernel<L_, nt>,
            (const void *)&fft_cols_r2c_self_kernel<L_>};
}
template <int L_>
RealKernels c2r_kernels() {
    constexpr int tx = rc_TX(L_), nt = narrow_TX(L_, tx) ? narrow_TX(L_, tx) : tx;
    return {(const void *)&fft_four_step_c2r_kernel<L_, tx>, (const void *)&fft_four_step_c2r_kernel<L_, nt>,
            (const void *)&fft_four_step_c2r_self_kernel<L_>};
}

// The self-paired columns, then the pairs of the columns [0, ncols / 2).
template <typename Args>
hipError_t launch_real(int L, const RealKernels &k, Args args, int ncols, hipStream_t s) {
    const bool narrow = use_narrow(L, rc_TX(L), ncols / 2, args.batch);
    const int tx = narrow ? narrow_TX(L, rc_TX(L)) : rc_TX(L);
    if (args.batch <= 0 || ncols % (2 * tx) != 0) return hipErrorInvalidValue;   // whole tiles
    args.ntiles = ncols / 2 / tx;
    const long long nblocks = (long long)args.ntiles * args.batch;
    if (nblocks > 0x7fffffffLL) return hipErrorInvalidValue;
    void *params[] = {&args};
    const hipError_t e = hipLaunchKernel(k.self, dim3(2u * (unsigned)args.batch), dim3(rcs_T(L)), params, 0, s);
    if (e != hipSuccess) return e;
    return hipLaunchKernel(narrow ? k.narrow : k.pairs, dim3((unsigned)nblocks), dim3(L / fs_E(L) * tx), params, 0, s);
}

}  // namespace

hipError_t launch_cols_r2c(int logL, const RealColArgs &a, hipStream_t s) {
    const int L = 1 << logL;
    if (!real_col_fused(logL) || (1 << a.log_cols) % rc_TX(L) != 0) return hipErrorInvalidValue;   // a tile in one image
    switch (logL) {
    case 6: return launch_real(L, r2c_kernels<64>(), a, a.m, s);
    case 7: return launch_real(L, r2c_kernels<128>(), a, a.m, s);
    case 8: return launch_real(L, r2c_kernels<256>(), a, a.m, s);
    case 9: return launch_real(L, r2c_kernels<512>(), a, a.m, s);
    default: return launch_real(L, r2c_kernels<1024>(), a, a.m, s);
    }
}

hipError_t launch_four_step_c2r(int logN1, const RealFourStepArgs &a, hipStream_t s) {
    const int L = 1 << logN1;
    if (!real_four_step_fused(logN1)) return hipErrorInvalidValue;
    switch (logN1) {
    case 8: return launch_real(L, c2r_kernels<256>(), a, a.n2, s);
    case 9: return launch_real(L, c2r_kernels<512>(), a, a.n2, s);
    default: return launch_real(L, c2r_kernels<1024>(), a, a.n2, s);
    }
}

}  // namespace mufft
