// Overlap-add filtering of a stream in one launch.
//
// A block of hop h = N/2 reals is an n = N/2 point complex transform, zero in
// its upper half.  Forward resolve (kernel.c:47-82), multiply by the filter's
// spectrum H and inverse resolve (kernel.c:36-45) are linear in Z[k] and
// conj(Z[n-k]); with theta = pi k / n, S = H[k] + conj(H[n-k]) and
// D = H[k] - conj(H[n-k]) they come to
//   Z'[k] = (S - D sin(theta)) Z[k] + (i D cos(theta)) conj(Z[n-k]),
// two coefficients per bin, formed once per filter in FP64 (1/N included).
//
// The slots of a workgroup (N / points-per-thread threads each) run forward
// passes, the filter and inverse passes on consecutive blocks with the points
// in registers; the second half of a block, its tail, passes to the next slot
// through LDS and is added there.  A workgroup's first slot runs the block
// before the workgroup's own ones for its tail (the very first one reads the
// previous call's), so workgroups stay independent.  Memory sees each sample
// once in and once out; three launches over spectra and blocks in memory
// moved ten times the samples (N = 4096 x 1024 blocks 28.7 -> 17.0 us, 64 x
// 65536 35.9 -> 11.6, 4096 x 16384 344 -> 138).  What bounds it is the chain of
// passes of one block at few blocks and the passes' instructions at many.
#include "kernels.h"
#include "stockham.h"

namespace mufft {

// MANY: more than one round of blocks per workgroup (a.run); one round needs no
// memory for the last slot's tail, which leaves four workgroups per CU.
template <int N, bool MANY>
__global__ void __launch_bounds__(ola_WG(N), ola_waves_per_simd(N, MANY)) ola_fused_kernel(OlaArgs a) {
    constexpr int E = ola_E(N);
    constexpr int LOGE = ilog2(E);
    constexpr int T = N / E;
    constexpr int B = ola_WG(N) / T;
    constexpr int TWM = N >= 512 ? TW_SPLIT : TW_FULL;
    constexpr bool WAVE = T <= 64;
    constexpr int LDSN = N + N / E;
    constexpr int H = E / 2;
    __shared__ float2 smem[B * LDSN];
    __shared__ float2 last[MANY ? N / 2 : 1];   // tail of the last slot's previous block
    const int tid = threadIdx.x;
    const int lt0 = tid & (T - 1);
    const int sub = tid / T;
    float2 *L = smem + sub * LDSN;
    const long long first = (long long)blockIdx.x * ((MANY ? a.run : 1) * B - 1) - 1;
    auto slot = [](int o) { return pad_slot<LOGE>(o); };

    // Blocks past the end work on zeros and store nothing.
    const int run = MANY ? a.run : 1;
    for (int i = 0; i < run; ++i) {
        int lt = lt0;
        // Keeps the table loads inside the loop: hoisted, they hold up to 120
        // registers and halve the workgroups per CU.
        asm volatile("" : "+v"(lt));
        const long long b = first + (long long)i * B + sub;
        const bool in = b >= 0 && b < a.nblocks;
        const float2 *src = a.in + (in ? b : 0) * (N / 2);
        float2 v[E];
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            v[c] = c < H && in ? src[lt + T * c] : make_float2(0.f, 0.f);
        });
        stockham_passes<N, E, -1, XM_PAD, TWM, E, WAVE, true>(v, lt, TwGlobal{a.tw_fwd}, L, nullptr, slot);
        // Z[n-k] of point k = lt + T*c.
        static_for<0, E>([&](auto C) { L[slot(lt + T * decltype(C)::value)] = v[decltype(C)::value]; });
        exchange_sync<WAVE>();
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            const int k = lt + T * c;
            const float2 zn = cconj(L[slot((N - k) & (N - 1))]);
            v[c] = cadd(cmul(a.ca[k], v[c]), cmul(a.cb[k], zn));
        });
        exchange_sync<WAVE>();
        stockham_passes<N, E, 1, XM_PAD, TWM, E, WAVE, true>(v, lt, TwGlobal{a.tw_inv}, L, nullptr, slot);
        if (b == -1) static_for<0, H>([&](auto C) { v[H + decltype(C)::value] = a.tail_in[lt + T * decltype(C)::value]; });
        static_for<0, H>([&](auto C) { L[slot(lt + T * decltype(C)::value)] = v[H + decltype(C)::value]; });
        __syncthreads();
        if (in && (i > 0 || sub > 0)) {
            float2 *dst = a.out + b * (N / 2);
            const float2 *P = L - LDSN;   // the previous slot's tail
            static_for<0, H>([&](auto C) {
                constexpr int c = decltype(C)::value;
                const float2 p = !MANY || sub > 0 ? P[slot(lt + T * c)] : last[lt + T * c];
                dst[lt + T * c] = cadd(v[c], p);
            });
            if (b == a.nblocks - 1)
                static_for<0, H>([&](auto C) { a.tail_out[lt + T * decltype(C)::value] = v[H + decltype(C)::value]; });
        }
        if constexpr (!MANY) break;
        __syncthreads();
        if (sub == B - 1) static_for<0, H>([&](auto C) { last[lt + T * decltype(C)::value] = v[H + decltype(C)::value]; });
    }
}

// The coefficients of the filter (see above) from its spectrum H[0..n].
__global__ void __launch_bounds__(256) ola_coeff_kernel(const float2 *H, float2 *ca, float2 *cb, int n) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const double norm = 0.5 / (double)n;   // 1/N
    const double hr = H[k].x, hi = H[k].y, gr = H[n - k].x, gi = -(double)H[n - k].y;
    const double sr = hr + gr, si = hi + gi, dr = hr - gr, di = hi - gi;
    const double theta = 3.14159265358979323846 * (double)k / (double)n;
    const double sn = sin(theta), cs = cos(theta);
    ca[k] = make_float2((float)(norm * (sr - dr * sn)), (float)(norm * (si - di * sn)));
    cb[k] = make_float2((float)(-norm * di * cs), (float)(norm * dr * cs));
}

hipError_t launch_ola_coeff(const float2 *H, float2 *ca, float2 *cb, int n, hipStream_t s) {
    hipLaunchKernelGGL(ola_coeff_kernel, dim3((n + 255) / 256), dim3(256), 0, s, H, ca, cb, n);
    return hipGetLastError();
}

template <int N>
static const void *ola_kernel(bool many) {
    if constexpr (ola_rounds(N))
        if (many) return (const void *)&ola_fused_kernel<N, true>;
    return (const void *)&ola_fused_kernel<N, false>;
}

static const void *ola_kernel_ptr(int logn, bool many) {
    switch (logn) {
    case 1: return ola_kernel<2>(many);
    case 2: return ola_kernel<4>(many);
    case 3: return ola_kernel<8>(many);
    case 4: return ola_kernel<16>(many);
    case 5: return ola_kernel<32>(many);
    case 6: return ola_kernel<64>(many);
    case 7: return ola_kernel<128>(many);
    case 8: return ola_kernel<256>(many);
    case 9: return ola_kernel<512>(many);
    case 10: return ola_kernel<1024>(many);
    case 11: return ola_kernel<2048>(many);
    case 12: return ola_kernel<4096>(many);
    default: return nullptr;
    }
}

hipError_t launch_ola_fused(int logn, const OlaArgs &a, hipStream_t s) {
    if (logn < 1 || logn > OLA_MAX_LOG2 || a.nblocks <= 0) return hipErrorInvalidValue;
    const int n = 1 << logn;
    OlaArgs args = a;
    args.run = ola_run(n, a.nblocks);
    const void *k = ola_kernel_ptr(logn, args.run > 1);
    if (!k) return hipErrorInvalidValue;
    const long long per = (long long)args.run * ola_slots(n) - 1;   // blocks per workgroup
    const long long nblk = (a.nblocks + per - 1) / per;
    if (nblk > 0x7fffffffLL) return hipErrorInvalidValue;
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3((unsigned)nblk), dim3(ola_WG(n)), params, 0, s);
}

}  // namespace mufft
