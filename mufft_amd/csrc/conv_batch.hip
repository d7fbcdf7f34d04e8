// Persistent kernel for a batch of fast convolutions of uneven sizes.
//
// The reference runs one convolution as three calls (fft.c:799-809): forward
// transform of each input block, then multiply + inverse transform.  Here a
// whole batch of such jobs, of any mix of sizes and of both methods (mono:
// r2c / r2c / c2r, stereo: c2c / full r2c / c2c, fft.c:583-600), runs in one
// persistent launch: forward tasks (both inputs of every job) and inverse
// tasks (the spectrum product fused into their prologue), each inverse task
// starting as soon as its own job group's forward tasks are done.  Tasks of
// equal shape are grouped up to one workgroup's capacity, job groups are
// spread over the XCDs longest-first, and each XCD's workgroups pull its
// tasks from its own queue (a ticket counter); see CBArgs for the ordering.
#include "conv_batch.h"
#include "rows_impl.h"

namespace mufft {

// Fused-kernel variant used inside the persistent kernel (1024 threads): 16
// points per thread with split twiddles; at 2^CB_SPLIT_LOG2 points the same
// variant runs each 16384-point half of the split transform.  It fits
// CB_LDS_BYTES.  The c2r steps read each bin once through mirrored lanes
// where a transform has whole waves (N >= 1024), in chunks below.
MUFFT_HD constexpr int cb_variant(int N) {
    return N >= 1024 ? rv_with_mirror_lanes(rv_make(16, 0, 1)) : rv_with_chunked_loads(rv_make(16, 0, 1));
}
MUFFT_HD constexpr int cb_sub_n(int logn) { return logn >= CB_SPLIT_LOG2 ? (1 << (logn - 1)) : (1 << logn); }

MUFFT_HD constexpr int cb_lds_bytes(int N) {
    return (CB_WG / rv_T(N, cb_variant(N))) * rv_lds_per(N, cb_variant(N)) *
           (rv_xm(cb_variant(N)) == 1 ? 4 : 8);
}

int cb_jobs_per_task(int logn) {
    const int N = cb_sub_n(logn);
    return CB_WG / rv_T(N, cb_variant(N));
}

int cb_points_per_thread(int logn) { return rv_E(cb_sub_n(logn), cb_variant(cb_sub_n(logn))); }

// Tasks and jobs are read by scalar loads, through a uniform pointer in the
// constant address space (the tables never change once a batch is made).  A
// task copied to the stack for the called functions cost every lane a store
// and a load of it, and its fields and the pointers that hang on them vector
// registers.  With the saves below, us: 640 jobs of mixed sizes 123 -> 97, 57
// of 32768 reals 57 -> 47, 128 of 65536 reals 102 -> 81, 256 stereo jobs of
// 16384 points 75 -> 60.
template <typename P>
using CBConst = const __attribute__((address_space(4))) P *;
template <typename P>
__device__ __forceinline__ CBConst<P> cb_const(const P *p) {
    const unsigned long long u = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return (CBConst<P>)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ CBTask cb_load_task(const CBTask *p) {
    CBConst<CBTask> q = cb_const(p);
    CBTask t;
    t.type = q->type;
    t.kind = q->kind;
    t.dir = q->dir;
    t.logn = q->logn;
    t.job0 = q->job0;
    t.njobs = q->njobs;
    t.flags = q->flags;
    t.norm = q->norm;
    t.tw = q->tw;
    t.tw_inv = q->tw_inv;
    t.rtw = q->rtw;
    t.k1 = q->k1;
    t.stw = q->stw;
    t.group = q->group;
    t.nprod = q->nprod;
    return t;
}
__device__ __forceinline__ CBJob cb_load_job(const CBJob *jobs, int i) {
    CBConst<CBJob> q = cb_const(jobs) + i;
    CBJob j;
    j.first = q->first;
    j.second = q->second;
    j.spec1 = q->spec1;
    j.spec2 = q->spec2;
    j.out = q->out;
    return j;
}

// The task functions keep no register of their caller's unless a call to them
// may be a tail call: then they save and restore up to 44 per lane.
#define CB_NOTAIL __attribute__((not_tail_called))

// Jobs [t.job0, t.job0 + t.njobs) of a task, one fused transform each; FL:
// the task's flags if fixed at compile time (RF_DYNAMIC: t.flags).
template <int KIND, int DIR, int LOGN, unsigned FL>
__device__ __forceinline__ void cb_run_rows(const CBTask &t, const CBJob *__restrict__ jobs, int tid,
                                            float2 *smem) {
    constexpr int N = 1 << LOGN;
    constexpr int VAR = cb_variant(N);
    constexpr int T = rv_T(N, VAR);
    constexpr int LDSN = rv_lds_per(N, VAR);
    static_assert(cb_lds_bytes(N) <= CB_LDS_BYTES, "LDS budget of the persistent kernel");
    const int lt = tid & (T - 1);
    const int sub = T >= 64 ? __builtin_amdgcn_readfirstlane(tid / T) : tid / T;
    const bool active = sub < t.njobs;
    const CBJob j = cb_load_job(jobs, t.job0 + (active ? sub : 0));
    const float2 *X;
    const float2 *Y = nullptr;
    float2 *Xo;
    if (t.type == CB_FWD_FIRST) {
        X = j.first;
        Xo = j.spec1;
    } else if (t.type == CB_FWD_SECOND) {
        X = j.second;
        Xo = j.spec2;
    } else {
        X = j.spec1;
        Y = j.spec2;
        Xo = j.out;
    }
    row_transform<N, DIR, KIND, VAR, FL>(X, Y, Xo, active, lt, t.tw, t.rtw, t.flags, t.norm,
                                      smem + sub * LDSN, reinterpret_cast<float *>(smem) + sub * LDSN);
}

// Half t.k1 of one job's transform over two workgroups (split_impl.h).
template <int KIND, int DIR, int LOGN, unsigned FL>
__device__ __forceinline__ void cb_run_split(const CBTask &t, const CBJob *__restrict__ jobs, int tid,
                                             float2 *smem) {
    constexpr int N2 = 1 << (LOGN - 1);
    constexpr int VAR = cb_variant(N2);
    static_assert(cb_lds_bytes(N2) <= CB_LDS_BYTES, "LDS budget of the persistent kernel");
    const CBJob j = cb_load_job(jobs, t.job0);
    const float2 *X = t.type == CB_FWD_FIRST ? j.first : (t.type == CB_FWD_SECOND ? j.second : j.spec1);
    const float2 *Y = t.type == CB_INV ? j.spec2 : nullptr;
    float2 *Xo = t.type == CB_FWD_FIRST ? j.spec1 : (t.type == CB_FWD_SECOND ? j.spec2 : j.out);
    split_transform<N2, 2, DIR, KIND, VAR, FL>(X, Y, Xo, t.k1, tid, t.tw, t.stw, t.rtw, t.flags, t.norm, smem,
                                           reinterpret_cast<float *>(smem));
}

template <int KIND, int DIR, int LOGN, unsigned FL>
__device__ __forceinline__ void cb_run_fl(const CBTask &t, const CBJob *__restrict__ jobs, int tid,
                                          float2 *smem) {
    if constexpr (LOGN >= CB_SPLIT_LOG2) cb_run_split<KIND, DIR, LOGN, FL>(t, jobs, tid, smem);
    else cb_run_rows<KIND, DIR, LOGN, FL>(t, jobs, tid, smem);
}

// The flag sets of the zero-padded convolutions (both inputs padded, the
// usual block convolution) run with their flags fixed at compile time; any
// other set reads them at run time.  Mono: r2c, r2c, c2r with the multiply;
// stereo: c2c, full r2c, c2c with the multiply (conv_batch_host.hip).
template <int KIND, int DIR, int LOGN>
__device__ __noinline__ CB_NOTAIL void cb_run(const CBTask *tp, const CBJob *__restrict__ jobs, int tid,
                                    float2 *smem) {
    const CBTask t = cb_load_task(tp);
    constexpr unsigned FWD = RF_ZERO_PAD | RF_KEEP_OUT;
    if constexpr (KIND == KIND_R2C) {
        if (t.flags == FWD) return cb_run_fl<KIND, DIR, LOGN, FWD>(t, jobs, tid, smem);
        if (t.flags == (FWD | RF_FULL)) return cb_run_fl<KIND, DIR, LOGN, FWD | RF_FULL>(t, jobs, tid, smem);
    } else if constexpr (KIND == KIND_C2C && DIR < 0) {
        if (t.flags == FWD) return cb_run_fl<KIND, DIR, LOGN, FWD>(t, jobs, tid, smem);
    } else {
        if (t.flags == RF_MUL) return cb_run_fl<KIND, DIR, LOGN, (unsigned)RF_MUL>(t, jobs, tid, smem);
    }
    cb_run_fl<KIND, DIR, LOGN, RF_DYNAMIC>(t, jobs, tid, smem);
}

// A pointer to global memory (its accesses are global, not flat, ones).
template <typename P>
struct CBGlobal {
    typedef __attribute__((address_space(1))) P *Ptr;
    Ptr p;
    __device__ __forceinline__ explicit CBGlobal(P *q) : p((Ptr)(uintptr_t)q) {}
    __device__ __forceinline__ std::remove_const_t<P> load(int i) const {
        if constexpr (sizeof(P) == 8) {
            const float x = ((__attribute__((address_space(1))) const float *)p)[2 * i];
            const float y = ((__attribute__((address_space(1))) const float *)p)[2 * i + 1];
            return make_float2(x, y);
        } else {
            return p[i];
        }
    }
    __device__ __forceinline__ void store(int i, float2 v) const {
        ((__attribute__((address_space(1))) float *)p)[2 * i] = v.x;
        ((__attribute__((address_space(1))) float *)p)[2 * i + 1] = v.y;
    }
};

// Whole jobs (CB_JOB, cb_whole_job): both inputs' forward passes, the product
// and the inverse passes with the points in registers.  In three tasks a job
// writes and reads its spectra and waits for its own group; whole, it takes one
// load and one store.  Bound by the latency of its chain of passes.  Stereo: the filter runs as a complex transform of zero imaginary part,
// so the product needs no other point.  Mono: the resolves (kernel.c:36-82)
// pair points k and N-k through LDS.
template <int LOGN, bool STEREO>
__device__ __noinline__ CB_NOTAIL void cb_run_job(const CBTask *tp, const CBJob *__restrict__ jobs, int tid, float2 *smem) {
    const CBTask t = cb_load_task(tp);
    constexpr int N = 1 << LOGN;
    constexpr int VAR = cb_variant(N);
    constexpr int E = rv_E(N, VAR);
    constexpr int LOGE = ilog2(E);
    constexpr int T = rv_T(N, VAR);
    constexpr int TWM = rv_twm(VAR);
    constexpr bool WAVE = T <= 64;
    static_assert(cb_lds_bytes(N) <= CB_LDS_BYTES, "LDS budget of the persistent kernel");
    constexpr bool BUF = T >= 64;   // a wave lies in one job: descriptors, one offset per lane
    const int lt = tid & (T - 1);
    const int sub = BUF ? __builtin_amdgcn_readfirstlane(tid / T) : tid / T;
    const bool active = sub < t.njobs;
    if (WAVE && !active) return;   // no barrier of the workgroup inside
    const CBJob j = cb_load_job(jobs, t.job0 + (active ? sub : 0));
    float2 *L = smem + sub * rv_lds_per(N, VAR);
    auto slot = [](int o) { return pad_slot<LOGE>(o); };
    const bool zp1 = (t.flags & 1u) != 0, zp2 = (t.flags & 2u) != 0;

    // The pointers come from memory: cast to the global address space, or the
    // accesses would be flat ones, which wait for the LDS as well.
    __amdgpu_buffer_rsrc_t rin1, rin2, rout;
    const CBGlobal<const float2> g1(j.first), g2(j.second);
    const CBGlobal<float2> go(j.out);
    if constexpr (BUF) {
        // Zero padding and idle slots by the descriptors' bounds.
        rin1 = make_rsrc(j.first, active ? (zp1 ? N / 2 : N) * 8u : 0u);
        rin2 = make_rsrc(j.second, active ? (zp2 ? N / 2 : N) * (STEREO ? 4u : 8u) : 0u);
        rout = make_rsrc(j.out, active ? N * 8u : 0u);
    }
    float2 u[E], v[E];
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if constexpr (BUF) u[c] = bload_nt(rin1, (unsigned)lt * 8u, T * c * 8u);
        else u[c] = !(zp1 && c >= E / 2) ? g1.load(lt + T * c) : make_float2(0.f, 0.f);
    });
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if constexpr (STEREO && BUF) {
            v[c] = make_float2(__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rin2, lt * 4, T * c * 4, 2)), 0.f);
        } else if constexpr (STEREO) {
            const CBGlobal<const float> f2(reinterpret_cast<const float *>(j.second));
            v[c] = make_float2(!(zp2 && c >= E / 2) ? f2.load(lt + T * c) : 0.f, 0.f);
        } else if constexpr (BUF) {
            v[c] = bload_nt(rin2, (unsigned)lt * 8u, T * c * 8u);
        } else {
            v[c] = !(zp2 && c >= E / 2) ? g2.load(lt + T * c) : make_float2(0.f, 0.f);
        }
    });
    auto passes = [&](auto DIR, float2(&z)[E]) {
        constexpr int dir = decltype(DIR)::value;
        const float2 *tw = dir < 0 ? t.tw : t.tw_inv;
        if constexpr (BUF) {
            constexpr unsigned ntw = (unsigned)(N - seq_first(N, E, np_for(N, E), true));
            stockham_passes<N, E, dir, XM_PAD, TWM, E, WAVE, true>(z, lt, TwBuffer{make_rsrc(tw, ntw * 8u)}, L, nullptr, slot);
        } else {
            const CBGlobal<const float2> g(tw);
            stockham_passes<N, E, dir, XM_PAD, TWM, E, WAVE, true>(
                z, lt, [&](int idx, int k) { return g.load(idx + k); }, L, nullptr, slot);
        }
    };
    constexpr std::integral_constant<int, -1> FWD;
    constexpr std::integral_constant<int, 1> INV;
    passes(FWD, u);
    if constexpr (STEREO) {
        passes(FWD, v);
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            u[c] = cscale(cmul(u[c], v[c]), t.norm);
        });
    } else {
        // Point N - k of every point k = lt + T*c, through LDS (point 0 its own).
        auto partners = [&](const float2(&z)[E], auto use) {
            static_for<0, E>([&](auto C) { L[slot(lt + T * decltype(C)::value)] = z[decltype(C)::value]; });
            exchange_sync<WAVE>();
            static_for<0, E>([&](auto C) {
                constexpr int c = decltype(C)::value;
                use(C, L[slot((N - lt - T * c) & (N - 1))]);
            });
            exchange_sync<WAVE>();
        };
        // W[k] = -i exp(-i pi k / N): one entry per thread and constant rotations.
        const float2 w0 = CBGlobal<const float2>(t.rtw).load(lt);
        // r2c resolve; thread 0's point 0 becomes (X[0], X[N]), both real.
        auto resolve = [&](float2(&z)[E]) {
            partners(z, [&](auto C, float2 p) {
                constexpr int c = decltype(C)::value;
                const float2 za = z[c], zb = cconj(p);
                const float2 x = cscale(cadd(cadd(za, zb), cmul(twc<c, 2 * E, -1>(w0), csub(za, zb))), 0.5f);
                z[c] = c == 0 && lt == 0 ? make_float2(za.x + za.y, za.x - za.y) : x;
            });
        };
        resolve(u);
        passes(FWD, v);
        resolve(v);
        static_for<0, E>([&](auto C) {
            constexpr int c = decltype(C)::value;
            const float2 y = c == 0 && lt == 0 ? make_float2(u[c].x * v[c].x, u[c].y * v[c].y) : cmul(u[c], v[c]);
            u[c] = cscale(y, t.norm);
        });
        // c2r resolve, W'[k] = conj(W[k]).
        partners(u, [&](auto C, float2 p) {
            constexpr int c = decltype(C)::value;
            const float2 ya = u[c], yb = cconj(p);
            const float2 z = cadd(cadd(ya, yb), cmul(csub(ya, yb), cconj(twc<c, 2 * E, -1>(w0))));
            u[c] = c == 0 && lt == 0 ? make_float2(ya.x + ya.y, ya.x - ya.y) : z;
        });
    }
    passes(INV, u);
    static_for<0, E>([&](auto C) {
        constexpr int c = decltype(C)::value;
        if constexpr (BUF) bstore_nt(rout, (unsigned)lt * 8u, T * c * 8u, u[c]);
        else go.store(lt + T * c, u[c]);
    });
}

template <int KIND_, int DIR_>
__device__ __forceinline__ void cb_dispatch_kind(const CBTask *tp, int logn, const CBJob *jobs, int tid, float2 *smem) {
    static_for<CB_MIN_LOG2, CB_SPLIT_LOG2 + 1>([&](auto L) {
        constexpr int l = decltype(L)::value;
        // Parts of the jobs that do not run whole: mono ones of l points, or
        // the stereo ones (whose filter's spectrum has half the points).
        constexpr bool used = KIND_ == KIND_C2C ? !cb_whole_job(l, true)
                                                : !cb_whole_job(l, false) || (KIND_ == KIND_R2C && !cb_whole_job(l + 1, true));
        if constexpr (used)
            if (logn == l) cb_run<KIND_, DIR_, l>(tp, jobs, tid, smem);
    });
}

__device__ __forceinline__ void cb_run_task(const CBTask *tp, const CBTask &t, const CBJob *jobs, int tid, float2 *smem) {
    if (t.type == CB_JOB) {
        static_for<CB_MIN_LOG2, CB_SPLIT_LOG2>([&](auto L) {
            constexpr int l = decltype(L)::value;
            if (t.logn != l) return;
            if (t.kind == KIND_C2C) {
                if constexpr (cb_whole_job(l, true)) cb_run_job<l, true>(tp, jobs, tid, smem);
            } else {
                if constexpr (cb_whole_job(l, false)) cb_run_job<l, false>(tp, jobs, tid, smem);
            }
        });
        return;
    }
    if (t.kind == KIND_R2C) cb_dispatch_kind<KIND_R2C, -1>(tp, t.logn, jobs, tid, smem);
    else if (t.kind == KIND_C2R) cb_dispatch_kind<KIND_C2R, 1>(tp, t.logn, jobs, tid, smem);
    else if (t.dir < 0) cb_dispatch_kind<KIND_C2C, -1>(tp, t.logn, jobs, tid, smem);
    else cb_dispatch_kind<KIND_C2C, 1>(tp, t.logn, jobs, tid, smem);
}

// XCD (die) this workgroup runs on: the hardware XCC_ID register, bits 3:0.
__device__ __forceinline__ int cb_xcd() {
    return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & (CB_XCDS - 1);
}

// Each iteration keeps all of thread 0's work (publishing the previous
// task, the next ticket, the readiness wait) in one region at its top,
// followed by barriers, so the loop compiles to one uniform loop (a second
// thread-0 region at the end of the body let the compiler's control-flow
// structurization send the other lanes of wave 0 back to the barriers ahead
// of thread 0).
__global__ void __launch_bounds__(CB_WG) conv_batch_kernel(CBArgs a) {
    __shared__ float2 smem[CB_LDS_BYTES / 8];
    __shared__ int s_local;
    const int tid = threadIdx.x;
    const int x = cb_xcd();
    const int qb = a.qbegin[x], qn = a.qbegin[x + 1] - qb;
    int prev_group = -1;          // forward task whose completion is to be published
    bool finished_one = false;
    for (;;) {
        if (tid == 0) {
            if (prev_group >= 0)
                __hip_atomic_fetch_add(a.ready + prev_group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (finished_one) atomicAdd(a.done, 1ull);
            const int local = (int)atomicAdd(a.head + x, 1u);
            s_local = local;
            if (local < qn) {
                const CBTask &t = a.tasks[qb + local];
                if (t.type == CB_INV) {
                    const unsigned need = (unsigned)t.nprod;
                    unsigned polls = 0;
                    while (__hip_atomic_load(a.ready + t.group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need) {
                        if (++polls > a.spin_limit) {
                            atomicAdd(a.timeouts, 1ull);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(2);
                    }
                    // Drop stale lines of this CU's L1: the spectra are read from the L2.
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                }
            }
        }
        __syncthreads();
        const int local = __builtin_amdgcn_readfirstlane(s_local);
        __syncthreads();
        if (local >= qn) break;
        const CBTask t = cb_load_task(a.tasks + qb + local);
        cb_run_task(a.tasks + qb + local, t, a.jobs, tid, smem);
        // Forward task: every thread's spectrum stores are complete (in this
        // XCD's L2) before thread 0 publishes the task at the next iteration.
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        __syncthreads();
        prev_group = t.type == CB_INV || t.type == CB_JOB ? -1 : t.group;
        finished_one = true;
    }
    // The last workgroup out clears the queue and readiness counters for the
    // next launch (every other workgroup has made its last access to them).
    if (tid == 0) {
        const unsigned long long f = atomicAdd(a.finish, 1ull);
        if ((f + 1) % gridDim.x == 0) {
            for (int i = 0; i < CB_XCDS; ++i) __hip_atomic_store(a.head + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (int g = 0; g < a.ngroups; ++g)
                __hip_atomic_store(a.ready + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

int cb_resident_workgroups() {
    int dev = 0, ncu = 0, occ = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, conv_batch_kernel, CB_WG, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return ncu * occ;
}

hipError_t launch_conv_batch(const CBArgs &a, int grid, hipStream_t s) {
    if (grid <= 0) return hipSuccess;
    hipLaunchKernelGGL(conv_batch_kernel, dim3(grid), dim3(CB_WG), 0, s, a);
    return hipGetLastError();
}

}  // namespace mufft
