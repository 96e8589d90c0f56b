// riemann_mixed.hip -- batched mixed-precision solve_for_flux kernels; the
// algorithm and its precision split are described in riemann_mixed_impl.h.
#include "riemann_mixed_impl.h"
#include "sfx_launch.h"

#include <algorithm>

namespace sfx {
namespace mixed {

#ifndef SFX_MIXED_WAVES  // waves per SIMD the exact kernels are held to (4M problems: 115 us;
#define SFX_MIXED_WAVES 6  // 5: 124, 4: 128, 8, spilling: 134)
#endif

template <int ND, int KIND, typename T, int ROOT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(ROOT != 0 ? SFX_MIXED_WAVES : 1, 10))) void solve_for_flux_kernel(
        CF c, Consts cd, int64_t N, const T* __restrict__ WL, const T* __restrict__ WR,
        const T* __restrict__ n, const T* __restrict__ v, const uint8_t* __restrict__ refl,
        T* __restrict__ F, uint8_t* __restrict__ status, unsigned long long* __restrict__ ctr) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned iters = 0, vac = 0, fail = 0, valid = 0;
    if(i < N) {
        valid = 1;
        double wl64[NC], wr64[NC], n64[ND], v64[ND], f[NC];
#pragma unroll
        for(int k = 0; k < NC; k++) {
            wl64[k] = (double)WL[k * N + i];
            wr64[k] = (double)WR[k * N + i];
        }
#pragma unroll
        for(int d = 0; d < ND; d++) {
            n64[d] = (double)n[d * N + i];
            v64[d] = v ? (double)v[d * N + i] : 0.0;
        }
        const bool r = refl ? refl[i] != 0 : false;
        uint8_t st;
        if(KIND == 0) {
            st = exact_mixed<ND, ROOT>(c, cd, r, wl64, wr64, n64, v64, f, iters, vac);
        } else {
            st = hllc_mixed<ND>(c, cd, wl64, wr64, n64, v64, r, f, vac);
        }
#pragma unroll
        for(int k = 0; k < NC; k++) F[k * N + i] = (T)f[k];
        if(status) status[i] = st;
        fail = st != 0;
    }
    const unsigned cv[CNT_N] = {valid, 0u, vac, iters, fail};
    block_add_counters(ctr, cv);
}

// One lane solves one problem (see ScalarIn).  Bounds as the batch kernels':
// the general path that they share, out of line, gets the registers of its
// least bound caller, and they reserve as many (134 instead of 80: 4,194,304
// problems 121 us instead of 92).
template <int ND, int KIND, int ROOT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(ROOT != 0 ? SFX_MIXED_WAVES : 1, 10))) void scalar_kernel(
        CF c, Consts cd, ScalarIn in, ScalarOut* __restrict__ out,
        unsigned long long* __restrict__ ctr) {
    if(threadIdx.x) return;
    unsigned iters = 0, vac = 0;
    double f[ND + 2];
    uint8_t st;
    if constexpr(KIND == 0)
        st = exact_mixed<ND, ROOT>(c, cd, in.reflective != 0, in.WL, in.WR, in.n, in.v, f, iters,
                                   vac);
    else
        st = hllc_mixed<ND>(c, cd, in.WL, in.WR, in.n, in.v, in.reflective != 0, f, vac);
    const unsigned cv[CNT_N] = {1u, 0u, vac, iters, st != 0};
    lane_add_counters(ctr, cv);
#pragma unroll
    for(int k = 0; k < ND + 2; k++) out->out[k] = f[k];
    out->mach = in.mach;
    out->status = st;
    // everything above is on its way before the host sees the number
    __hip_atomic_store(&out->seq, in.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- exact solver in two phases (wave-level compaction) -----------------
//
// Phase 1 runs every problem's setup and at most `stop` FP32 Newton
// iterations; problems still iterating after that (strong shocks, near
// vacuum) are written, with their iteration state, to their block's segment
// of a queue (slots from wave ballots and one LDS counter per block -- no
// global atomics), and the wave finishes the converged ones together instead
// of idling while a few lanes iterate on.  Phase 2 gives each block the
// stragglers of kSegs consecutive phase-1 segments, packed densely through a
// prefix sum of their counts, resumes each problem where it stopped and
// finishes it.  The iteration sequence per problem is unchanged, so results
// are bit-identical to the one-kernel path.
//
// Problems of the general iteration are queued as they are (it = -1) and
// solved at the end of phase 2: phase 1 holds no call.  With one, phase 1
// spilled 76 registers at the 6 waves of the one-kernel path, and 4,194,304
// 3D problems queued after 4 iterations took 240 us, 128 so (phase 2 at 4
// waves, where neither kernel spills).

struct Straggler {
    int32_t i;
    float p, lo, hi;  // the iterate (p, or z alone) and its bracket
    int32_t it;
};

// the two iterations' parts under one name; finish takes no problem of phase
// EX_GENERAL
template <int ND, int ROOT>
struct Parts {
    using Case = std::conditional_t<ROOT != 0, RootCase, ExactCase>;
    static __device__ __forceinline__ void setup(const CF& c, const Consts& cd, bool refl,
                                                 const double* WL, double* WR, const double* n,
                                                 Case& s) {
        if constexpr(ROOT != 0) {
            root_setup<ND, ROOT>(c, cd, refl, WL, WR, n, s);
        } else {
            float wl[ND + 2], wr[ND + 2], nn[ND];
#pragma unroll
            for(int k = 0; k < ND + 2; k++) {
                wl[k] = (float)WL[k];
                wr[k] = (float)WR[k];
            }
#pragma unroll
            for(int d = 0; d < ND; d++) nn[d] = (float)n[d];
            exact_setup<ND>(c, cd, wl, wr, nn, refl, WL, WR, n, s);
        }
    }
    static __device__ __forceinline__ void iterate(const CF& c, const Consts& cd, Case& s,
                                                   int stop) {
        if constexpr(ROOT != 0)
            root_iterate<ROOT>(c, cd, s, stop);
        else
            exact_iterate(c, s, stop);
    }
    static __device__ __forceinline__ uint8_t finish(const CF& c, const Consts& cd, const Case& s,
                                                     const double* WL, const double* WR,
                                                     const double* n, const double* v, bool refl,
                                                     double* F, unsigned& iters, unsigned& vac) {
        if constexpr(ROOT != 0)
            return root_finish<ND, ROOT, false>(c, cd, s, WL, WR, n, v, refl, F, iters, vac);
        else
            return exact_finish<ND>(c, cd, s, WL, WR, n, v, F, iters, vac);
    }
    static __device__ __forceinline__ void save(const Case& s, Straggler& g) {
        if constexpr(ROOT != 0) {
            g.p = s.z;
            g.lo = g.hi = 0.f;
        } else {
            g.p = s.p;
            g.lo = s.lo;
            g.hi = s.hi;
        }
        g.it = s.it;
    }
    static __device__ __forceinline__ void restore(const Straggler& g, Case& s) {
        if constexpr(ROOT != 0) {
            s.z = g.p;
        } else {
            s.p = g.p;
            s.lo = g.lo;
            s.hi = g.hi;
        }
        s.it = g.it;
    }
};

constexpr int kSegs = 16;  // phase-1 segments per phase-2 block

template <int ND, typename T>
__device__ __forceinline__ void load_problem(int64_t N, int64_t i, const T* __restrict__ WL,
                                             const T* __restrict__ WR, const T* __restrict__ n,
                                             const T* __restrict__ v, double* wl64, double* wr64,
                                             double* n64, double* v64) {
    const int NC = ND + 2;
#pragma unroll
    for(int k = 0; k < NC; k++) {
        wl64[k] = (double)WL[k * N + i];
        wr64[k] = (double)WR[k * N + i];
    }
#pragma unroll
    for(int d = 0; d < ND; d++) {
        n64[d] = (double)n[d * N + i];
        v64[d] = v ? (double)v[d * N + i] : 0.0;
    }
}

template <int ND, typename T, int ROOT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(ROOT != 0 ? SFX_MIXED_WAVES : 1, 10))) void exact_phase1_kernel(
        CF c, Consts cd, int64_t N, const T* __restrict__ WL, const T* __restrict__ WR,
        const T* __restrict__ n, const T* __restrict__ v, const uint8_t* __restrict__ refl,
        T* __restrict__ F, uint8_t* __restrict__ status, unsigned long long* __restrict__ ctr,
        Straggler* __restrict__ queue, unsigned* __restrict__ counts, int stop) {
    const int NC = ND + 2;
    __shared__ unsigned s_cnt;
    if(threadIdx.x == 0) s_cnt = 0u;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < N;
    unsigned iters = 0, vac = 0, fail = 0, done = 0;
    double wl64[NC], wr64[NC], n64[ND], v64[ND];
    using X = Parts<ND, ROOT>;
    typename X::Case s;
    s.phase = EX_DONE;
    bool r = false;
    if(valid) {
        load_problem<ND, T>(N, i, WL, WR, n, v, wl64, wr64, n64, v64);
        r = refl ? refl[i] != 0 : false;
        X::setup(c, cd, r, wl64, wr64, n64, s);
        if(s.phase == EX_ITER) X::iterate(c, cd, s, stop);
    }
    const bool strag = valid && (s.phase == EX_ITER || s.phase == EX_GENERAL);
    // slots in the block's segment: a ballot per wave, one LDS atomic per wave
    const unsigned long long mask = __ballot(strag);
    const int lane = __lane_id();
    unsigned base = 0;
    if(lane == 0 && mask) base = atomicAdd(&s_cnt, (unsigned)__popcll(mask));
    base = __shfl(base, 0);
    if(strag) {
        const unsigned slot = base + (unsigned)__popcll(mask & ((1ull << lane) - 1ull));
        Straggler g;
        g.i = (int32_t)i;
        if(s.phase == EX_GENERAL) {
            g.p = g.lo = g.hi = 0.f;
            g.it = -1;
        } else {
            X::save(s, g);
        }
        queue[(int64_t)blockIdx.x * blockDim.x + slot] = g;
    } else if(valid) {
        double f[NC];
        const uint8_t st = X::finish(c, cd, s, wl64, wr64, n64, v64, r, f, iters, vac);
#pragma unroll
        for(int k = 0; k < NC; k++) F[k * N + i] = (T)f[k];
        if(status) status[i] = st;
        fail = st != 0;
        done = 1;
    }
    __syncthreads();
    if(threadIdx.x == 0) counts[blockIdx.x] = s_cnt;
    const unsigned cv[CNT_N] = {done, 0u, vac, iters, fail};
    block_add_counters(ctr, cv);
}

template <int ND, typename T, int ROOT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(ROOT != 0 ? 4 : 1, 10))) void exact_phase2_kernel(
        CF c, Consts cd, int64_t N, const T* __restrict__ WL, const T* __restrict__ WR,
        const T* __restrict__ n, const T* __restrict__ v, const uint8_t* __restrict__ refl,
        T* __restrict__ F, uint8_t* __restrict__ status, unsigned long long* __restrict__ ctr,
        const Straggler* __restrict__ queue, const unsigned* __restrict__ counts,
        int64_t nsegs) {
    const int NC = ND + 2;
    using X = Parts<ND, ROOT>;
    __shared__ unsigned s_pre[kSegs + 1];
    const int64_t seg0 = (int64_t)blockIdx.x * kSegs;
    if(threadIdx.x == 0) {
        unsigned acc = 0;
        for(int q = 0; q < kSegs; q++) {
            s_pre[q] = acc;
            acc += (seg0 + q < nsegs) ? counts[seg0 + q] : 0u;
        }
        s_pre[kSegs] = acc;
    }
    __syncthreads();
    const unsigned total = s_pre[kSegs];
    unsigned iters = 0, vac = 0, fail = 0, done = 0;
    int general = 0;
    const auto entry = [&](unsigned k) {
        int q = 0;
        while(q + 1 < kSegs && s_pre[q + 1] <= k) q++;
        return queue[(seg0 + q) * blockDim.x + (k - s_pre[q])];
    };
    const auto put = [&](int64_t i, uint8_t st, const double* f) {
#pragma unroll
        for(int r = 0; r < NC; r++) F[r * N + i] = (T)f[r];
        if(status) status[i] = st;
        fail += st != 0;
        done++;
    };
    for(unsigned k = threadIdx.x; k < total; k += blockDim.x) {
        const Straggler g = entry(k);
        const int64_t i = g.i;
        if(ROOT != 0 && g.it < 0) {
            general = 1;
            continue;
        }
        double wl64[NC], wr64[NC], n64[ND], v64[ND], f[NC];
        load_problem<ND, T>(N, i, WL, WR, n, v, wl64, wr64, n64, v64);
        const bool rf = refl ? refl[i] != 0 : false;
        typename X::Case s;
        X::setup(c, cd, rf, wl64, wr64, n64, s);
        X::restore(g, s);
        X::iterate(c, cd, s, c.itmax);
        put(i, X::finish(c, cd, s, wl64, wr64, n64, v64, rf, f, iters, vac), f);
    }
    // the general iteration's problems in a loop of their own: a call in the
    // one above would spill its values
    if constexpr(ROOT != 0) {
        if(__syncthreads_or(general))
            for(unsigned k = threadIdx.x; k < total; k += blockDim.x) {
                const Straggler g = entry(k);
                if(g.it >= 0) continue;
                double wl64[NC], wr64[NC], n64[ND], v64[ND], f[NC];
                load_problem<ND, T>(N, g.i, WL, WR, n, v, wl64, wr64, n64, v64);
                unsigned vk = 0;
                put(g.i,
                    call_general<ND, 1>(c, cd, wl64, wr64, n64, v64, refl ? refl[g.i] != 0 : false,
                                        f, iters, vk),
                    f);
                vac += vk;
            }
    }
    const unsigned cv[CNT_N] = {done, 0u, vac, iters, fail};
    block_add_counters(ctr, cv);
}

}  // namespace mixed

hipError_t launch_scalar_mixed(int kind, int ndim, const Consts& c, const ScalarIn& in,
                               ScalarOut* out, unsigned long long* ctr, hipStream_t stream) {
    const mixed::CF cf = mixed::make_cf(c);
    auto run = [&](auto nd) {
        constexpr int ND = decltype(nd)::value;
        if(kind != 0)
            hipLaunchKernelGGL((mixed::scalar_kernel<ND, 1, 0>), dim3(1), dim3(64), 0, stream, cf, c,
                               in, out, ctr);
        else
            with_root<true>(c, [&](auto root) {
                hipLaunchKernelGGL((mixed::scalar_kernel<ND, 0, decltype(root)::value>), dim3(1),
                                   dim3(64), 0, stream, cf, c, in, out, ctr);
            });
    };
    if(ndim == 3)
        run(std::integral_constant<int, 3>());
    else
        run(std::integral_constant<int, 2>());
    return hipGetLastError();
}

size_t exact_split_scratch_bytes(int64_t N) {
    const int64_t nb = (std::max<int64_t>(N, 1) + 255) / 256;
    return (size_t)(((4 * nb + 255) / 256) * 256) + sizeof(mixed::Straggler) * (size_t)(nb * 256);
}

template <typename T>
hipError_t launch_exact_mixed_split(int ndim, const Consts& c, int64_t N, const T* WL,
                                    const T* WR, const T* n, const T* v, const uint8_t* refl,
                                    T* F, uint8_t* status, unsigned long long* ctr,
                                    void* scratch, int stop, int persistent_blocks,
                                    hipStream_t stream) {
    (void)persistent_blocks;
    if(N <= 0) return hipSuccess;
    const mixed::CF cf = mixed::make_cf(c);
    const int64_t nb = (N + 255) / 256;
    unsigned* counts = (unsigned*)scratch;
    mixed::Straggler* queue =
            (mixed::Straggler*)((char*)scratch + ((4 * nb + 255) / 256) * 256);
    const dim3 grid((unsigned)nb), block(256),
            grid2((unsigned)((nb + mixed::kSegs - 1) / mixed::kSegs));
    auto split = [&](auto nd) {
        constexpr int ND = decltype(nd)::value;
        with_root<true>(c, [&](auto root) {
            constexpr int ROOT = decltype(root)::value;
            hipLaunchKernelGGL((mixed::exact_phase1_kernel<ND, T, ROOT>), grid, block, 0, stream,
                               cf, c, N, WL, WR, n, v, refl, F, status, ctr, queue, counts, stop);
            hipLaunchKernelGGL((mixed::exact_phase2_kernel<ND, T, ROOT>), grid2, block, 0, stream,
                               cf, c, N, WL, WR, n, v, refl, F, status, ctr, queue, counts, nb);
        });
    };
    if(ndim == 3)
        split(std::integral_constant<int, 3>());
    else
        split(std::integral_constant<int, 2>());
    return hipGetLastError();
}

template hipError_t launch_exact_mixed_split<float>(int, const Consts&, int64_t, const float*,
                                                    const float*, const float*, const float*,
                                                    const uint8_t*, float*, uint8_t*,
                                                    unsigned long long*, void*, int, int,
                                                    hipStream_t);
template hipError_t launch_exact_mixed_split<double>(int, const Consts&, int64_t, const double*,
                                                     const double*, const double*, const double*,
                                                     const uint8_t*, double*, uint8_t*,
                                                     unsigned long long*, void*, int, int,
                                                     hipStream_t);

template <typename T>
hipError_t launch_solve_for_flux_mixed(int kind, int ndim, const Consts& c, int64_t N,
                                       const T* WL, const T* WR, const T* n, const T* v,
                                       const uint8_t* refl, T* F, uint8_t* status,
                                       unsigned long long* ctr, hipStream_t stream) {
    if(N <= 0) return hipSuccess;
    const mixed::CF cf = mixed::make_cf(c);
    const int bs = 256;
    dim3 grid((unsigned)((N + bs - 1) / bs)), block(bs);
    auto solve = [&](auto nd, auto k) {
        constexpr int ND = decltype(nd)::value, K = decltype(k)::value;
        with_root<K == 0>(c, [&](auto root) {
            hipLaunchKernelGGL((mixed::solve_for_flux_kernel<ND, K, T, decltype(root)::value>),
                               grid, block, 0, stream, cf, c, N, WL, WR, n, v, refl, F, status,
                               ctr);
        });
    };
    const std::integral_constant<int, 0> exact;
    const std::integral_constant<int, 1> hllc;
    const std::integral_constant<int, 2> d2;
    const std::integral_constant<int, 3> d3;
    if(ndim == 3) kind == 0 ? solve(d3, exact) : solve(d3, hllc);
    else kind == 0 ? solve(d2, exact) : solve(d2, hllc);
    return hipGetLastError();
}

template hipError_t launch_solve_for_flux_mixed<float>(int, int, const Consts&, int64_t,
                                                       const float*, const float*, const float*,
                                                       const float*, const uint8_t*, float*,
                                                       uint8_t*, unsigned long long*,
                                                       hipStream_t);
template hipError_t launch_solve_for_flux_mixed<double>(int, int, const Consts&, int64_t,
                                                        const double*, const double*,
                                                        const double*, const double*,
                                                        const uint8_t*, double*, uint8_t*,
                                                        unsigned long long*, hipStream_t);

}  // namespace sfx
