// riemann_fp64.hip -- plain FP64 Riemann solvers for gfx950.
//
// Compiled with -ffp-contract=off: expressions keep the association of
// the reference (Shadowfax src/riemann/ExactRiemannSolver.cpp,
// src/riemann/HLLCRiemannSolver.cpp), so results differ from the CPU
// reference only by round-off: the exact solver runs the same iteration over
// a cheaper pressure function (riemann_fp64_impl.h).
//
// One lane per problem, SoA loads/stores (fully coalesced, 144 B per 3D
// problem with v = 0).  The exact solver's Newton/Brent loops run per lane
// with an iteration cap; divergence handling is left to the hardware.

#include "riemann_fp64_impl.h"
#include "sfx_device.h"
#include "sfx_launch.h"

namespace sfx {
namespace fp64 {

// Waves per SIMD the kernels are held to: 4, and 3 for the exact solver of other
// gases than 5/3 and 7/5, whose pow() spills at 4 (gamma 1.66667, 262,144 3D
// problems: 115 us at 3, 123 at 4, 122 at 2; 2D 112, 123, 126).
template <int KIND, int ROOT>
constexpr int solver_waves() {
    return KIND == 0 && ROOT == 0 ? 3 : 4;
}

// --------------------------------------------------------------- kernels --

template <int ND, int KIND, int ROOT = 0>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(solver_waves<KIND, ROOT>()))) void solve_for_flux_kernel(
        Consts c, int64_t N, const double* __restrict__ WL, const double* __restrict__ WR,
        const double* __restrict__ n, const double* __restrict__ v,
        const uint8_t* __restrict__ refl, double* __restrict__ F,
        uint8_t* __restrict__ status, unsigned long long* __restrict__ ctr) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned iters = 0, brent = 0, vac = 0, fail = 0, valid = 0;
    if(i < N) {
        valid = 1;
        double wl[NC], wr[NC], nn[ND], vv[ND], f[NC];
#pragma unroll
        for(int k = 0; k < NC; k++) {
            wl[k] = WL[k * N + i];
            wr[k] = WR[k * N + i];
        }
#pragma unroll
        for(int d = 0; d < ND; d++) {
            nn[d] = n[d * N + i];
            vv[d] = v ? v[d * N + i] : 0.;
        }
        const bool r = refl ? refl[i] != 0 : false;
        uint8_t st;
        if(KIND == 0)
            st = ex_solve_for_flux<ND, ROOT>(c, wl, wr, nn, vv, r, f, iters, brent, vac);
        else
            st = hllc_solve_for_flux<ND>(c, wl, wr, nn, vv, r, f, vac);
#pragma unroll
        for(int k = 0; k < NC; k++) F[k * N + i] = f[k];
        if(status) status[i] = st;
        fail = st != 0;
    }
    const unsigned cv[CNT_N] = {valid, brent, vac, iters, fail};
    block_add_counters(ctr, cv);
}

template <int ND, int ROOT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(solver_waves<0, ROOT>()))) void exact_solve_kernel(
        Consts c, int64_t N, const double* __restrict__ WL, const double* __restrict__ WR,
        const double* __restrict__ n, const uint8_t* __restrict__ refl,
        double* __restrict__ Whalf, double* __restrict__ WRout, double* __restrict__ mach_io,
        uint8_t* __restrict__ status, unsigned long long* __restrict__ ctr) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned iters = 0, brent = 0, vac = 0, fail = 0, valid = 0;
    if(i < N) {
        valid = 1;
        double wl[NC], wr[NC], nn[ND], w[NC];
#pragma unroll
        for(int k = 0; k < NC; k++) {
            wl[k] = WL[k * N + i];
            wr[k] = WR[k * N + i];
        }
#pragma unroll
        for(int d = 0; d < ND; d++) nn[d] = n[d * N + i];
        double mach = mach_io ? mach_io[i] : 0.;
        uint8_t st = ex_solve<ND, ROOT>(c, wl, wr, nn, refl ? refl[i] != 0 : false, w, &mach,
                                  iters, brent, vac);
#pragma unroll
        for(int k = 0; k < NC; k++) {
            Whalf[k * N + i] = w[k];
            if(WRout) WRout[k * N + i] = wr[k];
        }
        if(mach_io) mach_io[i] = mach;
        if(status) status[i] = st;
        fail = st != 0;
    }
    const unsigned cv[CNT_N] = {valid, brent, vac, iters, fail};
    block_add_counters(ctr, cv);
}

// One lane solves one problem (see ScalarIn).  Bounds as the batch kernels':
// the general path that they share, out of line, gets the registers of its
// least bound caller, and they reserve as many (244 instead of 128: 262,144
// problems 60 us instead of 47).
template <int ND, int KIND, int ROOT, bool SOLVE>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(solver_waves<KIND, ROOT>()))) void scalar_kernel(
        Consts c, ScalarIn in, ScalarOut* __restrict__ out, unsigned long long* __restrict__ ctr) {
    if(threadIdx.x) return;
    unsigned iters = 0, brent = 0, vac = 0;
    double f[ND + 2], mach = in.mach;
    uint8_t st;
    if constexpr(SOLVE) {
        st = ex_solve<ND, ROOT>(c, in.WL, in.WR, in.n, in.reflective != 0, f, &mach, iters, brent,
                                vac);
    } else if constexpr(KIND == 0) {
        st = ex_solve_for_flux<ND, ROOT>(c, in.WL, in.WR, in.n, in.v, in.reflective != 0, f, iters,
                                         brent, vac);
    } else {
        st = hllc_solve_for_flux<ND>(c, in.WL, in.WR, in.n, in.v, in.reflective != 0, f, vac);
    }
    const unsigned cv[CNT_N] = {1u, brent, vac, iters, st != 0};
    lane_add_counters(ctr, cv);
#pragma unroll
    for(int k = 0; k < ND + 2; k++) out->out[k] = f[k];
    out->mach = mach;
    out->status = st;
    // everything above is on its way before the host sees the number
    __hip_atomic_store(&out->seq, in.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace fp64

// ------------------------------------------------------------ launchers --

hipError_t launch_scalar_fp64(int kind, int ndim, bool solve_only, const Consts& c,
                              const ScalarIn& in, ScalarOut* out, unsigned long long* ctr,
                              hipStream_t stream) {
    auto run = [&](auto nd) {
        constexpr int ND = decltype(nd)::value;
        if(kind != 0) {
            hipLaunchKernelGGL((fp64::scalar_kernel<ND, 1, 0, false>), dim3(1), dim3(64), 0, stream,
                               c, in, out, ctr);
            return;
        }
        with_root<true>(c, [&](auto root) {
            constexpr int ROOT = decltype(root)::value;
            if(solve_only)
                hipLaunchKernelGGL((fp64::scalar_kernel<ND, 0, ROOT, true>), dim3(1), dim3(64), 0,
                                   stream, c, in, out, ctr);
            else
                hipLaunchKernelGGL((fp64::scalar_kernel<ND, 0, ROOT, false>), dim3(1), dim3(64), 0,
                                   stream, c, in, out, ctr);
        });
    };
    if(ndim == 3)
        run(std::integral_constant<int, 3>());
    else
        run(std::integral_constant<int, 2>());
    return hipGetLastError();
}

static inline unsigned nblocks(int64_t N, int bs) { return (unsigned)((N + bs - 1) / bs); }

hipError_t launch_solve_for_flux_fp64(int kind, int ndim, const Consts& c, int64_t N,
                                      const double* WL, const double* WR, const double* n,
                                      const double* v, const uint8_t* refl, double* F,
                                      uint8_t* status, unsigned long long* ctr,
                                      hipStream_t stream) {
    if(N <= 0) return hipSuccess;
    const int bs = 256;
    dim3 grid(nblocks(N, bs)), block(bs);
    auto solve = [&](auto nd, auto k) {
        constexpr int ND = decltype(nd)::value, K = decltype(k)::value;
        with_root<K == 0>(c, [&](auto root) {
            hipLaunchKernelGGL((fp64::solve_for_flux_kernel<ND, K, decltype(root)::value>), grid,
                               block, 0, stream, c, N, WL, WR, n, v, refl, F, status, ctr);
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

hipError_t launch_exact_solve_fp64(int ndim, const Consts& c, int64_t N, const double* WL,
                                   const double* WR, const double* n, const uint8_t* refl,
                                   double* Whalf, double* WRout, double* mach, uint8_t* status,
                                   unsigned long long* ctr, hipStream_t stream) {
    if(N <= 0) return hipSuccess;
    const int bs = 256;
    dim3 grid(nblocks(N, bs)), block(bs);
    with_root<true>(c, [&](auto root) {
        constexpr int ROOT = decltype(root)::value;
        if(ndim == 3)
            hipLaunchKernelGGL((fp64::exact_solve_kernel<3, ROOT>), grid, block, 0, stream, c, N,
                               WL, WR, n, refl, Whalf, WRout, mach, status, ctr);
        else
            hipLaunchKernelGGL((fp64::exact_solve_kernel<2, ROOT>), grid, block, 0, stream, c, N,
                               WL, WR, n, refl, Whalf, WRout, mach, status, ctr);
    });
    return hipGetLastError();
}

}  // namespace sfx
