// sfx_device.h -- device-side building blocks shared by the HIP kernels.
//
// Layout conventions (all kernels):
//   states are SoA, component-major: X[k*N + i], k in [0, ndim+2)
//   W = [rho, v_1..v_ndim, p], Q = [m, p_1..p_ndim, e]
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace sfx {

// Solver constants derived from gamma exactly as the reference derives them
// (src/riemann/ExactRiemannSolver.cpp:52-61), computed on the host.
struct Consts {
    double gamma;
    double gp1d2g, gm1d2g, gm1dgp1, tdgp1, tdgm1, gm1d2, tgdgm1, ginv;
    double tol, cutoff;
    int itercap;   // bound on Newton and on Brent iterations (reference: none)
    int fast53;    // gamma == 5/3: exponents 0.2, 0.6, 0.8, 3, 5 (mixed path)
    // exact solvers: 2 gamma/(gamma-1) where that is 5 (gamma = 5/3) or 7
    // (gamma = 7/5), else 0; 1/root and (1 + 1/root)/(2 root), its root
    // series; sqrt(2/(gamma (gamma+1)))
    int root;
    // 1/root; ((g-1)/(2g) - 1/root) ln 2; (2/(g-1) - (root - 2)) ln 2
    float rootf, rootk, fank;
    double rn, rn2, kshock;
};

// f(std::integral_constant<int, ROOT>) for the kernels that take Consts::root
// as a template parameter: the exact solvers' (exact), 0 for HLLC's
template <bool exact, class Fn>
inline void with_root(const Consts& c, Fn f) {
    if constexpr(exact) {
        if(c.root == 5) return f(std::integral_constant<int, 5>());
        if(c.root == 7) return f(std::integral_constant<int, 7>());
    }
    f(std::integral_constant<int, 0>());
}

// status bits, one byte per problem / face / cell
enum : uint8_t {
    ST_SOLVER = 1,   // NaN or negative solution (RiemannSolverException)
    ST_NANFLUX = 2,  // NaN mass flux (FluxCalculationException)
    ST_ITERCAP = 4,  // iteration cap reached
    ST_UPDATEQ = 8,  // negative mass or energy after update (UpdateQException)
};

// counters accumulated by the batch kernels; the device array holds
// kCtrSlots copies (kCtrSlots x CNT_N) that blocks add into round-robin, so
// atomics from thousands of blocks do not queue on one address; readers sum
// the copies.
enum { CNT_NEVAL = 0, CNT_NBRENT, CNT_NVACUUM, CNT_NITER, CNT_NFAIL, CNT_N };
constexpr int kCtrSlots = 256;

// std::max / std::min as the reference's StateVector uses them
__device__ __forceinline__ double smax(double a, double b) { return (a < b) ? b : a; }
__device__ __forceinline__ double smin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ float smaxf(float a, float b) { return (a < b) ? b : a; }
__device__ __forceinline__ float sminf(float a, float b) { return (b < a) ? b : a; }

// The wave's sum of x, the same in every lane: a ballot and a population count
// per bit that some lane has set (the counters are 0, 1 or an iteration
// count), where six rounds of shuffles wait for each other.  With it and one
// barrier instead of two, the mixed exact faces of 250,000 3D cells went from
// 89 to 85 us, the 2D HLLC faces of 262,144 cells from 26 to 24.6 us and the
// 4M-problem batch from 96 to 92 us.
__device__ __forceinline__ unsigned long long wave_sum(unsigned x) {
    unsigned long long s = 0;
    for(int b = 0; __ballot(x != 0); b++, x >>= 1)
        s += (unsigned long long)__popcll(__ballot(x & 1u)) << b;
    return s;
}

// Adds per-lane counters v[0..CNT_N) over the whole block: wave sums, block
// sums in LDS, then one global atomic per counter into slot blockIdx.x %
// kCtrSlots.  Every thread of the block must call it (it synchronizes the
// block); ctr == nullptr is a uniform no-op.
__device__ __forceinline__ void block_add_counters(unsigned long long* ctr,
                                                   const unsigned (&v)[CNT_N]) {
    if(!ctr) return;
    __shared__ unsigned long long s_ctr[16][CNT_N];
    unsigned long long w[CNT_N];
#pragma unroll
    for(int k = 0; k < CNT_N; k++) w[k] = wave_sum(v[k]);
    if((threadIdx.x & 63) == 0) {
#pragma unroll
        for(int k = 0; k < CNT_N; k++) s_ctr[threadIdx.x >> 6][k] = w[k];
    }
    __syncthreads();
    if(threadIdx.x < CNT_N) {
        unsigned long long s = 0;
        for(unsigned q = 0; q < (blockDim.x + 63) / 64; q++) s += s_ctr[q][threadIdx.x];
        if(s) atomicAdd(ctr + (blockIdx.x % kCtrSlots) * CNT_N + threadIdx.x, s);
    }
}

// One counter that is zero nearly always: the waves that have some add it.
__device__ __forceinline__ void wave_add_counter(unsigned long long* ctr, int k, unsigned v) {
    if(!ctr || !__ballot(v != 0)) return;
    const unsigned long long s = wave_sum(v);
    if(__lane_id() == __ffsll(__ballot(true)) - 1)
        atomicAdd(ctr + (blockIdx.x % kCtrSlots) * CNT_N + k, s);
}

// One lane's counters, to slot 0.
__device__ __forceinline__ void lane_add_counters(unsigned long long* ctr,
                                                  const unsigned (&v)[CNT_N]) {
    if(!ctr) return;
#pragma unroll
    for(int k = 0; k < CNT_N; k++)
        if(v[k]) atomicAdd(ctr + k, (unsigned long long)v[k]);
}

// Workgroups are dispatched to the 8 XCDs of an MI355X round-robin
// (dispatch index b runs on XCD b % 8) and every XCD has its own L2.  This
// maps the dispatch index to a logical block index such that each XCD works
// through one contiguous range of blocks: kernels whose neighbouring items
// share data (cells and the faces between them) then find it in their own
// L2.  A bijection on [0, gridDim.x) for any grid size.
__device__ __forceinline__ int64_t xcd_block() {
    const int64_t nb = gridDim.x, b = blockIdx.x;
    const int64_t q = nb >> 3, r = nb & 7, x = b & 7, t = b >> 3;
    return x * q + (x < r ? x : r) + t;
}

}  // namespace sfx
