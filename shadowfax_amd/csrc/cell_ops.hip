// cell_ops.hip -- per-cell RiemannSolver operations over batches (FP64,
// contraction off, the reference's association): get_time_derivative,
// get_W, get_Q, and TimeLine::calculate_timestep.  Solver batches are
// component-major SoA: W, Q [ndim+2][N], grad [ndim][ndim+2][N]; the time
// step reads the mesh arrays, cell-major.
#include "flux_pass_impl.h"
#include "sfx_launch.h"
#include "shadowfax_amd.h"

namespace sfx {
namespace {

template <int ND>
__global__ __launch_bounds__(256) void time_derivative_kernel(double gamma, int64_t N,
                                                              const double* __restrict__ W,
                                                              const double* __restrict__ grad,
                                                              double* __restrict__ out) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= N) return;
    double w[NC], g[ND][NC], d[NC];
#pragma unroll
    for(int k = 0; k < NC; k++) w[k] = W[k * N + i];
#pragma unroll
    for(int l = 0; l < ND; l++)
#pragma unroll
        for(int k = 0; k < NC; k++) g[l][k] = grad[(l * NC + k) * N + i];
    flux::time_derivative<ND, double>(gamma, w, g, d);
#pragma unroll
    for(int k = 0; k < NC; k++) out[k * N + i] = d[k];
}

template <int ND>
__global__ __launch_bounds__(256) void get_W_kernel(double gamma, int64_t N,
                                                    const double* __restrict__ V,
                                                    double* __restrict__ Q,
                                                    double* __restrict__ W) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= N) return;
    double q[NC], w[NC];
#pragma unroll
    for(int k = 0; k < NC; k++) q[k] = Q[k * N + i];
    flux::get_W_state<ND>(gamma, V[i], q, w);
#pragma unroll
    for(int k = 0; k < NC; k++) {
        Q[k * N + i] = q[k];
        W[k * N + i] = w[k];
    }
}

template <int ND, int KIND>
__global__ __launch_bounds__(256) void get_Q_kernel(double gamma, int64_t N,
                                                    const double* __restrict__ V,
                                                    const double* __restrict__ W,
                                                    double* __restrict__ Q) {
    const int NC = ND + 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= N) return;
    double q[NC], w[NC];
#pragma unroll
    for(int k = 0; k < NC; k++) w[k] = W[k * N + i];
    flux::get_Q_state<ND, KIND>(gamma, V[i], w, q);
#pragma unroll
    for(int k = 0; k < NC; k++) Q[k * N + i] = q[k];
}

inline dim3 blocks(int64_t N) { return dim3((unsigned)((N + 255) / 256)); }

// TimeLine::get_realtime / get_realtime_interval (src/TimeLine.hpp:145-166),
// no cosmology
__device__ __forceinline__ double tl_realtime(const TimelineArgs& tl, uint64_t t) {
    double x = (double)t / (double)tl.integer_maxtime;
    return tl.tottime * x + tl.mintime;
}
__device__ __forceinline__ double tl_interval(const TimelineArgs& tl, uint64_t t) {
    double x = (double)t / (double)tl.integer_maxtime;
    return tl.tottime * x;
}

__global__ void timestep_init_kernel(uint64_t* result, uint64_t smax) {
    if(threadIdx.x == 0) {
        result[0] = smax;
        result[1] = 0;
    }
}

// The reference's step search, `S2 = M; while(interval(S2) > S) S2 >>= 1`,
// started near its end: the interval falls with every halving, so where
// interval(M >> k) > S still holds at the k that the exponents of tottime and
// S give (less 2), it held at every earlier one.  0 when no step is left.
__device__ __forceinline__ uint64_t tl_largest_step(const TimelineArgs& tl, double S) {
    uint64_t s2 = tl.integer_maxtime;
    const int k = __builtin_amdgcn_frexp_exp(tl.tottime) - __builtin_amdgcn_frexp_exp(S) - 2;
    if(k > 0 && k < 64) {
        const uint64_t near = s2 >> k;
        if(tl_interval(tl, near) > S) s2 = near;
    }
    while(s2 && tl_interval(tl, s2) > S) s2 >>= 1;  // at most 64 halvings
    return s2;
}
// `while(left % S2) S2 >>= 1`: the largest halving of S2 that divides what is
// left of the time line.  For a power of two that is left's lowest set bit.
__device__ __forceinline__ uint64_t tl_synchronise(uint64_t left, uint64_t s2) {
    if((s2 & (s2 - 1)) == 0) {
        const uint64_t low = left & (0 - left);
        return (low != 0 && low < s2) ? low : s2;
    }
    while(left % s2) s2 >>= 1;  // S2 = 1 divides everything: at most 64 halvings
    return s2;
}

// kTsCells cells a thread, 256 apart: one atomic a block and result then
// stands for 1,024 cells (blocks of 256 cells put 8,192 atomics a result on
// one address for 2,097,152 cells).
constexpr int kTsCells = 4;

// TimeLine::calculate_timestep's gas loop (src/TimeLine.cpp:248-320).  The
// smallest step and the active count go to result through one atomic each per
// block.  Bound by the cells' bytes (106 in 3D) and, for the cells whose step
// starts now, cbrt and two square roots; 2,097,152 3D cells with individual
// steps took 198 us when each active lane halved its way down from the whole
// time line (a division a halving, a 64-bit remainder after) and take
// 67 us (43 at copy rate).
template <int ND, int KIND>
__global__ __launch_bounds__(256) void timestep_kernel(
        TimelineArgs tl, double gamma, int64_t C, const double* __restrict__ W,
        const double* __restrict__ vel, const double* __restrict__ volume,
        uint64_t* __restrict__ starttime, uint64_t* __restrict__ endtime, double* __restrict__ dt,
        uint8_t* __restrict__ active, uint64_t* __restrict__ result, uint8_t* __restrict__ status) {
    constexpr int NC = ND + 2, P = ND + 1;
    __shared__ uint64_t s_min[4];
    __shared__ unsigned s_cnt[4];
    const uint64_t Smax = tl.max_timestep;
    uint64_t mine = Smax;
    unsigned count = 0;
    const int64_t i0 = (int64_t)blockIdx.x * (256 * kTsCells) + threadIdx.x;
    uint64_t ends[kTsCells];
#pragma unroll
    for(int u = 0; u < kTsCells; u++) {
        const int64_t i = i0 + u * 256;
        ends[u] = i < C ? endtime[i] : 0;
    }
#pragma unroll
    for(int u = 0; u < kTsCells; u++) {
        const int64_t i = i0 + u * 256;
        if(i >= C) break;
        uint8_t st = 0;
        const uint64_t end0 = ends[u];
        uint64_t start1 = 0, end1 = end0;
        const bool act = end0 == tl.current_time + tl.timestep;
        active[i] = act ? 1 : 0;
        if(act) {
            count++;
            const double* w = W + i * NC;
            // v = W.v - particle velocity; Vec::norm (src/Vec.hpp:140,378)
            const double vx = w[1] - vel[i * ND], vy = w[2] - vel[i * ND + 1];
            double vi;
            if(ND == 3) {
                const double vz = w[3] - vel[i * ND + 2];
                vi = sqrt(vx * vx + vy * vy + vz * vz);
            } else {
                vi = sqrt(vx * vx + vy * vy);
            }
            // get_soundspeed: the exact solver guards rho = 0, HLLC does not
            const double ci = (KIND == 0 && !(w[0] != 0.)) ? 0. : sqrt(gamma * w[P] / w[0]);
            // VorCell::set_h (src/VorCell.cpp:930-938)
            const double V = volume[i];
            const double pi = 3.14159265358979323846;
            const double h = (ND == 3) ? cbrt(V * 3. / 4. / pi) : sqrt(V / pi);
            const double S = tl.cfl * (h / (vi + ci));
            uint64_t S2;
            if(tl_interval(tl, Smax) < S) {
                S2 = Smax;
            } else {
                S2 = tl_largest_step(tl, S);
                if(!S2) {
                    st = SFX_ST_TIMESTEP;
                } else {
                    S2 = tl_synchronise(tl.integer_maxtime - end0, S2);
                    S2 = (S2 < tl.min_timestep) ? tl.min_timestep : S2;
                    S2 = (S2 > tl.max_timestep) ? tl.max_timestep : S2;
                }
            }
            if(!st) {
                mine = S2 < mine ? S2 : mine;
                start1 = end0;
                end1 = end0 + S2;
                if(!tl.global_timestep) {
                    starttime[i] = start1;
                    endtime[i] = end1;
                }
            }
        }
        if(status) status[i] = st;
        if(!tl.global_timestep) {
            if(!act || st) start1 = starttime[i];
            dt[i] = tl_realtime(tl, end1 - start1);
        }
    }
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) {
        const uint64_t o = __shfl_xor(mine, off, 64);
        mine = o < mine ? o : mine;
        count += __shfl_xor(count, off, 64);
    }
    if((threadIdx.x & 63) == 0) {
        s_min[threadIdx.x >> 6] = mine;
        s_cnt[threadIdx.x >> 6] = count;
    }
    __syncthreads();
    if(threadIdx.x == 0) {
#pragma unroll
        for(int q = 1; q < 4; q++) {
            mine = s_min[q] < mine ? s_min[q] : mine;
            count += s_cnt[q];
        }
        if(mine < Smax) atomicMin((unsigned long long*)result, (unsigned long long)mine);
        if(count) atomicAdd((unsigned long long*)(result + 1), (unsigned long long)count);
    }
}

// global time step (src/TimeLine.cpp:418-431): every cell takes the system step
__global__ __launch_bounds__(256) void timestep_global_kernel(
        TimelineArgs tl, int64_t C, const uint64_t* __restrict__ result,
        uint64_t* __restrict__ starttime, uint64_t* __restrict__ endtime, double* __restrict__ dt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= C) return;
    const uint64_t S = result[0];
    const uint64_t e = endtime[i];
    starttime[i] = e;
    endtime[i] = e + S;
    dt[i] = tl_realtime(tl, S);
}

}  // namespace

hipError_t launch_hydro_timestep(int kind, int ndim, double gamma, int64_t C,
                                 const TimelineArgs& tl, const double* W, const double* vel,
                                 const double* volume, uint64_t* starttime, uint64_t* endtime,
                                 double* dt, uint8_t* active, uint64_t* result,
                                 uint8_t* status, hipStream_t s) {
    hipLaunchKernelGGL(timestep_init_kernel, dim3(1), dim3(64), 0, s, result, tl.max_timestep);
    if(C > 0) {
#define SFX_TS(ND, K)                                                                       \
    hipLaunchKernelGGL((timestep_kernel<ND, K>),                                              \
                       dim3((unsigned)((C + 256 * kTsCells - 1) / (256 * kTsCells))), dim3(256), 0, \
                       s, tl, gamma, C, W,                                                  \
                       vel, volume, starttime, endtime, dt, active, result, status)
        if(ndim == 3) {
            if(kind == 1)
                SFX_TS(3, 1);
            else
                SFX_TS(3, 0);
        } else {
            if(kind == 1)
                SFX_TS(2, 1);
            else
                SFX_TS(2, 0);
        }
#undef SFX_TS
        if(tl.global_timestep)
            hipLaunchKernelGGL(timestep_global_kernel, blocks(C), dim3(256), 0, s, tl, C, result,
                               starttime, endtime, dt);
    }
    return hipGetLastError();
}

hipError_t launch_cell_op(int op, int kind, int ndim, double gamma, int64_t N,
                          const double* a, const double* b, double* c, double* d,
                          hipStream_t s) {
    if(N <= 0) return hipSuccess;
    switch(op) {
        case 0:  // time derivative: a = W, b = grad, c = out
            if(ndim == 3)
                hipLaunchKernelGGL(time_derivative_kernel<3>, blocks(N), dim3(256), 0, s, gamma,
                                   N, a, b, c);
            else
                hipLaunchKernelGGL(time_derivative_kernel<2>, blocks(N), dim3(256), 0, s, gamma,
                                   N, a, b, c);
            break;
        case 1:  // get_W: a = V, d = Q (in/out), c = W
            if(ndim == 3)
                hipLaunchKernelGGL(get_W_kernel<3>, blocks(N), dim3(256), 0, s, gamma, N, a, d, c);
            else
                hipLaunchKernelGGL(get_W_kernel<2>, blocks(N), dim3(256), 0, s, gamma, N, a, d, c);
            break;
        default:  // get_Q: a = V, b = W, c = Q
            if(ndim == 3) {
                if(kind == 1)
                    hipLaunchKernelGGL((get_Q_kernel<3, 1>), blocks(N), dim3(256), 0, s, gamma,
                                       N, a, b, c);
                else
                    hipLaunchKernelGGL((get_Q_kernel<3, 0>), blocks(N), dim3(256), 0, s, gamma,
                                       N, a, b, c);
            } else {
                if(kind == 1)
                    hipLaunchKernelGGL((get_Q_kernel<2, 1>), blocks(N), dim3(256), 0, s, gamma,
                                       N, a, b, c);
                else
                    hipLaunchKernelGGL((get_Q_kernel<2, 0>), blocks(N), dim3(256), 0, s, gamma,
                                       N, a, b, c);
            }
    }
    return hipGetLastError();
}

}  // namespace sfx
