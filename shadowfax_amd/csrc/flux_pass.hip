// flux_pass.hip -- FP64 parity instantiation of the flux-pass kernels
// (flux_pass_impl.h), compiled with -ffp-contract=off so every expression
// keeps the reference's association.
#include "flux_pass_impl.h"
#include "sfx_launch.h"

namespace sfx {

static inline dim3 grid_for(int64_t n, int bs) { return dim3((unsigned)((n + bs - 1) / bs)); }

template <>
hipError_t launch_entry_geometry<double>(int ndim, const flux::MeshView<double>& m, int64_t E,
                                     double* egeo, hipStream_t s) {
    if(m.egrp) {
        // grouped layout: a block per group of 64 cells (the last one padded)
        if(m.C <= 0) return hipSuccess;
        const dim3 g((unsigned)((m.C + 63) / 64));  // one block per group
        const unsigned egeo_lds = flux::occupancy_lds_bytes(SFX_EGEO_WAVES, m.C, SFX_BIG_MESH, 1024);
        if(ndim == 3)
            hipLaunchKernelGGL((flux::entry_geometry_grouped_kernel<3, double>), g, dim3(256), egeo_lds,
                               s, m, egeo);
        else
            hipLaunchKernelGGL((flux::entry_geometry_grouped_kernel<2, double>), g, dim3(256), egeo_lds,
                               s, m, egeo);
        return hipGetLastError();
    }
    if(E <= 0) return hipSuccess;
    if(ndim == 3)
        hipLaunchKernelGGL((flux::entry_geometry_kernel<3, double>), grid_for(E, 256), dim3(256), 0,
                           s, m, E, egeo);
    else
        hipLaunchKernelGGL((flux::entry_geometry_kernel<2, double>), grid_for(E, 256), dim3(256), 0,
                           s, m, E, egeo);
    return hipGetLastError();
}

template <>
hipError_t launch_gradients<double>(int ndim, const flux::MeshView<double>& m, double* grad,
                                    hipStream_t s) {
    if(m.C <= 0) return hipSuccess;
    if(ndim == 3)
        hipLaunchKernelGGL((flux::gradient_kernel<3, double, double, false>), grid_for(m.C, 256),
                           dim3(256), 0, s, m, grad);
    else
        hipLaunchKernelGGL((flux::gradient_kernel<2, double, double, false>), grid_for(m.C, 256),
                           dim3(256), 0, s, m, grad);
    return hipGetLastError();
}

template <>
hipError_t launch_face_fluxes<double>(int ndim, int kind, const flux::MeshView<double>& m,
                                      const double* grad, const Consts& c, double* dQL,
                                      uint8_t* fstatus, unsigned long long* ctr,
                                      hipStream_t s) {
    if(m.F <= 0) return hipSuccess;
    const mixed::CF cf = mixed::make_cf(c);
    auto face = [&](auto nd, auto k) {
        constexpr int ND = decltype(nd)::value, K = decltype(k)::value;
        with_root<K == 0>(c, [&](auto root) {
            hipLaunchKernelGGL((flux::face_flux_kernel<ND, K, 0, double, double, false,
                                                       decltype(root)::value>),
                               grid_for(m.F, 256), dim3(256), 0, s, m, grad, c, cf, dQL, fstatus,
                               ctr);
        });
    };
    const std::integral_constant<int, 0> exact;
    const std::integral_constant<int, 1> hllc;
    const std::integral_constant<int, 2> d2;
    const std::integral_constant<int, 3> d3;
    if(ndim == 3) kind == 0 ? face(d3, exact) : face(d3, hllc);
    else kind == 0 ? face(d2, exact) : face(d2, hllc);
    return hipGetLastError();
}

hipError_t launch_gather_fp64(int ndim, int64_t C, const int64_t* goff,
                              const int32_t* gent, const double* dQL, double* dQ,
                              hipStream_t s) {
    if(C <= 0) return hipSuccess;
    flux::gather_shape<double>(ndim, [&](auto shape) {
        using S = decltype(shape);
        hipLaunchKernelGGL((flux::gather_kernel<S::ND, double, S::CELLS, S::NT, S::KPT, S::ROWS, S::U>),
                           dim3((unsigned)((C + S::CELLS - 1) / S::CELLS)), dim3(S::NT), 0, s, C, goff,
                           gent, dQL, dQ);
    });
    return hipGetLastError();
}

hipError_t launch_update(int ndim, const Consts& c, int64_t C, double* Q, double* dQ,
                         const double* volume, double* W, const uint64_t* endtime,
                         uint64_t tnow, uint8_t* cstatus, double* mass,
                         unsigned long long* ctr, hipStream_t s) {
    if(C <= 0) return hipSuccess;
    if(ndim == 3)
        hipLaunchKernelGGL((flux::update_kernel<3>), grid_for(C, 256), dim3(256), 0, s, c, C, Q,
                           dQ, volume, W, endtime, tnow, cstatus, mass, ctr);
    else
        hipLaunchKernelGGL((flux::update_kernel<2>), grid_for(C, 256), dim3(256), 0, s, c, C, Q,
                           dQ, volume, W, endtime, tnow, cstatus, mass, ctr);
    return hipGetLastError();
}

}  // namespace sfx
