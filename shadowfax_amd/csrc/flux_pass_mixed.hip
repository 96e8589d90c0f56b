// flux_pass_mixed.hip -- mixed instantiation of the flux-pass kernels
// (flux_pass_impl.h): FP32 storage of generator velocities, gradients and
// face geometry (half the bytes of those gathers); the primitive states stay
// FP64 (a face flux driven by the small difference of two large pressures,
// as between the hot cells of a Sedov blast, cannot be recovered from
// FP32-rounded states: rounding the states alone gave 6e-6 face errors);
// gradient estimation (in the closure-free difference form), limiting and
// the MUSCL-Hancock predictor evaluated in FP64 registers; the mixed Riemann
// solvers (riemann_mixed_impl.h); face fluxes dt A F formed in FP64 and
// stored in FP32 (a 6e-8 relative rounding per face; each stored value
// enters its two cells with opposite signs); FP64 accumulation.  Each
// periodic boundary face is evaluated once and applied with opposite signs
// to its two cells, so mass, momentum and energy are conserved to FP64
// round-off (the reference evaluates both copies, src/VorFace.cpp:913-948).
#include "flux_pass_impl.h"
#include "sfx_launch.h"

namespace sfx {

static inline dim3 grid_for(int64_t n, int bs) { return dim3((unsigned)((n + bs - 1) / bs)); }

template <>
hipError_t launch_entry_geometry<float>(int ndim, const flux::MeshView<float>& m, int64_t E,
                                     float* egeo, hipStream_t s) {
    if(m.egrp) {
        // grouped layout: a block per group of 64 cells (the last one padded)
        if(m.C <= 0) return hipSuccess;
        const dim3 g((unsigned)((m.C + 63) / 64));  // one block per group
        if(ndim == 3)
            hipLaunchKernelGGL((flux::entry_geometry_grouped_kernel<3, float>), g, dim3(256), 0, s, m,
                               egeo);
        else
            hipLaunchKernelGGL((flux::entry_geometry_grouped_kernel<2, float>), g, dim3(256), 0, s, m,
                               egeo);
        return hipGetLastError();
    }
    if(E <= 0) return hipSuccess;
    if(ndim == 3)
        hipLaunchKernelGGL((flux::entry_geometry_kernel<3, float>), grid_for(E, 256), dim3(256), 0,
                           s, m, E, egeo);
    else
        hipLaunchKernelGGL((flux::entry_geometry_kernel<2, float>), grid_for(E, 256), dim3(256), 0,
                           s, m, E, egeo);
    return hipGetLastError();
}

template <>
hipError_t launch_gradients<float>(int ndim, const flux::MeshView<float>& m, float* grad,
                                   hipStream_t s) {
    if(m.C <= 0) return hipSuccess;
    // the conditions under which gradient_kernel reads grouped records
    // through the buffer descriptor (rec_buffer)
    const bool buf = SFX_REC_BUFFER && m.egrp && m.egeo_bytes > 0 && m.egeo_bytes <= 0x7FFFFFF0ull;
    if(ndim == 3 && buf && SFX_GRAD_LDS_K > 0)
        hipLaunchKernelGGL((flux::gradient_lds_kernel<3>), grid_for(m.C, 256), dim3(256), 0, s, m,
                           grad);
    else if(ndim == 2 && buf && SFX_GRAD_LDS_K_2D > 0)
        hipLaunchKernelGGL((flux::gradient_lds_kernel<2>), grid_for(m.C, 256), dim3(256), 0, s, m,
                           grad);
    else if(ndim == 3)
        hipLaunchKernelGGL((flux::gradient_kernel<3, float, double, true>), grid_for(m.C, 256),
                           dim3(256), 0, s, m, grad);
    else
        hipLaunchKernelGGL((flux::gradient_kernel<2, float, double, true>), grid_for(m.C, 256),
                           dim3(256), 0, s, m, grad);
    return hipGetLastError();
}

template <>
hipError_t launch_face_fluxes<float>(int ndim, int kind, const flux::MeshView<float>& m,
                                     const float* grad, const Consts& c, float* dQL,
                                     uint8_t* fstatus, unsigned long long* ctr, hipStream_t s) {
    if(m.F <= 0) return hipSuccess;
    const mixed::CF cf = mixed::make_cf(c);
    // with the per-face records, the variant that reads them
    auto face = [&](auto nd, auto k) {
        constexpr int ND = decltype(nd)::value, K = decltype(k)::value;
        with_root<K == 0>(c, [&](auto root) {
            constexpr int ROOT = decltype(root)::value;
            if(m.frec)
                hipLaunchKernelGGL((flux::face_flux_kernel<ND, K, 1, float, double, true, ROOT>),
                                   grid_for(m.F, 256), dim3(256), 0, s, m, grad, c, cf, dQL,
                                   fstatus, ctr);
            else
                hipLaunchKernelGGL((flux::face_flux_kernel<ND, K, 1, float, double, false, ROOT>),
                                   grid_for(m.F, 256), dim3(256), 0, s, m, grad, c, cf, dQL,
                                   fstatus, ctr);
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

hipError_t launch_face_records(int ndim, const flux::MeshView<float>& m, float* frec,
                               hipStream_t s) {
    if(m.F <= 0) return hipSuccess;
    float4* out = reinterpret_cast<float4*>(frec);
    if(ndim == 3)
        hipLaunchKernelGGL((flux::face_record_kernel<3>), grid_for(m.F, 256), dim3(256), 0, s, m,
                           out);
    else
        hipLaunchKernelGGL((flux::face_record_kernel<2>), grid_for(m.F, 256), dim3(256), 0, s, m,
                           out);
    return hipGetLastError();
}

hipError_t launch_gather_mixed(int ndim, int64_t C, const int64_t* goff,
                               const int32_t* gent, const float* dQL, double* dQ, hipStream_t s) {
    if(C <= 0) return hipSuccess;
    flux::gather_shape<float>(ndim, [&](auto shape) {
        using S = decltype(shape);
        hipLaunchKernelGGL((flux::gather_kernel<S::ND, float, S::CELLS, S::NT, S::KPT, S::ROWS, S::U>),
                           dim3((unsigned)((C + S::CELLS - 1) / S::CELLS)), dim3(S::NT), 0, s, C, goff,
                           gent, dQL, dQ);
    });
    return hipGetLastError();
}


}  // namespace sfx
