// ensemble_queue_launch.h -- the launch of the persistent serving kernel,
// shared by ensemble_queue_fp64.hip and ensemble_queue_mixed.hip.
#pragma once

#include <algorithm>

#include "ensemble_impl.h"
#include "ensemble_queue.h"

namespace sfx {

template <typename T, int MIXED>
hipError_t ens_queue_impl(int ndim, int kind, const EnsArgs<T>& a, const QueueArgs& qa, int ncu,
                          hipStream_t s, int* blocks) {
    mixed::CF cf = mixed::make_cf(a.c);
    const void* fn = nullptr;
    if(kind != 0)
        fn = ndim == 3 ? (const void*)ens::queue_kernel<3, 1, MIXED, T, double, 0>
                       : (const void*)ens::queue_kernel<2, 1, MIXED, T, double, 0>;
    else
        with_root<true>(a.c, [&](auto root) {
            constexpr int ROOT = decltype(root)::value;
            fn = ndim == 3 ? (const void*)ens::queue_kernel<3, 0, MIXED, T, double, ROOT>
                           : (const void*)ens::queue_kernel<2, 0, MIXED, T, double, ROOT>;
        });
    const size_t shmem = 4 * (size_t)qa.nmesh_words;
    int per_cu = 0;
    hipError_t err = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, a.block, shmem);
    if(err != hipSuccess) return err;
    if(per_cu < 1) return hipErrorInvalidConfiguration;
    // no more blocks than the kernel is compiled for, although some variants'
    // registers leave room: the barriers between the phases cost with every
    // block (FP64 HLLC, 16 2D meshes of 4,900 cells served: 67 us a request
    // with 3 blocks of 256 a CU, 42 with 2)
    const int waves = ndim == 3 ? ens::queue_waves<3>() : ens::queue_waves<2>();
    per_cu = std::min(per_cu, std::max(1, waves * 256 / a.block));
    *blocks = per_cu * ncu;
    EnsArgs<T> aa = a;
    QueueArgs q = qa;
    void* args[] = {&aa,          &cf,        &q.q,           &q.box,         &q.box_mesh,
                    &q.box_done,  &q.mc0,     &q.mnc,         &q.mf0,         &q.mnf,
                    &q.arena_cells, &q.arena_faces, &q.nmesh_words};
    return hipLaunchCooperativeKernel(fn, dim3((unsigned)*blocks), dim3((unsigned)a.block), args,
                                      (unsigned)shmem, s);
}

}  // namespace sfx
