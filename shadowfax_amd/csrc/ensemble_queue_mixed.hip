// ensemble_queue_mixed.hip -- the persistent serving kernel of the mixed ensembles,
// in a translation unit of its own (it is the longest to compile), with the
// flags of the standalone flux pass of that precision.
#include "ensemble_queue_launch.h"

namespace sfx {

template <>
hipError_t ens_launch_queue<float>(int ndim, int kind, const EnsArgs<float>& a, const QueueArgs& qa,
                                int ncu, hipStream_t s, int* blocks) {
    return ens_queue_impl<float, 1>(ndim, kind, a, qa, ncu, s, blocks);
}


}  // namespace sfx
