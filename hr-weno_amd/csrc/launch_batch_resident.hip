// launch_batch_resident.hip -- launcher of the whole-integration kernel of a batch.
#include "launch.hpp"

namespace hrw {
namespace {

template <int FLUX, int R> hipError_t run(long long blocks, const BatchResArgs &a, hipStream_t s)
{
    batch_resident_kernel<FLUX, R>
        <<<(unsigned)blocks, 64 * kBatchResWaves, res_lds_bytes<R>(kBatchResWaves), s>>>(a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_batch_resident(int flux, int r, long long blocks, const BatchResArgs &a, hipStream_t s)
{
    if (flux == LF) return r == 2 ? run<LF, 2>(blocks, a, s) : run<LF, 4>(blocks, a, s);
    return r == 2 ? run<GODUNOV, 2>(blocks, a, s) : run<GODUNOV, 4>(blocks, a, s);
}

}  // namespace hrw
