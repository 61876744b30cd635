// launch_batch_resident.hip -- launcher of the whole-integration kernel of a batch.
#include "launch.hpp"

namespace hrw {
namespace {

template <int FLUX, int R> hipError_t run(long long blocks, const BatchResArgs &a, hipStream_t s)
{
    return launch_kernel(batch_resident_kernel<FLUX, R>, (unsigned)blocks, 64 * kBatchResWaves,
                         res_lds_bytes<R>(kBatchResWaves), s, a);
}

template <int FLUX> hipError_t run_r(int r, long long blocks, const BatchResArgs &a, hipStream_t s)
{
    return r == 2 ? run<FLUX, 2>(blocks, a, s) : r == 4 ? run<FLUX, 4>(blocks, a, s) : run<FLUX, 5>(blocks, a, s);
}

}  // namespace

hipError_t launch_batch_resident(int flux, int r, long long blocks, const BatchResArgs &a, hipStream_t s)
{
    return flux == LF ? run_r<LF>(r, blocks, a, s) : run_r<GODUNOV>(r, blocks, a, s);
}

hipError_t launch_batch_recover(int flux, int lines, const BatchRecoverArgs &a, hipStream_t s)
{
    return flux == LF ? launch_kernel(batch_recover_kernel<LF>, lines, kResThreads, 0, s, a)
                      : launch_kernel(batch_recover_kernel<GODUNOV>, lines, kResThreads, 0, s, a);
}

}  // namespace hrw
