// launch_adjoint_resident.hip -- launcher of the whole-integration reverse kernel.
#include "launch.hpp"

namespace hrw {
namespace {

template <int K, bool LFP, int FLUX, bool AMAX>
hipError_t run(const AresPlan &pl, const AresArgs &a, hipStream_t s)
{
    if (pl.chunks <= 4)
        return launch_kernel(adjoint_resident_kernel<K, LFP, FLUX, AMAX, 4>, pl.blocks, 64 * pl.chunks, pl.lds, s, a);
    return launch_kernel(adjoint_resident_kernel<K, LFP, FLUX, AMAX, 8>, pl.blocks, 64 * pl.chunks, pl.lds, s, a);
}
template <int K>
hipError_t run_k(bool lfp, int flux, bool amax, const AresPlan &pl, const AresArgs &a, hipStream_t s)
{
    if (lfp) return amax ? run<K, true, LF, true>(pl, a, s) : run<K, true, LF, false>(pl, a, s);
    if (flux == LF) return amax ? run<K, false, LF, true>(pl, a, s) : run<K, false, LF, false>(pl, a, s);
    return run<K, false, GODUNOV, false>(pl, a, s);
}

}  // namespace

hipError_t launch_adjoint_resident(int k, bool lfp, int flux, bool alphamax, const AresPlan &pl, const AresArgs &a,
                                   hipStream_t s)
{
    return k == 3 ? run_k<3>(lfp, flux, alphamax, pl, a, s) : run_k<2>(lfp, flux, alphamax, pl, a, s);
}

}  // namespace hrw
