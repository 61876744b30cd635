// launch_resident.hip -- launcher of the whole-integration kernel for one WENO order, HRW_K (the
// build compiles this file once per K = 1, 2, 3).
#include "launch.hpp"

#ifndef HRW_K
#error "compile with -DHRW_K=1, 2 or 3"
#endif

namespace hrw {
namespace {

template <int FLUX, bool FAST, bool CNU, int R, bool REC>
hipError_t run(const ResPlan &pl, const ResArgs &a, hipStream_t s)
{
    const size_t lds = res_lds_bytes<R>(pl.waves);
    if (pl.blocks == 1)
        return launch_kernel(resident_kernel<HRW_K, FLUX, FAST, CNU, R, true, REC>, 1, 64 * pl.waves, lds, s, a, pl.waves);
    return launch_kernel(resident_kernel<HRW_K, FLUX, FAST, CNU, R, false, REC>, pl.blocks,
                         64 * (pl.waves + (a.amax ? 1 : 0)), lds, s, a, pl.waves);
}
template <int FLUX, bool FAST, bool REC>
hipError_t run_r(const ResPlan &pl, const ResArgs &a, hipStream_t s)
{
    if (pl.r == 1) return run<FLUX, FAST, false, 1, REC>(pl, a, s);
    if (pl.r == 2) return run<FLUX, FAST, false, 2, REC>(pl, a, s);
    if (pl.r == 4) return run<FLUX, FAST, false, 4, REC>(pl, a, s);
    if constexpr (FAST) {
        if (pl.r == 5) return run<FLUX, FAST, false, 5, REC>(pl, a, s);
        return run<FLUX, FAST, false, 8, REC>(pl, a, s);
    }
    return hipErrorInvalidValue;
}
template <int FLUX, bool FAST>
hipError_t run_form(const ResPlan &pl, const ResArgs &a, hipStream_t s)
{
    if (a.tape) return a.cnu ? hipErrorInvalidValue : run_r<FLUX, FAST, true>(pl, a, s);
    return a.cnu ? run<FLUX, FAST, true, 1, false>(pl, a, s) : run_r<FLUX, FAST, false>(pl, a, s);
}

}  // namespace

#define HRW_CAT2(a, b) a##b
#define HRW_CAT(a, b) HRW_CAT2(a, b)
hipError_t HRW_CAT(launch_resident_k, HRW_K)(int flux, bool fast, const ResPlan &pl, const ResArgs &a,
                                             hipStream_t s)
{
    if (flux == LF) return fast ? run_form<LF, true>(pl, a, s) : run_form<LF, false>(pl, a, s);
    return fast ? run_form<GODUNOV, true>(pl, a, s) : run_form<GODUNOV, false>(pl, a, s);
}

}  // namespace hrw
