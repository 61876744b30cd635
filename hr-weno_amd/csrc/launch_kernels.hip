// launch_kernels.hip -- launchers of the LDS-tile 1D stage, the 2D stage and the batch stage.
#include "launch.hpp"

namespace hrw {
namespace {

constexpr int kCPT = 4;   // cells per thread in the 1D stage kernel

template <int K, int FLUX, bool PER, bool FAST, bool AMAX>
static void l1d(const Stage1DArgs &a, hipStream_t s)
{
    constexpr int TILE = kBlock * kCPT - 2;
    const unsigned grid = (unsigned)((a.n + TILE - 1) / TILE);
    stage1d_kernel<K, FLUX, PER, FAST, AMAX, kCPT><<<grid, kBlock, 0, s>>>(a);
}
template <int K, int FLUX, bool PER, bool FAST>
static void l1d_a(bool amax, const Stage1DArgs &a, hipStream_t s)
{
    if constexpr (FLUX == LF) {
        if (amax) return l1d<K, FLUX, PER, FAST, true>(a, s);
    }
    l1d<K, FLUX, PER, FAST, false>(a, s);
}
template <int K, int FLUX, bool PER>
static void l1d_f(bool fast, bool amax, const Stage1DArgs &a, hipStream_t s)
{
    if (fast) l1d_a<K, FLUX, PER, true>(amax, a, s);
    else l1d_a<K, FLUX, PER, false>(amax, a, s);
}
template <int K, int FLUX>
static void l1d_p(bool per, bool fast, bool amax, const Stage1DArgs &a, hipStream_t s)
{
    if (per) l1d_f<K, FLUX, true>(fast, amax, a, s);
    else l1d_f<K, FLUX, false>(fast, amax, a, s);
}
template <int K>
static void l1d_x(int flux, bool per, bool fast, bool amax, const Stage1DArgs &a, hipStream_t s)
{
    if (flux == LF) l1d_p<K, LF>(per, fast, amax, a, s);
    else l1d_p<K, GODUNOV>(per, fast, amax, a, s);
}
// Rows per wavefront of an untuned 2D launch.  A wavefront takes about ty + 1.5 row times (its
// prologue reconstructs two rows); with w wavefronts on a SIMD a row takes 1, 1.4, 2, 2.7 times what
// it takes alone (0.6 us FAST, 1.05 us EXACT: latency, then FP64 issue), and wavefronts past the
// resident ones run in further turns.  The ty with the least (ty + 1.5) * that is taken; measured us
// per stage with 8 rows at least, and so: 250 x 250 FAST 8.7, 5.1, EXACT 12.3, 6.2; 500 x 500 FAST
// 9.1, 6.8; 1000 x 1000 FAST 15.1, 12.2, EXACT 23.9, 19.1; 2048 x 2048 as before (18 rows).
static int rows_per_wave(int n2, int nstrips, int resident)
{
    const long long simds = 4LL * device_cus();
    auto slowdown = [](long long w) { return w <= 1 ? 1.0 : (w == 2 ? 1.4 : 2.0 + 0.67 * (double)(w - 3)); };
    int best = 1;
    double least = 1e300;
    for (int ty = 1; ty <= std::max(64, (int)(n2 * (long long)nstrips / (simds * resident)) + 1); ty = ty < 64 ? ty + 1 : ty + ty / 16) {
        const long long w = ((long long)nstrips * ((n2 + ty - 1) / ty) + simds - 1) / simds;   // per SIMD
        const double cost = (ty + 1.5) * ((double)(w / resident) * slowdown(resident) +
                                          (w % resident ? slowdown(w % resident) : 0.0));
        if (cost < least) {
            least = cost;
            best = ty;
        }
    }
    return best;
}
template <int K, int BC, bool FAST>
static void l2d(Stage2DArgs a, hipStream_t s)
{
    if (a.ty <= 0) {
        static int per_cu = 0;
        if (!per_cu) {
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pbe2d_kernel<K, BC, FAST>, kBlock, 0) !=
                    hipSuccess || per_cu <= 0)
                per_cu = 4;
        }
        a.ty = rows_per_wave(a.n2, a.nstrips, per_cu);
    }
    const long long nsy = (a.n2 + a.ty - 1) / a.ty;
    const long long waves = nsy * a.nstrips;
    const unsigned grid = (unsigned)((waves * 64 + kBlock - 1) / kBlock);
    pbe2d_kernel<K, BC, FAST><<<grid, kBlock, 0, s>>>(a);
}
template <int K>
static void l2d_b(int bc, bool fast, const Stage2DArgs &a, hipStream_t s)
{
    if (bc == HRW_BC_ZERO_FLUX) {
        if (fast) l2d<K, 0, true>(a, s);
        else l2d<K, 0, false>(a, s);
    } else {
        if (fast) l2d<K, 1, true>(a, s);
        else l2d<K, 1, false>(a, s);
    }
}
template <int FLUX, bool AMAX, int R>
static void lbatch_r(const BatchArgs &a, hipStream_t s)
{
    const unsigned grid = (unsigned)((a.nchunks * 64 + kBlock - 1) / kBlock);
    switch (stage_npw(a.stage)) {
    case 1: batch_stage_kernel<FLUX, AMAX, R, 1><<<grid, kBlock, 0, s>>>(a); break;
    default: batch_stage_kernel<FLUX, AMAX, R, 0><<<grid, kBlock, 0, s>>>(a); break;
    }
}
// Persistent form: as many blocks as fit on the device at once (occupancy of this
// instantiation, asked once), never more than there are chunks.
template <int FLUX, bool AMAX, int R, int NPW>
static void lbatch_pf_n(const BatchArgs &a, hipStream_t s)
{
    static int per_cu = 0;
    if (!per_cu) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &nb, reinterpret_cast<const void *>(&batch_pf_kernel<FLUX, AMAX, R, NPW>), kBlock, 0) != hipSuccess ||
            nb <= 0)
            nb = 2;
        per_cu = nb;
    }
    const long long want = (a.nchunks + kBlock / 64 - 1) / (kBlock / 64);
    const unsigned grid = (unsigned)std::max<long long>(1, std::min<long long>(want, (long long)per_cu * device_cus()));
    batch_pf_kernel<FLUX, AMAX, R, NPW><<<grid, kBlock, 0, s>>>(a);
}
template <int FLUX, bool AMAX, int R>
static void lbatch_pf_r(const BatchArgs &a, hipStream_t s)
{
    switch (stage_npw(a.stage)) {
    case 1: lbatch_pf_n<FLUX, AMAX, R, 1>(a, s); break;
    default: lbatch_pf_n<FLUX, AMAX, R, 0>(a, s); break;
    }
}
template <int FLUX, bool AMAX>
static void lbatch(int R, int form, const BatchArgs &a, hipStream_t s)
{
    if (form == HRW_BATCH_PERSISTENT) {
        if (R == 4) lbatch_pf_r<FLUX, AMAX, 4>(a, s);
        else if (R == 6) lbatch_pf_r<FLUX, AMAX, 6>(a, s);
        else lbatch_pf_r<FLUX, AMAX, 8>(a, s);
        return;
    }
    if (R == 4) lbatch_r<FLUX, AMAX, 4>(a, s);
    else if (R == 6) lbatch_r<FLUX, AMAX, 6>(a, s);
    else lbatch_r<FLUX, AMAX, 8>(a, s);
}

}  // namespace

void launch_tile_1d(int k, int flux, bool periodic, bool fast, bool alphamax, const Stage1DArgs &a,
                    hipStream_t s)
{
    if (k == 1) l1d_x<1>(flux, periodic, fast, alphamax, a, s);
    else if (k == 2) l1d_x<2>(flux, periodic, fast, alphamax, a, s);
    else l1d_x<3>(flux, periodic, fast, alphamax, a, s);
}

void launch_pbe2d(int k, int bc, bool fast, const Stage2DArgs &a, hipStream_t s)
{
    if (k == 1) l2d_b<1>(bc, fast, a, s);
    else if (k == 2) l2d_b<2>(bc, fast, a, s);
    else l2d_b<3>(bc, fast, a, s);
}

void launch_batch_stage(int flux, bool alphamax, int R, int form, const BatchArgs &a, hipStream_t s)
{
    if (flux == LF && alphamax) lbatch<LF, true>(R, form, a, s);
    else if (flux == LF) lbatch<LF, false>(R, form, a, s);
    else lbatch<GODUNOV, false>(R, form, a, s);
}

}  // namespace hrw
