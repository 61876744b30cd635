// kernels_resident.hpp -- a whole rktvd integration of one 1D Burgers line in one launch.
//
// A line that fits on the chip spends its time, with one launch per stage, on the launches: a
// stage of 1000 cells takes 5 us of which its arithmetic is a few hundred ns.  Here the state stays
// in LDS and registers for every step of the call (src/hrweno_tvdode.f90:136-171): block b owns M
// consecutive cells, its lanes R consecutive cells each, and a stage reads the block's LDS copy of
// the stage input and writes the other copy.  One block needs nothing else.  Several blocks (at
// most one per CU, so that all come to be resident) exchange, after each step, the cells at each of
// their ends that the next step's stages reach (three per stage) with their neighbours, and after
// each stage the block maxima of |u| (alpha = max|u|) with every block.  Within a step they compute
// the cells past their ends that the later stages need themselves: the same values as their owners',
// operation for operation.  A block may store its result over the input only once its neighbours have
// loaded their halo cells from it: they have when it has read their words, of the second step's cells
// or of the first maximum (resident_rules.hpp: a launch of one step without maxima is never in place).
//
// An exchange takes 1.4 us between neighbours and 1.6 / 1.7 / 2.3 us among 64 / 128 / 256 blocks
// (each block's words on a cache line of their own; packed, writers and readers of one line queue
// up: 2.3 / 2.7 / 3.1).  What does not wait for it runs beside it: the reconstruction of a stage
// needs no alpha, so one wavefront more per block sees to the maxima while the others reconstruct,
// and only the wavefronts that read a halo wait for the neighbours' cells, once a step.
//
// The exchange takes no fence.  A double travels as two 64-bit words, each half of it beside the
// 32-bit number of the exchange; a maximum (a non-negative double) as one word with a bit of the
// number in place of its sign.  All are stored and loaded with relaxed agent-scope atomics, so a
// word that carries the expected number carries its data.  Words of exchange e live in buffer
// e % 4.  A block publishes e + 4 behind the barrier that follows its reads of e + 2; its
// neighbours (for the maxima, every block) published those behind a barrier that follows their
// reads of e: no word is overwritten before it is read.  Numbers go on from launch to launch.  A
// wait is bounded; a wave that runs out of polls sets a status word and waits no more, so every
// launch ends.  The blocks have saved the initial state by then, and the caller goes on from it
// with one launch per stage.
//
// Per cell the arithmetic is that of the per-stage kernels, operation for operation
// (kernels_1d_fast.hpp for the FAST form, weno_math.hpp for EXACT), so the results are theirs bit
// for bit whatever the split into blocks and lanes.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels_1d_fast.hpp"
#include "resident_rules.hpp"

namespace hrw {

constexpr int kResHalo = 3;        // cells a stage reaches past each end (a face needs K = 3 each side)
constexpr int kResEdge = 9;        // cells exchanged at each end at most (the three stages of a step)
constexpr int kResMaxBlocks = 256;
// words per block and exchange: the maximum on a cache line of its own (read by every block), from
// word 16 on the first and the last kResEdge cells
constexpr int kResLine = 64;
constexpr int kResThreads = 1024;
constexpr size_t kResWords = 4 * (size_t)kResMaxBlocks * kResLine;   // one object's exchange words

// A launch's status: two words that the host has cleared, set by plain stores (they lie in host
// memory, as a rule).
enum { RES_NONFINITE = 0, RES_TIMEOUT = 1 };
__device__ __forceinline__ void set_status(unsigned long long *status, int which)
{
    __hip_atomic_store(status + which, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A stage's combination of u0 (the state at the start of the step), its input us and L = rhs(us):
// FAST  fma(C, L, fma(A, us - u0, u0))                        (kernels_1d_fast.hpp)
// EXACT ((p u0 + s us) + g L) q, or the division by 3         (stage_update; p, s, q exact factors)
// In a first stage u0 is us itself (A = 1; p = 0, s = 1).
struct ResCoef {
    double A, C, p, s, g, q;
    int div3;
};
__host__ __device__ inline ResCoef res_coef(int stage, double h)
{
    const StageCoef c = stage_coef(stage, h);
    const double post = c.div3 ? 1.0 / 3.0 : c.post;
    ResCoef r{c.A * post, c.C * post, 0.0, 1.0, h, 1.0, 0};
    if (stage == RK2_2) r.p = 1.0, r.q = 0.5;
    if (stage == RK3_2) r.p = 3.0, r.q = 0.25;
    if (stage == RK3_3) r.p = 1.0, r.s = 2.0, r.g = 2.0 * h, r.div3 = 1;
    return r;
}

struct ResArgs {
    const double *in;              // initial state
    double *saved;                 // receives the initial state, or nullptr
    long long n;
    int M;                         // cells per block (the last block: what is left, >= kResEdge)
    int order, nsteps, periodic, amax;
    double eps, alpha, xmin, rx;
    ResCoef coef[3];               // of the step's stages
    const double *width, *cnu;     // non-uniform grid, else nullptr
    unsigned long long *words;     // kResWords words
    unsigned long long *status;
    unsigned tag;                  // number of the first exchange (>= kResFirstTag)
    int polls;
    double *out;                   // final state (may be in: resident_in_place)
    // recording: the output of stage q, but the last, at tape + q*tape_stride, and the alpha of
    // stage q at alpha_rec[q]; or nullptr
    double *tape, *alpha_rec;
    long long tape_stride;
};

// A block's part of a line: cells [base, base + m) of n, and whom it exchanges with.
struct ResPart {
    const double *in;              // the line
    double *out, *saved, *tape, *alpha_rec;   // as in ResArgs
    long long tape_stride;
    long long n, base;
    int m, order, nsteps;
    bool per, amax;
    double eps, alpha, xmin, rx;
    const double *width, *cnu;
    unsigned long long *words;     // lines of kResLine words, words_per per buffer
    unsigned words_per;
    int self, left, right;         // the block's line, its neighbours' (-1: an end of the line)
    int g0, group;                 // the line's blocks: lines [g0, g0 + group)
    unsigned tag;
    int polls;
    unsigned long long *status;    // (of one block: or nullptr)
};

__device__ __forceinline__ unsigned long long word_load(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void word_store(unsigned long long *p, unsigned long long w)
{
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// cell_index in 32 bits (a line here has fewer than 2^31 cells, and i lies near it).
__device__ __forceinline__ int line_cell(long long i, long long n, bool periodic)
{
    const int j = (int)i, c = (int)n;
    if (j >= 0 && j < c) return j;
    if (!periodic) return j < 0 ? 0 : c - 1;
    const int r = j % c;
    return r < 0 ? r + c : r;
}

// The words of exchange `tag`; block b's line starts at word b*kResLine.
__device__ __forceinline__ unsigned long long *res_words(const ResPart &a, unsigned tag)
{
    return a.words + (tag & 3) * (size_t)a.words_per;
}
__device__ __forceinline__ unsigned long long tag_phase(unsigned tag)   // in a maximum's sign bit
{
    return (unsigned long long)((tag >> 2) & 1) << 63;
}

// v_max_f64 (a quiet NaN gives the other operand), and the maximum over each row of 16 lanes into its
// lane 15 (non-negative values; a lane with no source keeps its own).
__device__ __forceinline__ double max_f64(double x, double y)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
template <int CTRL> __device__ __forceinline__ double dpp_own(double v)
{
    return __builtin_bit_cast(double, dpp_u64<CTRL, 0xF>(__builtin_bit_cast(unsigned long long, v)));
}
__device__ __forceinline__ double row_max(double v)
{
    v = max_f64(v, dpp_own<0x111>(v));
    v = max_f64(v, dpp_own<0x112>(v));
    v = max_f64(v, dpp_own<0x114>(v));
    return max_f64(v, dpp_own<0x118>(v));
}

// *p = max(*p, v) in LDS for the lanes at work, completed (v non-negative, compared as bits; the
// compiler would walk the lanes one by one first).
__device__ __forceinline__ void lds_max(unsigned long long *p, double v)
{
    const unsigned at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned long long *)p;
    asm volatile("ds_max_u64 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"(at), "v"(v) : "memory");
}

// Face values vl, vr of a lane's R cells from their window v (cells -(K-1) .. R+K-2).  FAST: the
// scaled forms of chunk_stage; CNU: each cell's own coefficients ci.
template <int K, bool FAST, bool CNU, int R>
__device__ __forceinline__ void lane_recon(const double *v, double eps, const double *ci, double *vl,
                                           double *vr)
{
    if constexpr (CNU) {
#pragma unroll
        for (int t = 0; t < R; ++t) weno_cell_exact<K>(v + t, eps, ci + t * (K * (K + 1)), vl[t], vr[t]);
    } else if constexpr (K == 3) {
        Tri3 t2 = FAST ? tri3(v[0], v[1], v[2]) : tri3_exact(v[0], v[1], v[2]);
        Tri3 t1 = FAST ? tri3(v[1], v[2], v[3]) : tri3_exact(v[1], v[2], v[3]);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const Tri3 t0 = FAST ? tri3(v[t + 2], v[t + 3], v[t + 4]) : tri3_exact(v[t + 2], v[t + 3], v[t + 4]);
            if constexpr (FAST) recon3<true, true>(12.0 * eps, t2, t1, t0, vl[t], vr[t]);
            else recon3_exact(eps, t2, t1, t0, vl[t], vr[t]);
            t2 = t1;
            t1 = t0;
        }
    } else if constexpr (K == 2) {
        Pair2 p1 = FAST ? pair2(v[0], v[1]) : pair2_exact(v[0], v[1]);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const Pair2 p0 = FAST ? pair2(v[t + 1], v[t + 2]) : pair2_exact(v[t + 1], v[t + 2]);
            if constexpr (FAST) recon2<true>(eps, p1, p0, vl[t], vr[t]);
            else recon2_exact(eps, p1, p0, vl[t], vr[t]);
            p1 = p0;
        }
    } else {
#pragma unroll
        for (int t = 0; t < R; ++t) vl[t] = vr[t] = FAST ? v[t] : 0.0 + v[t];
    }
}

template <int K, int FLUX, bool FAST, bool CNU>
__device__ __forceinline__ double face_flux(double vm, double vp, double alpha)
{
    if constexpr (CNU || !FAST) {
        return burgers_numflux<FLUX, FAST>(vm, vp, alpha);
    } else {
        constexpr double S = K == 3 ? 6.0 : (K == 2 ? 2.0 : 1.0);
        const double cq = 0.25 / (S * S), ca = (-0.5 / S) * alpha, cg = 0.5 / (S * S);
        if constexpr (FLUX == GODUNOV) return godunov((vm * vm) * cg, (vp * vp) * cg, vm, vp);
        else return fma_(cq, fma_(vm, vm, vp * vp), ca * (vp - vm));
    }
}

// The extra wavefront's part of an exchange: publishes the block's maximum and waits for every
// block's of the line (at most GROUP); false when the polls ran out.
template <int GROUP>
__device__ __forceinline__ bool gather_max(const ResPart &a, unsigned tag, int polls, unsigned long long mine,
                                           double *line_max)
{
    constexpr int N = GROUP / 64;
    const int lane = threadIdx.x & 63, B = a.group;
    const unsigned long long ph = tag_phase(tag);
    unsigned long long *all = res_words(a, tag);
    if (lane == 0) word_store(all + a.self * kResLine, mine | ph);
    const unsigned long long *words = all + a.g0 * kResLine;
    for (int q = 0; q < polls; ++q) {
        unsigned long long w[N], miss = 0;
#pragma unroll
        for (int i = 0; i < N; ++i)   // (lanes past the last block read its word)
            w[i] = i == 0 || 64 * i < B ? word_load(words + min(64 * i + lane, B - 1) * kResLine) : ph;
        double x = 0.0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            w[i] ^= ph;
            miss |= w[i];
            x = max_f64(x, __builtin_bit_cast(double, w[i]));
        }
        if (!__any((long long)miss < 0)) {
            *line_max = __builtin_bit_cast(double, wave_umax(__builtin_bit_cast(unsigned long long, x)));
            return true;
        }
    }
    return false;
}

// A wavefront that reads a halo waits for the neighbours' end cells, `width` of them each, and puts
// them around buf: word 2e + half of the left neighbour's last cells by lanes 0 .. 2 width - 1, of
// the right one's first cells by as many lanes from 32 on.  An end of the line repeats its end cell
// (src/hrweno_weno.f90:171-173).  False when the polls ran out (the halo is NaN then).
__device__ __forceinline__ bool gather_halo(const ResPart &a, unsigned tag, int polls, int width, double *buf, bool lo,
                                            bool hi)
{
    const int lane = threadIdx.x & 63, m = a.m, w = lane & 31;
    const bool left = lane < 32, use = w < 2 * width && (left ? lo : hi);
    const int nb = left ? a.left : a.right;
    const bool wait = use && nb >= 0;
    // (a block's words: its first cells, then its last ones)
    const unsigned long long *p =
        res_words(a, tag) + (wait ? nb * kResLine + 16 + (left ? 2 * (kResEdge + kResEdge - width) : 0) + w : 0);
    unsigned long long x = 0;
    bool ok = false;
    for (int q = 0; q < polls; ++q) {
        if (wait) x = word_load(p);
        if (__all(!wait || (unsigned)x == tag)) {
            ok = true;
            break;
        }
    }
    const unsigned half = (unsigned)(x >> 32);
    const unsigned other = (unsigned)__builtin_amdgcn_update_dpp(0, (int)half, 0xB1, 0xF, 0xF, true);   // lane ^ 1
    if (use && !(lane & 1)) {
        double c = __builtin_bit_cast(double, ((unsigned long long)other << 32) | half);
        if (nb < 0) c = buf[left ? 0 : m - 1];
        else if (!ok) c = __builtin_nan("");
        buf[(left ? -width : m) + (w >> 1)] = c;
    }
    return ok;
}

// LDS: two copies of the block's cells with kResPad cells on each side (the halo, and room for what
// the wave-edge lanes read beyond it, which feeds no cell), and after each copy one cell more that
// takes the writes of cells the block does not keep.
template <int R> constexpr int kResPad = R + kResEdge + 1;
// Cells past each end that a block of several computes in a step's first stage.
__host__ __device__ constexpr int res_extra(int order) { return kResHalo * (order - 1); }
template <int R> __host__ __device__ constexpr int res_copy(int waves) { return waves * kOutLanes * R + 2 * kResPad<R> + 2; }
template <int R> constexpr size_t res_lds_bytes(int waves) { return 2 * (size_t)res_copy<R>(waves) * sizeof(double); }

// The block's part: `waves` wavefronts that own cells; with ONE false and alpha = max|u| one more
// takes part, and `threads` counts them all.  lds, s_mx (4 words) and s_alpha: the block's LDS.  A
// wait in vain leaves NaN behind, and the wavefront waits no more.  REC: the stages and their alphas are
// recorded.  SCAN: a result that is not finite is reported.
constexpr int kInVain = -1;
template <int K, int FLUX, bool FAST, bool CNU, int R, bool ONE, int GROUP, bool REC, bool SCAN>
__device__ __forceinline__ void resident_part(const ResPart &a, const ResCoef *coef, int waves, int threads,
                                              double *lds, unsigned long long *s_mx, double *s_alpha)
{
    constexpr int H = K - 1, PAD = kResPad<R>;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cap = waves * kOutLanes * R, copy = res_copy<R>(waves);
    double *cur = lds + PAD, *nxt = cur + copy;
    const long long base = a.base;
    const int m = a.m;
    const int extra = ONE ? 0 : res_extra(a.order), width = extra + kResHalo;
    const int w0 = wv * kOutLanes * R - extra, c0 = w0 + (lane - 1) * R;   // the lane's first cell in the block
    const bool owned = lane >= 1 && lane <= kOutLanes;
    const bool amax = FLUX == LF && a.amax, per = a.per;
    const bool comm = !ONE && wv >= waves;   // the extra wavefront
    const bool tiny = ONE && per && m < 2 * kResHalo + 2;   // a cell has several images past the ends

    // the initial state and its halo, R + 1 loads in flight per thread; what the copies hold beyond
    // feeds no cell (EXACT: zero, so that no lane takes the divides over it)
    if (!FAST || CNU)
        for (int j = tid; j < 2 * copy; j += threads) lds[j] = 0.0;
    if (tid < 4) s_mx[tid] = 0ull;
    __syncthreads();
    double x0 = 0.0;
    for (int j0 = tid - width; j0 < m + width; j0 += (R + 1) * threads) {
        double x[R + 1];
#pragma unroll
        for (int i = 0; i <= R; ++i) {
            const int j = j0 + i * threads;
            if (j < m + width) x[i] = a.in[line_cell(base + j, a.n, per)];
        }
#pragma unroll
        for (int i = 0; i <= R; ++i) {
            const int j = j0 + i * threads;
            if (j >= m + width) continue;
            cur[j] = x[i];
            if (j >= 0 && j < m) {
                // (a signalling NaN would take x0 with it: its own maximum is a quiet one)
                const double x1 = fabs(x[i]);
                x0 = max_f64(x0, max_f64(x1, x1));
                if (a.saved) a.saved[base + j] = x[i];
            }
        }
    }
    if (amax) {
        x0 = row_max(x0);
        if ((lane & 15) == 15) lds_max(&s_mx[0], x0);
    }

    // what does not change with the steps: cell widths (FAST: their reciprocals), the non-uniform
    // grid's coefficients, which cells are the block's, where the lane writes its cells (`spare`:
    // those it does not keep) and (the only block of a line) their images past its ends
    const int spare = cap + PAD;
    double wd[R];
    [[maybe_unused]] double ci[CNU ? R * K * (K + 1) : 1];
    bool mine[R];
    int at[R];
    [[maybe_unused]] int image[R];
    const double inv_rx = rcp_nr(a.rx);
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int j = c0 + t;
        const long long g = base + j;
        const int gc = line_cell(g, a.n, per);
        mine[t] = owned && j >= 0 && j < m;
        at[t] = owned && j >= -extra && j < m + extra && (per || (g >= 0 && g < a.n)) ? j : spare;
        image[t] = !mine[t] || tiny ? spare : (per ? (j < kResHalo ? m + j : (j >= m - kResHalo ? j - m : spare)) : spare);
        if constexpr (CNU) {
            wd[t] = a.width[gc];
#pragma unroll
            for (int q = 0; q < K * (K + 1); ++q) ci[t * K * (K + 1) + q] = a.cnu[(long long)gc * (K * (K + 1)) + q];
        } else {
            const double w = linear_edge(a.xmin, a.rx, gc + 1) - linear_edge(a.xmin, a.rx, gc);
            wd[t] = FAST ? fma_(inv_rx, fma_(-w, inv_rx, 1.0), inv_rx) : w;
        }
    }
    // zero-gradient ends (example1:103-104): the lane's cell that is cell 0, and cell n-1 (-1: none)
    const long long gf = -base - c0, gl = a.n - 1 - base - c0;
    const int first = !per && owned && gf >= 0 && gf < R ? (int)gf : -1;
    const int last = !per && owned && gl >= 0 && gl < R ? (int)gl : -1;
    // this wavefront owns end cells that are exchanged (or have images) / reads halo cells / holds
    // an end of the line
    const bool own_end = w0 < m && (wv == 0 || w0 + kOutLanes * R > m - width);
    const bool read_lo = wv == 0, read_hi = w0 + 63 * R + H > m;
    const bool line_end = __any(first >= 0 || last >= 0);

    const int stages = a.order * a.nsteps;
    double u0[R];
    double alpha = a.alpha;
    bool bad = false;
    int polls = a.polls, st = 0;   // stage of the step
    for (int q = 0;; ++q) {
        const unsigned tag = a.tag + (unsigned)q;
        __syncthreads();   // cur and its maximum are complete
        if (amax && tid == 0) s_mx[(q + 2) & 3] = 0ull;
        if (tiny) {
            if (tid < 2 * kResHalo) {
                const int j = tid < kResHalo ? tid - kResHalo : m + tid - kResHalo;
                cur[j] = cur[line_cell(j, m, true)];
            }
            __syncthreads();
        }
        if (REC && !comm && q > 0) {   // (from the LDS copy: whole lines of memory at a time)
            double *y = a.tape + (long long)(q - 1) * a.tape_stride + base;
            for (int j = tid; j < m; j += 64 * waves) y[j] = cur[j];
        }
        double v[R + 2 * H], vl[R], vr[R], vr_left = 0.0, vl_right = 0.0;
        if (!comm) {
            if constexpr (!ONE) {
                if (st == 0 && q > 0 && (read_lo || read_hi)) {
                    // (these wavefronts first: theirs is the longer way)
                    __builtin_amdgcn_s_setprio(2);
                    if (!gather_halo(a, tag, polls, width, cur, read_lo, read_hi)) {
                        polls = SCAN ? 1 : kInVain;
                        if (SCAN && a.status && lane == 0) set_status(a.status, RES_TIMEOUT);
                    }
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_s_setprio(0);
                }
            }
#pragma unroll
            for (int t = 0; t < R + 2 * H; ++t) v[t] = cur[c0 - H + t];
            if (ONE && amax) alpha = __builtin_bit_cast(double, s_mx[q & 3]);
            lane_recon<K, FAST, CNU, R>(v, a.eps, ci, vl, vr);
            vr_left = shfl_up1(vr[R - 1]);
            vl_right = shfl_down1(vl[0]);
        } else {
            double x = __builtin_nan("");
            if (!gather_max<GROUP>(a, tag, polls, s_mx[q & 3], &x)) {
                polls = SCAN ? 1 : kInVain;
                if (SCAN && a.status && lane == 0) set_status(a.status, RES_TIMEOUT);
            }
            if (lane == 0) *s_alpha = x;
        }
        if (!ONE && amax) {
            __syncthreads();   // the line's maximum is known
            alpha = *s_alpha;
        }
        if (comm) {
            if (q + 1 == stages) break;
            continue;
        }
        if (REC && amax && base == 0 && tid == 0) a.alpha_rec[q] = alpha;
        double f[R + 1], un[R];
        f[0] = face_flux<K, FLUX, FAST, CNU>(vr_left, vl[0], alpha);
#pragma unroll
        for (int t = 1; t < R; ++t) f[t] = face_flux<K, FLUX, FAST, CNU>(vr[t - 1], vl[t], alpha);
        f[R] = face_flux<K, FLUX, FAST, CNU>(vr[R - 1], vl_right, alpha);
        if (line_end) {
#pragma unroll
            for (int t = 0; t < R; ++t)
                if (t == first) f[t] = f[t + 1];
#pragma unroll
            for (int t = 0; t < R; ++t)
                if (t == last) f[t + 1] = f[t];
        }
        const ResCoef &co = coef[st];
        if (st == 0) {
#pragma unroll
            for (int t = 0; t < R; ++t) u0[t] = v[H + t];
        }
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const double us = v[H + t];
            if constexpr (!CNU && FAST) {
                const double L = (f[t] - f[t + 1]) * wd[t];
                un[t] = fma_(co.C, L, fma_(co.A, us - u0[t], u0[t]));
            } else {
                const double L = (f[t] - f[t + 1]) / wd[t];
                if constexpr (FAST) un[t] = fma_(co.g, L, fma_(co.p, u0[t], co.s * us));
                else un[t] = (co.p * u0[t] + co.s * us) + co.g * L;
            }
        }
        if constexpr (CNU || !FAST) {
            if (co.div3) {
#pragma unroll
                for (int t = 0; t < R; ++t) un[t] = FAST ? div3_fast(un[t]) : un[t] / 3;
            } else {
#pragma unroll
                for (int t = 0; t < R; ++t) un[t] = un[t] * co.q;
            }
        }
        if (q + 1 == stages) {
#pragma unroll
            for (int t = 0; t < R; ++t)
                if (mine[t]) {
                    a.out[base + c0 + t] = un[t];
                    bad |= SCAN && !isfinite(un[t]);
                }
            break;
        }
#pragma unroll
        for (int t = 0; t < R; ++t) nxt[at[t]] = un[t];
        if (line_end) {   // the line's ends repeat their end cells (src/hrweno_weno.f90:171-173)
#pragma unroll
            for (int t = 0; t < R; ++t) {
                if (t == first) nxt[-1] = nxt[-2] = nxt[-3] = un[t];
                if (t == last) nxt[m] = nxt[m + 1] = nxt[m + 2] = un[t];
            }
        }
        if constexpr (ONE) {
            if (own_end && per) {
#pragma unroll
                for (int t = 0; t < R; ++t) nxt[image[t]] = un[t];
            }
        } else if (own_end && st + 1 == a.order) {
            // words for the neighbours' next step
            unsigned long long *line = res_words(a, tag + 1) + a.self * kResLine + 16;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const int j = c0 + t;
                const unsigned long long bits = __builtin_bit_cast(unsigned long long, un[t]);
                const unsigned long long wl = (bits << 32) | (tag + 1);
                const unsigned long long wh = (bits & 0xffffffff00000000ull) | (tag + 1);
                if (mine[t] && j < width) {
                    word_store(line + 2 * j, wl);
                    word_store(line + 2 * j + 1, wh);
                }
                if (mine[t] && j >= m - width) {
                    unsigned long long *e = line + 2 * (j - m + 2 * kResEdge);
                    word_store(e, wl);
                    word_store(e + 1, wh);
                }
            }
        }
        if (amax) {
            double x = 0.0;
#pragma unroll
            for (int t = 0; t < R; ++t) x = max_f64(x, mine[t] ? fabs(un[t]) : 0.0);
            x = row_max(x);
            if ((lane & 15) == 15) lds_max(&s_mx[(q + 1) & 3], x);
        }
        double *sw = cur;
        cur = nxt;
        nxt = sw;
        if (++st == a.order) st = 0;
    }
    if (!ONE && !SCAN && polls == kInVain && lane == 0) set_status(a.status, RES_TIMEOUT);
    if (SCAN && a.status && __any(bad) && lane == 0) set_status(a.status, RES_NONFINITE);
}

// One line over the whole grid.
// (R = 8: three wavefronts per SIMD and 168 VGPRs.  Spilled VGPRs over several blocks, K = 3: 8-19 of
// them there, 4-12 at R = 5, EXACT 11-21 at R = 4; a recording has the larger numbers.)
template <int K, int FLUX, bool FAST, bool CNU, int R, bool ONE, bool REC>
__global__ __launch_bounds__(R == 8 ? 768 : kResThreads) void resident_kernel(ResArgs a, int waves)
{
    extern __shared__ double lds[];
    __shared__ unsigned long long s_mx[4];   // block maxima of |u|, in turn
    __shared__ double s_alpha;
    const int b = blockIdx.x, B = gridDim.x;
    ResPart p;
    p.in = a.in;
    p.out = a.out;
    p.saved = a.saved;
    if constexpr (REC) {
        p.tape = a.tape;
        p.tape_stride = a.tape_stride;
        p.alpha_rec = a.alpha_rec;
    }
    p.n = a.n;
    p.base = (long long)b * a.M;
    p.m = (int)min((long long)a.M, a.n - p.base);
    p.order = a.order;
    p.nsteps = a.nsteps;
    p.per = a.periodic != 0;
    p.amax = a.amax != 0;
    p.eps = a.eps;
    p.alpha = a.alpha;
    p.xmin = a.xmin;
    p.rx = a.rx;
    p.width = a.width;
    p.cnu = a.cnu;
    p.words = a.words;
    p.words_per = kResMaxBlocks * kResLine;
    p.self = b;
    p.left = b > 0 ? b - 1 : (p.per ? B - 1 : -1);
    p.right = b + 1 < B ? b + 1 : (p.per ? 0 : -1);
    p.g0 = 0;
    p.group = B;
    p.tag = a.tag;
    p.polls = a.polls;
    p.status = a.status;
    resident_part<K, FLUX, FAST, CNU, R, ONE, kResMaxBlocks, REC, true>(p, a.coef, waves, blockDim.x, lds, s_mx, &s_alpha);
}

// ---- an ensemble of periodic lines (kernels_1d_fast.hpp's batch), each on a block or a few ----
// Block i of the table works on cells [base, base + m) of one line for nsteps RK3 steps: 16 bytes
// of memory traffic per cell and launch instead of 64 per cell and step.  The blocks of one line
// are neighbours in the table, and a block takes the table entry of its turn to start, so at any
// time at most one line has some of its blocks waiting for others that have not started: the lines
// ahead of it run to their ends and make room.  Two blocks of eight wavefronts share a CU; one
// computes while the other waits for its exchange.
//
// Other kernels of the device can still keep a line's blocks off it for longer than a wait lasts.
// Nobody reads a result on the host, so what waited in vain is made good in the stream: a line of
// several blocks saves its initial state (8 bytes per cell and launch) and a wait in vain marks it;
// batch_recover_kernel, launched behind, computes the marked lines anew, each in one block.
constexpr int kBatchResWaves = 8;
struct ResBlock {
    long long off;                      // the line's first cell in the flat state
    int line, n, k, base, m;            // the line, its length and order; this block's cells
    int g0, group;                      // the line's blocks [g0, g0 + group)
    int mark;                           // of a line of several blocks: its number among those
    double h, xmin, rx;
};
struct BatchResArgs {
    double *u;
    const ResBlock *blocks;
    unsigned *ticket;                   // starts counted so far
    unsigned ticket0;                   // ... before this launch
    int nsteps, amax, polls;
    double eps, alpha;
    unsigned long long *words;
    unsigned words_per, tag;
    double *saved;                      // receives the initial state of the lines of several blocks
    unsigned long long *status;         // two status words for each of them
};

template <int FLUX, int R>
__global__ __launch_bounds__(64 * kBatchResWaves) __attribute__((amdgpu_waves_per_eu(4))) void batch_resident_kernel(
    BatchResArgs a)
{
    extern __shared__ double lds[];
    __shared__ unsigned long long s_mx[4];
    __shared__ double s_alpha;
    __shared__ ResCoef s_coef[3];
    __shared__ unsigned s_turn;
    const int wv = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_turn = atomicAdd(a.ticket, 1u) - a.ticket0;
    __syncthreads();
    const int turn = __builtin_amdgcn_readfirstlane((int)s_turn);
    const ResBlock &b = a.blocks[turn];
    const int waves = (b.m + (b.group > 1 ? 2 * res_extra(3) : 0) + kOutLanes * R - 1) / (kOutLanes * R);
    const int threads = 64 * (waves + (b.group > 1 && a.amax ? 1 : 0));
    if (threadIdx.x < 3) s_coef[threadIdx.x] = res_coef(RK3_1 + (int)threadIdx.x, b.h);
    if (64 * wv >= threads) return;   // (whole wavefronts; a barrier counts those that are left)
    ResPart p;
    p.in = p.out = a.u + b.off;
    p.saved = b.group > 1 ? a.saved + b.off : nullptr;
    p.n = b.n;
    p.base = b.base;
    p.m = b.m;
    p.order = 3;
    p.nsteps = a.nsteps;
    p.per = true;
    p.amax = a.amax != 0;
    p.eps = a.eps;
    p.alpha = a.alpha;
    p.xmin = b.xmin;
    p.rx = b.rx;
    p.width = p.cnu = nullptr;
    p.words = a.words;
    p.words_per = a.words_per;
    p.self = turn;
    p.left = b.base > 0 ? turn - 1 : b.g0 + b.group - 1;
    p.right = b.base + b.m < b.n ? turn + 1 : b.g0;
    p.g0 = b.g0;
    p.group = b.group;
    p.tag = a.tag;
    p.polls = a.polls;
    p.status = b.group > 1 ? a.status + 2 * b.mark : nullptr;
#define HRW_RES_PART(K)                                                                                       \
    if (b.group == 1)                                                                                         \
        resident_part<K, FLUX, true, false, R, true, kBatchResGroup, false, false>(p, s_coef, waves, threads, lds, s_mx, &s_alpha); \
    else                                                                                                      \
        resident_part<K, FLUX, true, false, R, false, kBatchResGroup, false, false>(p, s_coef, waves, threads, lds, s_mx, &s_alpha)
    if (b.k == 3) {
        HRW_RES_PART(3);
    } else if (b.k == 2) {
        HRW_RES_PART(2);
    } else {
        HRW_RES_PART(1);
    }
#undef HRW_RES_PART
}

// A marked line anew from its saved state, one block per line of several, through memory: per cell
// the operations of resident_part, so the results are the same.  (It returns at once as a rule; a
// marked line takes one block's time.)
struct BatchRecoverArgs {
    double *u, *y1, *y2;                // the state; stage results (y1 holds the saved states first)
    const ResBlock *blocks;
    const int *first;                   // a line's first block in the table
    unsigned long long *status;
    int nsteps, amax;
    double eps, alpha;
};
template <int K, int FLUX>
__device__ __forceinline__ void recover_stage(const ResBlock &b, const BatchRecoverArgs &a, const ResCoef &co, const double *us,
                                              const double *u0, double *out, double *s_red)
{
    constexpr int H = K - 1;
    const int tid = threadIdx.x, n = b.n;
    double alpha = a.alpha;
    if (FLUX == LF && a.amax) {
        double m = 0.0;
        for (int i = tid; i < n; i += kResThreads) m = fmax(m, fabs(us[i]));
        m = __builtin_bit_cast(double, wave_umax(__builtin_bit_cast(unsigned long long, m)));
        if ((tid & 63) == 0) s_red[tid >> 6] = m;
        __syncthreads();
        alpha = 0.0;
        for (int w = 0; w < kResThreads / 64; ++w) alpha = fmax(alpha, s_red[w]);
    }
    const double inv_rx = rcp_nr(b.rx);
    for (int i = tid; i < n; i += kResThreads) {
        double v[2 * H + 3], vl[3], vr[3];   // cells i-1-H .. i+1+H; reconstructions of i-1, i, i+1
#pragma unroll
        for (int t = 0; t < 2 * H + 3; ++t) v[t] = us[line_cell(i - 1 - H + t, n, true)];
        lane_recon<K, true, false, 3>(v, a.eps, nullptr, vl, vr);
        const double f0 = face_flux<K, FLUX, true, false>(vr[0], vl[1], alpha);
        const double f1 = face_flux<K, FLUX, true, false>(vr[1], vl[2], alpha);
        const double w = linear_edge(b.xmin, b.rx, i + 1) - linear_edge(b.xmin, b.rx, i);
        const double L = (f0 - f1) * fma_(inv_rx, fma_(-w, inv_rx, 1.0), inv_rx), x0 = u0[i];
        out[i] = fma_(co.C, L, fma_(co.A, v[H + 1] - x0, x0));
    }
    __syncthreads();
}
template <int K, int FLUX>
__device__ __forceinline__ void recover_line(const ResBlock &b, const BatchRecoverArgs &a, double *s_red)
{
    double *u = a.u + b.off, *y1 = a.y1 + b.off, *y2 = a.y2 + b.off;
    for (int i = threadIdx.x; i < b.n; i += kResThreads) u[i] = y1[i];
    __syncthreads();
    for (int q = 0; q < a.nsteps; ++q) {
        recover_stage<K, FLUX>(b, a, res_coef(RK3_1, b.h), u, u, y1, s_red);
        recover_stage<K, FLUX>(b, a, res_coef(RK3_2, b.h), y1, u, y2, s_red);
        recover_stage<K, FLUX>(b, a, res_coef(RK3_3, b.h), y2, u, u, s_red);
    }
}
template <int FLUX> __global__ __launch_bounds__(kResThreads) void batch_recover_kernel(BatchRecoverArgs a)
{
    __shared__ double s_red[kResThreads / 64];
    unsigned long long *mark = a.status + 2 * (size_t)blockIdx.x + RES_TIMEOUT;
    if (*mark == 0) return;
    const ResBlock &b = a.blocks[a.first[blockIdx.x]];
    if (b.k == 3) recover_line<3, FLUX>(b, a, s_red);
    else if (b.k == 2) recover_line<2, FLUX>(b, a, s_red);
    else recover_line<1, FLUX>(b, a, s_red);
    if (threadIdx.x == 0) *mark = 0;
}

}  // namespace hrw
