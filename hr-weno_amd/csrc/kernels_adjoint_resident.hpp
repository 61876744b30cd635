// kernels_adjoint_resident.hpp -- the reverse of a whole recorded rktvd integration of one 1D
// Burgers line (K = 2, 3) in one launch.
//
// With one launch per reversed stage (kernels_adjoint.hpp, kernels_adjoint_blocked.hpp) a stage of
// a line of up to some 100,000 cells is bound by the launch and its chain of waits.  Here the
// cotangents stay in LDS for every stage of the call: block b owns M consecutive cells, each of its
// wavefronts one chunk of them, two cells per lane.  The stage inputs come from the recording, two
// stages ahead of their use.  What a stage needs of them alone (weights, faces and their
// derivatives: half of its work) is computed between the barrier that ends the stage before and
// the waits for other blocks, so those waits run beside it.  A chain of dependent FP64 operations
// at one or two wavefronts per SIMD bounds a stage (1.7 us with no exchange; 2.4 with the loads one
// stage ahead and the two parts in turn), and with several blocks the exchange (3.0 us instead of
// 3.8 Godunov, 4.8 instead of 5.3 Lax-Friedrichs; one launch per stage 4.8 and 7.7, 5000 cells).
//
// Blocks (at most one per CU, so that all come to be resident) exchange the three cells at each of
// their ends after every stage, in words that carry the number of the launch beside half a double
// (kernels_resident.hpp); each stage has words of its own, so none is overwritten.  A wavefront
// publishes an end cell as soon as it has it, and only the wavefronts that read a halo wait.
//
// alpha = max|s|: alpha-bar, a sum over the line, lands on the first cell attaining the maximum.
// Only the block that holds such a cell needs the sum: every block publishes its groups' shares and
// its first such cell behind the stage's barrier and goes on; that block waits for all of them,
// adds the correction to its copy and publishes the end cells it had held back.
//
// Per cell the arithmetic, and the order of alpha-bar's sum, are those of the launches per stage:
// chunk_adjoint and line_alpha_bar for periodic Lax-Friedrichs lines (chunks of 124 cells, lanes 0
// and 63 halo lanes), bvjp_chunk and rhs_vjp_alpha_fixup for the others (120 cells, two halo lanes
// on each side), so the gradients are theirs bit for bit.
//
// Waits are bounded as in resident_kernel; the caller then goes on from the saved cotangent with
// one launch per stage.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels_adjoint.hpp"
#include "kernels_adjoint_blocked.hpp"
#include "kernels_resident.hpp"

namespace hrw {

constexpr int kAresWaves = 8;      // chunks of a block at most
constexpr int kAresHalo = 3;       // cells a reversed stage reaches past each end
constexpr int kAresPad = 8;        // LDS cells on each side of a copy (the halo and what discarded lanes read)
constexpr int kAresLine = 16;      // words of a block and stage: two per end cell, then its first cell at the maximum
template <bool LFP> constexpr int kAresChunk = LFP ? 124 : 120;   // cells of a chunk

struct AresArgs {
    const double *x0;              // input of the first stage, of stage q > 0 at tape + (q-1)*tape_stride
    const double *tape, *alpha_rec;
    long long tape_stride;
    const double *g;               // the cotangent of the result
    double *out;                   // that of the initial state (may be g)
    double *saved;                 // receives g, or nullptr
    long long n;
    int M;                         // cells per block, a multiple of four chunks (the last: what is left, >= 3)
    int chunks;                    // = wavefronts of a block
    int order, nsteps, periodic, constw;
    double eps, alpha, xmin, rx, dt;
    unsigned long long *words;     // per stage: a line per block; behind them, two words per unit of alpha-bar's sum
    int units;                     // of the whole line
    unsigned long long *status;
    unsigned tag;                  // the launch's number (never 0)
    int polls;
};

// LDS in doubles: three copies of the block's cells, a block's shares of alpha-bar for two stages,
// the line's.
__host__ __device__ inline int ares_copy(int chunks, int chunk) { return chunks * chunk + 2 * kAresPad; }
__host__ __device__ inline size_t ares_lds_bytes(int chunks, int chunk, int units, bool amax)
{
    return (3 * (size_t)ares_copy(chunks, chunk) + (amax ? 2 * (size_t)chunks + (size_t)units : 0)) * sizeof(double);
}

// The stage (out = ca lam + cc h J^T lam + e1 x1 + e2 x2) reversed st-th in a step.
struct AresCoef {
    double ca, cc, e1, e2;
};
__device__ __forceinline__ AresCoef ares_coef(int order, int st)
{
    if (order == 3) {
        if (st == 0) return {2.0 / 3.0, 2.0 / 3.0, 0.0, 0.0};
        if (st == 1) return {0.25, 0.25, 0.0, 0.0};
        return {1.0, 1.0, 0.75, 1.0 / 3.0};
    }
    if (order == 2) {
        if (st == 0) return {0.5, 0.5, 0.0, 0.0};
        return {1.0, 1.0, 0.5, 0.0};
    }
    return {1.0, 1.0, 0.0, 0.0};
}

__device__ __forceinline__ void put_double(unsigned long long *p, double v, unsigned tag)
{
    const unsigned long long bits = __builtin_bit_cast(unsigned long long, v);
    word_store(p, (bits << 32) | tag);
    word_store(p + 1, (bits & 0xffffffff00000000ull) | tag);
}

// LFP: periodic Lax-Friedrichs lines; else FLUX with either kind of ends.
template <int K, bool LFP, int FLUX, bool AMAX, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void adjoint_resident_kernel(AresArgs a)
{
    constexpr int R = 2, H = K - 1, NV = R + 2 * H, HL = LFP ? 1 : 2, CH = kAresChunk<LFP>;
    constexpr int kNone = 0x7fffffff;
    extern __shared__ double lds[];
    __shared__ int s_peak[4];                // the block's first cell at the maximum, stages in turn: twice
                                             // the cell, and 1 if s is negative there
    __shared__ int s_held[4];                // end cells were held back
    __shared__ int s_first;                  // the line's first cell at the maximum
    const int tid = threadIdx.x, lane = tid & 63, c = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x, B = gridDim.x, threads = 64 * a.chunks;
    const bool per = LFP || a.periodic != 0;
    const int n = (int)a.n, base = b * a.M;
    const int m = b + 1 < B ? a.M : n - base;
    const int nch = (m + CH - 1) / CH, copy = ares_copy(a.chunks, CH);
    double *const L0 = lds + kAresPad;
    double *const part = lds + 3 * copy, *const sums = part + 2 * a.chunks;
    const int stages = a.order * a.nsteps;
    const size_t per_stage = (size_t)B * kAresLine + (AMAX ? 2 * (size_t)a.units : 0);
    int polls = a.polls;

    // the cotangent with its halo, and a copy of it for the caller
    for (int j = tid - kAresHalo; j < m + kAresHalo; j += threads) {
        const double x = a.g[line_cell(base + j, n, per)];
        L0[j] = x;
        if (a.saved && j >= 0 && j < m) a.saved[base + j] = x;
    }
    if (tid < 4) s_peak[tid] = kNone, s_held[tid] = 0;

    // what does not change with the stages: where the lane's window lies in a state (images or end
    // cells past the ends; positions that feed no cell get one in range), 1/width of its cells
    // (LFP: half of it), the halo it reads
    const bool work = c < nch;
    const int W = c * CH, c0 = W + (lane - HL) * R, g0 = base + c0;
    const bool owned = lane >= HL && lane < 64 - HL;
    auto cell_of = [&](int g) {
        if (per) g = g < 0 ? g + n : (g >= n ? g - n : g);
        return min(max(g, 0), n - 1);
    };
    auto inv_w = [&](int g) {
        double r;
        if (a.constw) {
            r = rcp_nr(a.rx);
        } else {
            const int i = cell_of(g);
            r = rcp_nr(linear_edge(a.xmin, a.rx, i + 1) - linear_edge(a.xmin, a.rx, i));
        }
        return LFP ? 0.5 * r : r;
    };
    int at[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) at[i] = cell_of(g0 - H + i);
    double iw[R];
#pragma unroll
    for (int t = 0; t < R; ++t) iw[t] = inv_w(g0 + t);
    const int hc = lane < 32 ? W - R - 1 : W + 63 * R;   // LFP: the cell beyond the wavefront's
    const double iw_edge = LFP ? inv_w(base + hc) : 0.0;
    const bool lo = c == 0, hi = W + CH + kAresHalo > m, halo = work && (lo || hi);
    // lanes 0..5 wait for the left neighbour's last cells, lanes 32..37 for the right one's first
    const int hw = lane & 31, left = b > 0 ? b - 1 : (per ? B - 1 : -1), right = b + 1 < B ? b + 1 : (per ? 0 : -1);
    const int nb = lane < 32 ? left : right;
    const bool wait = hw < 2 * kAresHalo && nb >= 0 && (lane < 32 ? lo : hi);
    const unsigned long long *const hp = a.words + (wait ? nb * kAresLine + (lane < 32 ? 2 * kAresHalo : 0) + hw : 0);

    auto load_window = [&](int e, double *v) {
        const int q = stages - 1 - e;
        const double *x = q ? a.tape + (long long)(q - 1) * a.tape_stride : a.x0;
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = x[at[i]];
    };
    // the part of a stage that its input gives: the cells' reconstructions, (not LFP) the flux's
    // derivatives at the lane's interfaces, |s| = alpha
    using Rev = std::conditional_t<K == 3, Weno5Rev, Weno3Rev>;
    Rev w[R];
    [[maybe_unused]] double dm[R + 1], dp[R + 1], da[R + 1];
    double alpha = a.alpha;
    int cand = kNone;
    bool peak[R] = {};
    auto window_part = [&](const double *v) {
        if constexpr (!LFP) {
            double vr[R], vl[R];
            if constexpr (K == 3) {
                Tri3 T[R + 2];
#pragma unroll
                for (int j = 0; j < R + 2; ++j) T[j] = tri3(v[j], v[j + 1], v[j + 2]);
#pragma unroll
                for (int t = 0; t < R; ++t) recon3<false, true>(12.0 * a.eps, T[t], T[t + 1], T[t + 2], vl[t], vr[t]);
            } else {
                Pair2 P[R + 1];
#pragma unroll
                for (int j = 0; j < R + 1; ++j) P[j] = pair2(v[j], v[j + 1]);
#pragma unroll
                for (int t = 0; t < R; ++t) recon2(a.eps, P[t], P[t + 1], vl[t], vr[t]);
            }
            const double vr_prev = shfl_up1(vr[R - 1]), vl_next = shfl_down1(vl[0]);
#pragma unroll
            for (int f = 0; f <= R; ++f)
                gflux_partials<FLUX>(alpha, f == 0 ? vr_prev : vr[f - 1], f == R ? vl_next : vl[f], dm[f], dp[f], da[f]);
        }
#pragma unroll
        for (int t = 0; t < R; ++t) {
            if constexpr (K == 3) weno5_rev_window(12.0 * a.eps, v + t, w[t]);
            else weno3_rev_window(a.eps, pair2(v[t], v[t + 1]), pair2(v[t + 1], v[t + 2]), w[t]);
        }
        if constexpr (AMAX) {
            cand = kNone;
#pragma unroll
            for (int t = R - 1; t >= 0; --t) {
                peak[t] = owned && c0 + t < m && fabs(v[H + t]) == alpha;
                if (peak[t]) cand = 2 * (c0 + t) + (v[H + t] < 0.0);
            }
        }
    };

    double vn[NV], alpha_next = alpha;
    if (AMAX) alpha = a.alpha_rec[stages - 1], alpha_next = a.alpha_rec[stages - 2];
    if (work) {
        double v[NV];
        load_window(0, v);
        load_window(1, vn);
        window_part(v);
    }
    __syncthreads();
    int in = 0, o1 = copy, st = 0;   // lam of the step's end; the first copy of a stage in it
    const int o2 = 2 * copy;
    for (int e = 0; e < stages; ++e) {
        const AresCoef co = ares_coef(a.order, st);
        const bool last_st = st + 1 == a.order;
        // order 3: in -> o1 -> o2 -> in; order 2: in -> o1 -> in; order 1: in -> o1, then they swap
        double *const cur = L0 + (st == 0 ? in : (st == 1 ? o1 : o2));
        double *const nxt = L0 + (a.order == 1 || st == 0 ? o1 : (last_st ? in : o2));
        const double *const x1 = L0 + (a.order == 3 ? o1 : in), *const x2 = L0 + in;
        const bool with_x1 = last_st && a.order > 1, with_x2 = last_st && a.order == 3;
        const double ch = co.cc * a.dt;
        unsigned long long *const words = a.words + (size_t)e * per_stage;
        unsigned long long *const mine = words + (size_t)b * kAresLine;
        if (halo && e > 0) {
            if (B == 1) {
                if (per && lane < 2 * kAresHalo) {
                    const int j = lane < kAresHalo ? lane - kAresHalo : m + lane - kAresHalo;
                    cur[j] = cur[lane < kAresHalo ? m + j : j - m];
                }
            } else {
                const unsigned long long *p = hp + (size_t)(e - 1) * per_stage;
                unsigned long long x = 0;
                bool ok = false;
                for (int t = 0; t < polls && !ok; ++t) {
                    if (wait) x = word_load(p);
                    ok = __all(!wait || (unsigned)x == a.tag);
                }
                if (!ok) {
                    polls = 1;
                    if (lane == 0) set_status(a.status, RES_TIMEOUT);
                }
                const unsigned half = (unsigned)(x >> 32);
                const unsigned other = (unsigned)__builtin_amdgcn_update_dpp(0, (int)half, 0xB1, 0xF, 0xF, true);
                if (wait && !(lane & 1))
                    cur[(lane < 32 ? -kAresHalo : m) + (hw >> 1)] =
                        __builtin_bit_cast(double, ((unsigned long long)other << 32) | half);
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (work) {
            double mu[R], phi[R + 2], acc[NV], p1v[R], p2v[R], abar = 0.0;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                mu[t] = cur[c0 + t];
                p1v[t] = x1[c0 + t];
                p2v[t] = x2[c0 + t];
            }
#pragma unroll
            for (int t = 0; t < NV; ++t) acc[t] = 0.0;
            if constexpr (LFP) {
                const double lam_edge = cur[hc];
#pragma unroll
                for (int t = 0; t < R; ++t) phi[t + 1] = mu[t] * iw[t];
                phi[0] = shfl_up1(phi[R]);
                phi[R + 1] = shfl_down1(phi[1]);
                const double ph = lam_edge * iw_edge;
                if (lane == 0) phi[0] = ph;
                if (lane == 63) phi[R + 1] = ph;
            } else {
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    const bool end = !per && (g0 + t < 1 || g0 + t > n - 2);
                    phi[t + 1] = end ? 0.0 : fma_(0.0, 0.0, mu[t]) * iw[t];
                }
                phi[0] = shfl_up1(phi[R]);
                phi[R + 1] = shfl_down1(phi[1]);
                if constexpr (AMAX) {
#pragma unroll
                    for (int t = 0; t < R; ++t)
                        if (owned && c0 + t < m) abar = fma_(phi[t + 2] - phi[t + 1], da[t + 1], abar);
                }
            }
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const double Gp = phi[t + 2] - phi[t + 1], Gm = phi[t + 1] - phi[t];
                double gr, gl;
                if constexpr (LFP) {
                    gr = Gp * (w[t].vr + alpha);
                    gl = Gm * (w[t].vl - alpha);
                    const double ab = fma_(Gp, w[t].vr, -(Gm * w[t].vl));
                    if (owned && c0 + t < m) abar += ab;
                } else {
                    gr = Gp * dm[t + 1];
                    gl = Gm * dp[t];
                }
                if constexpr (K == 3) weno5_rev_apply(w[t], gr * w[t].ir, gl * w[t].il, acc + t);
                else weno3_rev_apply(w[t], gr * w[t].ir, gl * w[t].il, acc + t);
            }
            // the spills into the neighbours' cells
#pragma unroll
            for (int t = 0; t < H; ++t) {
                const double fromR = shfl_down1(acc[t]);
                const double fromL = shfl_up1(acc[R + H + t]);
                acc[R + t] += fromR;
                acc[H + t] += fromL;
            }
            if constexpr (!LFP) {
                // window positions past an end of the line are the end cell
                if (!per && (base + W < 1 || base + W + CH + R >= n)) {
                    if (g0 == 0) {
                        double t = 0.0;
#pragma unroll
                        for (int k = 0; k < H; ++k) t += acc[k];
                        acc[H] += t;
                    }
                    const int jl = n - 1 - g0;
                    if (jl >= 0 && jl < R) {
                        double t = 0.0;
#pragma unroll
                        for (int k = 0; k < NV; ++k)
                            if (k > H + jl) t += acc[k];
#pragma unroll
                        for (int k = 0; k < R; ++k)
                            if (k == jl) acc[H + k] += t;
                    }
                }
            }
            bool held = false;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const int j = c0 + t;
                double y;
                if constexpr (LFP) {
                    y = fma_(ch, acc[H + t], co.ca * mu[t]);
                    if (with_x1) y = fma_(co.e1, p1v[t], y);
                    if (with_x2) y = fma_(co.e2, p2v[t], y);
                } else {
                    y = fma_(0.0, 0.0, co.ca * mu[t]);
                    if (with_x1) y = fma_(co.e1, p1v[t], y);
                    if (with_x2) y = fma_(co.e2, p2v[t], y);
                    y = fma_(ch, acc[H + t], y);
                }
                if (!(owned && j < m)) continue;
                nxt[j] = y;
                if (B > 1 && (j < kAresHalo || j >= m - kAresHalo)) {
                    if (AMAX && peak[t]) {
                        held = true;
                    } else {
                        if (j < kAresHalo) put_double(mine + 2 * j, y, a.tag);
                        if (j >= m - kAresHalo) put_double(mine + 2 * (j - m + 2 * kAresHalo), y, a.tag);
                    }
                }
            }
            if constexpr (AMAX) {
                const double share = wave_sum(abar);
                if (lane == 0) part[(e & 1) * a.chunks + c] = share;
                if (cand != kNone) atomicMin(&s_peak[e & 3], cand);
                if (held) s_held[e & 3] = 1;
            }
        }
        __syncthreads();   // the stage's result is complete, but for the correction
        unsigned long long *const unit = words + (size_t)B * kAresLine;
        if constexpr (AMAX) {
            // alpha-bar's shares: groups of four chunks, and (periodic lines) the last chunks of the
            // line one by one; then the block's first cell at the maximum
            if (tid == 0) s_peak[(e + 2) & 3] = kNone, s_held[(e + 2) & 3] = 0;
            const int groups = LFP ? nch / 4 : (nch + 3) / 4, own = LFP ? groups + nch % 4 : groups;
            const int first_unit = base / CH / 4;
            if (tid < own) {
                const double *p = part + (e & 1) * a.chunks;
                double s;
                if (tid < groups) {
                    double f[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) f[k] = LFP || 4 * tid + k < nch ? p[4 * tid + k] : 0.0;
                    s = ((f[0] + f[1]) + f[2]) + f[3];
                } else {
                    s = p[4 * groups + tid - groups];
                }
                if (B == 1) sums[tid] = s;
                else put_double(unit + 2 * (first_unit + tid), s, a.tag);
            }
            if (tid == 0 && B > 1) {
                const int x = s_peak[e & 3];
                word_store(mine + 4 * kAresHalo,
                           ((unsigned long long)(x == kNone ? 0xffffffffu : (unsigned)(base + (x >> 1))) << 32) | a.tag);
            }
        }
        // the next stage's part that needs no cotangent
        [[maybe_unused]] const double alpha_now = alpha;
        if (e + 1 < stages) {
            alpha = alpha_next;
            if (AMAX) alpha_next = a.alpha_rec[max(stages - 3 - e, 0)];
            if (work) {
                double v[NV];
#pragma unroll
                for (int i = 0; i < NV; ++i) v[i] = vn[i];
                load_window(min(e + 2, stages - 1), vn);
                window_part(v);
            }
        }
        if constexpr (AMAX) {
            const int top = s_peak[e & 3];
            if (top != kNone) {   // (the same for the whole block)
                const int cell = top >> 1;
                if (tid == 0) s_first = B == 1 ? base + cell : kNone;
                __syncthreads();
                bool ok = true;
                for (int i = tid; B > 1 && i < a.units + B; i += threads) {
                    const unsigned long long *p = i < a.units ? unit + 2 * i : words + (size_t)(i - a.units) * kAresLine + 4 * kAresHalo;
                    unsigned long long x = 0, y = 0;
                    bool got = false;
                    for (int t = 0; t < polls && !got; ++t) {
                        x = word_load(p);
                        y = i < a.units ? word_load(p + 1) : x;
                        got = (unsigned)x == a.tag && (unsigned)y == a.tag;
                    }
                    ok = ok && got;
                    if (i < a.units) sums[i] = __builtin_bit_cast(double, (y & 0xffffffff00000000ull) | (x >> 32));
                    else if ((unsigned)(x >> 32) != 0xffffffffu) atomicMin(&s_first, (int)(x >> 32));
                }
                if (!__all(ok)) {
                    polls = 1;
                    if (lane == 0) set_status(a.status, RES_TIMEOUT);
                }
                __syncthreads();
                if (c == 0 && s_first == base + cell) {
                    double sum;
                    if constexpr (LFP) {
                        const int whole = (n + CH - 1) / CH / 4;
                        double s = 0.0;
                        for (int i = lane; i < whole; i += 64) s += sums[i];
                        const double single = whole + lane < a.units ? sums[whole + lane] : 0.0;
                        sum = wave_sum(s) + wave_sum(single);
                    } else {
                        double s[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            s[k] = 0.0;
                            for (int i = lane + 64 * k; i < a.units; i += kGenTile) s[k] += sums[i];
                        }
                        sum = (s[0] + s[2]) + (s[1] + s[3]);
                        for (int k = 32; k > 0; k >>= 1) sum = sum + __shfl_down(sum, k);
                    }
                    if (lane == 0) nxt[cell] += ch * sum * (top & 1 ? -1.0 : (alpha_now > 0.0 ? 1.0 : 0.0));
                }
                __syncthreads();
                if (B > 1 && s_held[e & 3] && tid < 2 * kAresHalo) {
                    const int j = tid < kAresHalo ? tid : m + tid - 2 * kAresHalo;
                    put_double(mine + 2 * tid, nxt[j], a.tag);
                }
            }
        }
        if (last_st) {
            if (a.order == 1) {
                const int t = in;
                in = o1;
                o1 = t;
            }
            st = 0;
        } else {
            ++st;
        }
    }
    for (int j = tid; j < m; j += threads) a.out[base + j] = L0[in + j];
}

}  // namespace hrw
