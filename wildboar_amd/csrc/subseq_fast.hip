// subseq_fast.hip -- FP32 subsequence scans with a certified exact finish.
//
// Semantics are those of _PairwiseSubsequenceDistance (distance/_cdistance.pyx:
// 1001-1015): for sample i and shapelet s, the minimum over windows of the
// squared cost (dtw_subsequence_distance, distance/_elastic.pyx:622-655, or
// euclidean_distance, distance/_metric.pyx:654-683), the first window that
// attains it, and sqrt of that minimum.
//
// Pass 1 (FP32): one (sample, shapelet) task per 64-lane wave.  For DTW each
//   lane runs the register-band recursion of lane.hip on a window (all lanes
//   share the shapelet, so the geometry is uniform); for euclidean each lane
//   sums (x - s)^2 over its windows.  A window is a candidate when its FP32 cost c satisfies
//   c <= tau(c*) = rho (c* + A) + A, c* the smallest FP32 cost so far: by the
//   bound in rerank.hip no other window can hold the float64 minimum.  The
//   wave keeps up to 64 candidates with their costs in LDS and drops those
//   that fail tau of the current best when the list fills; at the end the
//   ones within tau(final best) are stored (at most kMaxCand, else the task
//   is marked as overflowed).  The order in which windows are looked at does
//   not change the candidates, so DTW takes 64 windows spread over the series
//   first and then only those whose LB_Keogh sum (the window against the
//   shapelet's envelope of the band's radius, four FP32 instructions a value
//   against three per band slot) does not exceed tau of the best so far.  Sum
//   and cost carry the same kind of rounding: with K = 2 L + 2 roundings each
//   way the sum is at most rho times the window's FP32 cost, so a sum above
//   rho^2 tau leaves the cost above tau.
// Pass 2 (FP64): one candidate per lane, evaluated with the reference's exact
//   arithmetic (DTW: min(min(up, left), diag) + v*v, no FMA; euclidean: the
//   sequential sum), then per task the first strictly smallest candidate wins.
// Overflowed tasks are rescanned exactly (subseq.hip).
#pragma clang fp contract(off)

#include "block_dtw.h"
#include "lane_common.h"
#include "lane64_cost.h"
#include "subseq_fast.h"

namespace wbx {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}

// Wave-level candidate list in LDS: (window, FP32 cost) pairs, up to kCap.
// A window enters when its cost is within tau(best so far); when the list
// would overflow, entries no longer within tau(best now) are dropped (the
// best only decreases, so a dropped entry could never pass the final test).
constexpr int kCap = 64;

struct CandList {
    int count;
    bool overflow;
};

__device__ __forceinline__ void cand_push(CandList &cl, int *s_win, float *s_cost, bool take,
                                          int ws, float c, float tau) {
    const int lane = threadIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t mask = __ballot(take);
    const int npush = (int)__popcll(mask);
    if (npush == 0 || cl.overflow) return;  // uniform
    if (cl.count + npush > kCap) {
        __syncthreads();
        const bool has = lane < cl.count;
        const int w = has ? s_win[lane] : 0;
        const float cc = has ? s_cost[lane] : WBX_INF_F;
        const bool keep = has && cc <= tau;
        const uint64_t km = __ballot(keep);
        __syncthreads();
        if (keep) {
            const int pos = (int)__popcll(km & below);
            s_win[pos] = w;
            s_cost[pos] = cc;
        }
        cl.count = (int)__popcll(km);
        __syncthreads();
        if (cl.count + npush > kCap) {
            cl.overflow = true;
            return;
        }
    }
    if (take) {
        const int pos = cl.count + (int)__popcll(mask & below);
        s_win[pos] = ws;
        s_cost[pos] = c;
    }
    cl.count += npush;
}

// Final list: the entries within tau(final best), at most kMaxCand of them,
// else the task is marked for the exact rescan (count kMaxCand + 1).
__device__ __forceinline__ void cand_finish(const CandList &cl, const int *s_win,
                                            const float *s_cost, float tau, float best,
                                            SubCand *__restrict__ out) {
    const int lane = threadIdx.x;
    __syncthreads();
    const bool has = !cl.overflow && lane < cl.count;
    const int w = has ? s_win[lane] : 0;
    const float cc = has ? s_cost[lane] : WBX_INF_F;
    const bool keep = has && cc <= tau;
    const uint64_t km = __ballot(keep);
    const int n = (int)__popcll(km);
    const bool ovf = cl.overflow || n > kMaxCand;
    if (!ovf && keep) out->win[__popcll(km & ((1ull << lane) - 1ull))] = w;
    if (lane == 0) {
        out->count = ovf ? kMaxCand + 1 : n;
        out->best32 = best;
    }
}

// Four consecutive floats of a row of length T starting at e (e >= 0): one
// 16-byte load when it lies inside the row, else each index clamped to T - 1
// (those values only feed windows past the last one).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4u row4(const float *__restrict__ row, int e, int T) {
    if (e + 3 < T) return *(const f4u *)(row + e);
    f4u v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = row[e + q < T ? e + q : T - 1];
    return v;
}

// FP32 cost of the window at Y of every lane against the shapelet S (scalar
// loads through Sc), band of BP = 2 off + 1 slots; sw: the lane's window
// start (columns left of it are read when every lane has off of them).  +inf
// once every lane's row minimum is above lim (row minima only grow).
template <int BP, int U>
__device__ __forceinline__ float window_cost32(const float *__restrict__ S,
                                               const __attribute__((address_space(4))) float *Sc,
                                               int L, const float *__restrict__ Y, int sw,
                                               float lim) {
    static_assert(U % 4 == 0, "groups of whole 16-byte loads");
    constexpr int W = BP + U - 1, off = (BP - 1) / 2;
    // the tests on it below stay here: formed once for all calls they are
    // several hundred scalar values, spilled and read back for every call
    asm volatile("" : "+s"(L));
    float row[BP];
#pragma unroll
    for (int k = 0; k < BP; ++k) row[k] = (k == off) ? 0.0f : WBX_INF_F;
    float yw[W];
    if (__ballot(sw < off) == 0 && W - off <= L) {
        // uniform: every lane's columns -off .. W - off - 1 are inside the
        // series row and end inside the window; the first off are left of it
        // (+inf)
        const float *__restrict__ Yb = Y - off;
#pragma unroll
        for (int q = 0; q < W; q += 4) {
            if (q + 4 <= W) {
                const f4a v = *(const f4a *)(Yb + q);
#pragma unroll
                for (int u = 0; u < 4; ++u) yw[q + u] = v[u];
            } else {
#pragma unroll
                for (int u = 0; q + u < W; ++u) yw[q + u] = Yb[q + u];
            }
        }
#pragma unroll
        for (int m = 0; m < W; ++m) yw[m] = m < off ? WBX_INF_F : yw[m];
    } else {
#pragma unroll
        for (int m = 0; m < W; ++m) yw[m] = ldy(Y, m - off, L);
    }
    auto cells = [&](const float *y, float xi) {
        float left = WBX_INF_F;
#pragma unroll
        for (int k = 0; k < BP; ++k) {
            const float up = (k + 1 < BP) ? row[k + 1] : WBX_INF_F;
            const float mn = fminf(fminf(up, left), row[k]);
            const float d = xi - y[k];
            const float c = __builtin_fmaf(d, d, mn);
            row[k] = c;
            left = c;
        }
    };
    const int rem = L % U;
    for (int i = 0; i < rem; ++i) {
        cells(yw, S[i]);
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, i + 1 - off + W - 1, L);
    }
    for (int i0 = rem; i0 < L; i0 += U) {
        // This group's new window entries, columns jn .. jn + U - 1 (jn >=
        // 0).  Every lane has the same shapelet and row, so when they lie
        // inside the window (the usual case) they are plain vector loads,
        // waited for only at the window shift.  The shapelet values are
        // scalar loads (the shapelet stays in the scalar cache).
        float yn[U];
        const int jn = i0 - off + W;
        if (jn + U <= L) {
#pragma unroll
            for (int u = 0; u < U; u += 4) {
                const f4a b = *(const f4a *)(Y + jn + u);
#pragma unroll
                for (int q = 0; q < 4; ++q) yn[u + q] = b[q];
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) yn[u] = ldy(Y, jn + u, L);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) cells(yw + u, Sc[i0 + u]);
#pragma unroll
        for (int m = 0; m < W - U; ++m) yw[m] = yw[m + U];
#pragma unroll
        for (int u = 0; u < U; ++u) yw[W - U + u] = yn[u];
        if (BP > 3 && ((i0 - rem) / U & 3) == 3) {  // every fourth group
            float rm = row[0];
#pragma unroll
            for (int k = 1; k < BP; ++k) rm = fminf(rm, row[k]);
            if (__ballot(!(rm > lim)) == 0) return WBX_INF_F;
        }
    }
    float c = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < BP; ++k)
        if (k == off) c = row[k];
    return c;
}

// LB_Keogh sums against the DTW they save: per value of the shapelet the sums
// of 256 windows take the time of about 24 instructions and their DTW has 12 B,
// so they pay where more than 2 / B of the windows fall to them.  What share
// that is shows on the spread windows first; where it is smaller, the next four
// groups of 256 go straight to the DTW, after a further group that falls short
// the next eight, and so on up to kLbPause (the best so far falls, so a task can
// come to pay).  Tasks of few windows (subseq_bounds) take them in order.
// Starting with one group takes 1 % less time on the shapelets below and 5 %
// more on white noise.
constexpr int kLbPause = 16;
// whether `kept` of n windows are too many for the sums to pay
__device__ __forceinline__ bool subseq_short(int B, int kept, int n) {
    return (n - kept) * B < 2 * n;
}

// 256 shapelets of 16 .. 128 over 500 series of 1024, r = 0.1: 3.4 ms for
// all classes, 7.9 ms when every window's DTW was computed.
template <int BP, int U>
__global__ __launch_bounds__(64) void k_subseq_dtw32(TaskMap tasks, SubGeo sg,
                                                     SubCand *__restrict__ cands) {
    // every shapelet of the launch has a band of 2 w - 1 == BP slots
    const int lane = threadIdx.x;
    const SubTask tk = tasks.at(blockIdx.x);
    // the shapelet is the same for every lane and is not written by the
    // launch: read through the constant address space, its values are scalar
    // loads into SGPRs
    typedef const __attribute__((address_space(4))) float *cfp;
    const int64_t so = sg.off[tk.shapelet];
    const float *__restrict__ S = sg.S + so;
    const cfp Sc = (cfp)S, lo = (cfp)(sg.lo + so), hi = (cfp)(sg.hi + so);
    const int L = __builtin_amdgcn_readfirstlane((int)sg.len[tk.shapelet]);
    const int T = sg.T, nwin = T - L + 1;
    const float *__restrict__ Xrow = sg.X + (int64_t)tk.sample * sg.xstride;
    __shared__ int s_win[kCap];
    __shared__ float s_cost[kCap];
    __shared__ int queue[64 + 256];
    CandList cl{0, false};
    float best = WBX_INF_F, tau = WBX_INF_F;
    if (!subseq_bounds(BP, nwin)) {
        for (int b0 = 0; b0 < nwin; b0 += 64) {
            const int ws = b0 + lane;
            const bool active = ws < nwin;
            const int wc = active ? ws : nwin - 1;
            float c = window_cost32<BP, U>(S, Sc, L, Xrow + wc, wc, tau);
            if (!active) c = WBX_INF_F;
            best = fminf(best, wave_min(c));
            tau = sg.rho * (best + sg.A) + sg.A;
            cand_push(cl, s_win, s_cost, active && c <= tau, ws, c, tau);
        }
        cand_finish(cl, s_win, s_cost, tau, best, cands + blockIdx.x);
        return;
    }
    const int step = (nwin + 63) / 64;  // >= 2; the spread windows are lane * step
    int nq = 0, b0 = 0;
    // The windows that go straight to the DTW: the others of [.., b0), by their
    // number i0 .. i1 - 1 among the others; di, dr: the lane's number over and
    // modulo step - 1.
    int i0 = 0, i1 = 0, di = 0, dr = 0, pause = 4;
    auto others = [&](int s) { return s - (s + step - 1) / step; };  // below window s
    auto straight = [&]() {
        const int e = b0 + 256 * pause < nwin ? b0 + 256 * pause : nwin;
        pause = 2 * pause < kLbPause ? 2 * pause : kLbPause;
        i0 = others(b0);
        i1 = others(e);
        di = (i0 + lane) / (step - 1);
        dr = (i0 + lane) % (step - 1);
        b0 = e;
    };
    for (bool first = true;; first = false) {
        int ws = lane * step;
        bool active = ws < nwin;
        if (!first && i0 < i1) {
            active = i0 + lane < i1;
            ws = active ? di * step + dr + 1 : 0;
            i0 += 64;
            di += 64 / (step - 1);
            dr += 64 % (step - 1);
            if (dr >= step - 1) {
                dr -= step - 1;
                ++di;
            }
        } else if (!first) {
            while (nq < 64 && b0 < nwin) {
                // lane l forms the sums of the windows w0 .. w0 + 3
                const int w0 = b0 + 4 * lane;
                const float lim = tau * sg.rho * sg.rho * 1.000001f;
                float lb[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                {
                    float xw[8];
                    const f4u a = row4(Xrow, w0 < T ? w0 : T - 1, T),
                              b = row4(Xrow, w0 + 4 < T ? w0 + 4 : T - 1, T);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        xw[q] = a[q];
                        xw[4 + q] = b[q];
                    }
                    // the last L % 4 terms are left out
                    for (int j0 = 0; j0 + 4 <= L; j0 += 4) {
                        const f4u nx = row4(Xrow, w0 + j0 + 8 < T ? w0 + j0 + 8 : T - 1, T);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float h = hi[j0 + u], l = lo[j0 + u];
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const float d =
                                    fmaxf(fmaxf(xw[q + u] - h, l - xw[q + u]), 0.0f);
                                lb[q] = __builtin_fmaf(d, d, lb[q]);
                            }
                        }
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            xw[q] = xw[4 + q];
                            xw[4 + q] = nx[q];
                        }
                        if ((j0 & 12) == 12) {
                            const float m = fminf(fminf(lb[0], lb[1]), fminf(lb[2], lb[3]));
                            if (__ballot(!(m > lim)) == 0) break;
                        }
                    }
                }
                int kept = 0, rem = w0 % step;  // rem 0: a spread window
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int s = w0 + q;
                    const bool keep = s < nwin && rem != 0 && !(lb[q] > lim);
                    const uint64_t km = __ballot(keep);
                    if (keep) queue[nq + kept + (int)__popcll(km & ((1ull << lane) - 1ull))] = s;
                    kept += (int)__popcll(km);
                    rem = rem + 1 == step ? 0 : rem + 1;
                }
                nq += kept;
                const bool few = subseq_short(BP, kept, min(256, nwin - b0));
                b0 += 256;
                __syncthreads();
                if (few && b0 < nwin) {
                    straight();
                    break;
                }
                if (!few) pause = 4;
            }
            if (nq < 64 && i0 < i1) continue;
            if (nq == 0) break;
            active = lane < nq;
            // the newest 64 of the queue
            ws = queue[active ? (nq < 64 ? lane : nq - 64 + lane) : 0];
            nq = nq < 64 ? 0 : nq - 64;
            __syncthreads();
        }
        const int wc = active ? ws : (first ? 0 : ws);
        float c = window_cost32<BP, U>(S, Sc, L, Xrow + wc, wc, tau);
        if (!active) c = WBX_INF_F;
        best = fminf(best, wave_min(c));
        tau = sg.rho * (best + sg.A) + sg.A;
        cand_push(cl, s_win, s_cost, active && c <= tau, ws, c, tau);
        if (first) {  // how many of these would their sums have kept
            const float lim = tau * sg.rho * sg.rho * 1.000001f;
            const float *__restrict__ x = Xrow + wc;
            float lb = 0.0f;
            for (int j0 = 0; j0 + 4 <= L; j0 += 4) {
                const f4a v = *(const f4a *)(x + j0);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float d = fmaxf(fmaxf(v[u] - hi[j0 + u], lo[j0 + u] - v[u]), 0.0f);
                    lb = __builtin_fmaf(d, d, lb);
                }
            }
            const int kept = (int)__popcll(__ballot(active && !(lb > lim)));
            if (subseq_short(BP, kept, (int)__popcll(__ballot(active)))) straight();
        }
    }
    cand_finish(cl, s_win, s_cost, tau, best, cands + blockIdx.x);
}

// Envelope of each packed shapelet over the band's columns, |k - j| < w.
__global__ __launch_bounds__(64) void k_subseq_envelope(const float *__restrict__ S,
                                                        const int64_t *__restrict__ off,
                                                        const int64_t *__restrict__ len, double r,
                                                        float *__restrict__ lo,
                                                        float *__restrict__ hi) {
    const int64_t j = blockIdx.x;
    const int L = (int)len[j];
    const int rad = band_w(L, L, r) - 1;
    const float *__restrict__ s = S + off[j];
    for (int k = threadIdx.x; k < L; k += 64) {
        const int a = k - rad > 0 ? k - rad : 0, b = k + rad < L - 1 ? k + rad : L - 1;
        float l = s[a], h = s[a];
        for (int q = a + 1; q <= b; ++q) {
            l = fminf(l, s[q]);
            h = fmaxf(h, s[q]);
        }
        lo[off[j] + k] = l;
        hi[off[j] + k] = h;
    }
}

// Lane l owns the U = 4 consecutive windows w0 .. w0 + 3 (w0 = b0 + 4 l) and
// keeps x[w0 + j .. w0 + j + 8) in registers: four steps of j use static
// indices (window q at step u reads xw[q + u]), then the window moves by four
// with one 16-byte load.  Each window's sum runs over j in order.
template <int U>
__global__ __launch_bounds__(64) void k_subseq_euclid32(TaskMap tasks, SubGeo sg,
                                                        SubCand *__restrict__ cands) {
    static_assert(U == 4, "four windows per lane");
    const int lane = threadIdx.x;
    const SubTask tk = tasks.at(blockIdx.x);
    const float *__restrict__ S = sg.S + sg.off[tk.shapelet];
    const int L = (int)sg.len[tk.shapelet];
    const int T = sg.T;
    const int nwin = T - L + 1;
    const float *__restrict__ Xrow = sg.X + (int64_t)tk.sample * sg.xstride;
    __shared__ int s_win[kCap];
    __shared__ float s_cost[kCap];
    CandList cl{0, false};
    float best = WBX_INF_F;
    for (int b0 = 0; b0 < nwin; b0 += 64 * U) {
        const int w0 = b0 + lane * U;
        float acc[U];
#pragma unroll
        for (int q = 0; q < U; ++q) acc[q] = 0.0f;
        float xw[2 * U];
        {
            const f4u lo = row4(Xrow, w0, T), hi = row4(Xrow, w0 + U, T);
#pragma unroll
            for (int q = 0; q < U; ++q) {
                xw[q] = lo[q];
                xw[U + q] = hi[q];
            }
        }
        int j0 = 0;
        for (; j0 + U <= L; j0 += U) {
            const f4u nx = row4(Xrow, w0 + j0 + 2 * U, T);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float sj = S[j0 + u];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    const float d = xw[q + u] - sj;
                    acc[q] = __builtin_fmaf(d, d, acc[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < U; ++q) {
                xw[q] = xw[U + q];
                xw[U + q] = nx[q];
            }
        }
        for (int u = 0; j0 + u < L; ++u) {  // the last L % U steps
            const float sj = S[j0 + u];
#pragma unroll
            for (int q = 0; q < U; ++q) {
                float xv = xw[q];
#pragma unroll
                for (int t = 1; t < U; ++t)
                    if (u == t) xv = xw[q + t];
                const float d = xv - sj;
                acc[q] = __builtin_fmaf(d, d, acc[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const int ws = w0 + q;
            const bool active = ws < nwin;
            const float c = active ? acc[q] : WBX_INF_F;
            best = fminf(best, wave_min(c));
            const float tau = sg.rho * (best + sg.A) + sg.A;
            cand_push(cl, s_win, s_cost, active && c <= tau, ws, c, tau);
        }
    }
    cand_finish(cl, s_win, s_cost, sg.rho * (best + sg.A) + sg.A, best,
                cands + blockIdx.x);
}

// ------------------------------------------------------------------ exact
// Float64 cost of one candidate window per lane; per-lane geometry (all lanes
// of a launch share BP).  Same arithmetic as dtw_distance: rows of S against
// the window, cost = min(min(up, left), diag) + v * v.  A wave lists the
// candidates of `per` tasks in LDS and its lanes go over the list: most tasks
// have one or two of the kMaxCand, and a lane for each place leaves seven of
// eight idle.  (A list of the whole launch in memory takes a counter that every
// task adds to, 13 ns each in turn: 1.03 ms for 80000 tasks of any length, 0.15
// ms without.  Four waves of a block over one list take three times as long as
// one wave where there are few tasks.)
constexpr int kCandTasks = 48;

template <int BP>
__global__ __launch_bounds__(64) void k_subseq_cand64(TaskMap tasks,
                                                      const SubCand *__restrict__ cands,
                                                      int64_t n_tasks, int per,
                                                      const double *__restrict__ S64,
                                                      const int64_t *__restrict__ soff,
                                                      const int64_t *__restrict__ slen,
                                                      const double *__restrict__ X64,
                                                      int64_t xstride, int T, double r, int kind,
                                                      double *__restrict__ cost64) {
    __shared__ uint16_t list[kCandTasks * kMaxCand];  // (task - t0) * kMaxCand + place
    const int lane = threadIdx.x;
    const int64_t t0 = (int64_t)blockIdx.x * per;
    int c = lane < per && t0 + lane < n_tasks ? cands[t0 + lane].count : 0;
    if (c > kMaxCand) c = 0;  // rescanned
    int inc = c;              // inclusive scan over the lanes
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    for (int s = 0; s < c; ++s) list[inc - c + s] = (uint16_t)(lane * kMaxCand + s);
    const int n = __shfl(inc, 63);
    __syncthreads();
    for (int q = lane; q < n; q += 64) {
        const int64_t at = t0 * kMaxCand + list[q];
        const int64_t t = at / kMaxCand;
        const SubTask tk = tasks.at(t);
        const double *S = S64 + soff[tk.shapelet];
        const int L = (int)slen[tk.shapelet];
        const double *Y = X64 + (int64_t)tk.sample * xstride + cands[t].win[at - t * kMaxCand];
        double res;
        if (kind == WBX_EUCLIDEAN) {
            double dist = 0.0;
            for (int j = 0; j < L; ++j) {
                double v = Y[j];
                v -= S[j];
                dist += v * v;
            }
            res = dist;
        } else {
            // the band row in registers with a sliding window of the
            // candidate's values (the float64 lane kernels' cell arithmetic,
            // bit for bit); a launch holds one band class, B in (BP - 8, BP),
            // whose padding slot B the routine resets every row
            const int w = band_w(L, L, r);
            res = lane64_cost<BP, 4, false, false, true>(S, L, Y, L, w - 1, 2 * w - 1, w - 1,
                                                         nullptr, L);
        }
        cost64[at] = res;
    }
}

// Per task: the smallest exact cost among the candidates, of equal ones the
// first window (the list is in the order in which the windows were looked at).
__global__ __launch_bounds__(256) void k_subseq_select(TaskMap tasks,
                                                       const SubCand *__restrict__ cands,
                                                       int64_t n_tasks,
                                                       const double *__restrict__ cost64,
                                                       int64_t n_shapelets,
                                                       double *__restrict__ dist,
                                                       int64_t *__restrict__ idx,
                                                       int32_t *__restrict__ overflow,
                                                       int *__restrict__ n_overflow) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n_tasks) return;
    const SubCand &cd = cands[t];
    const SubTask tk = tasks.at(t);
    if (cd.count > kMaxCand || cd.count == 0) {
        const int o = atomicAdd(n_overflow, 1);
        overflow[o] = (int32_t)t;
        return;
    }
    double best = WBX_INF_D;
    int bw = 0x7fffffff;
    for (int s = 0; s < cd.count; ++s) {
        const double c = cost64[t * kMaxCand + s];
        const int wv = cd.win[s];
        if (c < best || (c == best && wv < bw)) {
            best = c;
            bw = wv;
        }
    }
    const int64_t o = (int64_t)tk.sample * n_shapelets + tk.shapelet;
    dist[o] = sqrt(best);
    idx[o] = bw;
}

// Exact full scan of the tasks whose candidate list overflowed: one task per
// 64-lane block, windows in order (the plain kernel's block recursion).
__global__ __launch_bounds__(64) void k_subseq_rescan(TaskMap tasks, const int32_t *__restrict__ list,
                                                      const int *__restrict__ n_list, int kind,
                                                      const double *__restrict__ S64,
                                                      const int64_t *__restrict__ soff,
                                                      const int64_t *__restrict__ slen,
                                                      const double *__restrict__ X64,
                                                      int64_t xstride, int T, double r, int cap,
                                                      int64_t n_shapelets, double *__restrict__ dist,
                                                      int64_t *__restrict__ idx) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *buf = reinterpret_cast<double *>(smem_raw);
    if ((int)blockIdx.x >= *n_list) return;
    const SubTask tk = tasks.at(list[blockIdx.x]);
    const double *S = S64 + soff[tk.shapelet];
    const int L = (int)slen[tk.shapelet];
    const double *x = X64 + (int64_t)tk.sample * xstride;
    double best = WBX_INF_D;
    int64_t bi = 0;
    if (kind == WBX_EUCLIDEAN) {
        if (threadIdx.x == 0) {
            for (int s = 0; s < T - L + 1; ++s) {
                double d = 0.0;
                for (int k = 0; k < L; ++k) {
                    if (d >= best) break;
                    double v = x[s + k];
                    v -= S[k];
                    d += v * v;
                }
                if (d < best) {
                    best = d;
                    bi = s;
                }
            }
        }
    } else {
        const int w = band_w(L, L, r);
        for (int s = 0; s <= T - L; ++s) {
            const double c = block_dtw<double>(S, L, x + s, L, w, nullptr, buf, buf + cap,
                                               buf + 2 * cap);
            if (c < best) {
                best = c;
                bi = s;
            }
        }
    }
    if (threadIdx.x == 0) {
        const int64_t o = (int64_t)tk.sample * n_shapelets + tk.shapelet;
        dist[o] = sqrt(best);
        idx[o] = bi;
    }
}

int launch_subseq_rescan(TaskMap tasks, const int32_t *list, const int *n_list_dev,
                         int n_list_host, int kind, const double *S64, const int64_t *soff,
                         const int64_t *slen, const double *X64, int64_t xstride, int T, double r,
                         int max_len, int64_t n_shapelets, double *dist, int64_t *idx,
                         hipStream_t st) {
    if (n_list_host <= 0) return WBX_OK;
    const size_t lds = (size_t)3 * (size_t)max_len * sizeof(double);
    if (lds > 64 * 1024) return fail(WBX_EUNSUPPORTED, "shapelet too long for the rescan");
    hipLaunchKernelGGL(k_subseq_rescan, dim3((unsigned)n_list_host), dim3(64), lds, st, tasks, list,
                       n_list_dev, kind, S64, soff, slen, X64, xstride, T, r, max_len, n_shapelets,
                       dist, idx);
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

// ------------------------------------------------------------------ launch
// FP32 scans are compiled for every odd band width B = 2 w - 1 <= 63 (equal
// lengths), so no slot beyond the band is computed.
#define SUB_SCAN_CASES(X)                                                                        \
    X(1, 8) X(3, 8) X(5, 8) X(7, 8) X(9, 8) X(11, 8) X(13, 8) X(15, 8) X(17, 8) X(19, 8) X(21, 8) \
        X(23, 8) X(25, 8) X(27, 8) X(29, 8) X(31, 8) X(33, 4) X(35, 4) X(37, 4) X(39, 4)        \
            X(41, 4) X(43, 4) X(45, 4) X(47, 4) X(49, 4) X(51, 4) X(53, 4) X(55, 4) X(57, 4)     \
                X(59, 4) X(61, 4) X(63, 4)
#define SUB_DTW_CASES(X) X(8, 8) X(16, 8) X(24, 8) X(32, 8) X(40, 8) X(48, 8) X(56, 8) X(64, 8)

int launch_subseq_envelope(const float *S, const int64_t *off, const int64_t *len, int64_t n_s,
                           double r, float *lo, float *hi, hipStream_t st) {
    if (n_s <= 0) return WBX_OK;
    hipLaunchKernelGGL(k_subseq_envelope, dim3((unsigned)n_s), dim3(64), 0, st, S, off, len, r, lo,
                       hi);
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

int launch_subseq_fast(int kind, int B, TaskMap tasks, int64_t n_tasks, SubGeo sg,
                       SubCand *cands, hipStream_t st) {
    if (n_tasks <= 0) return WBX_OK;
    if (n_tasks > 0x7fffffff) return fail(WBX_EUNSUPPORTED, "too many subsequence tasks");
    const dim3 grid((unsigned)n_tasks);
    if (kind == WBX_EUCLIDEAN) {
        hipLaunchKernelGGL(k_subseq_euclid32<4>, grid, dim3(64), 0, st, tasks, sg, cands);
    } else {
        switch (B) {
#define SD_CASE(B_, U_) \
    case B_:                                                                                   \
        hipLaunchKernelGGL((k_subseq_dtw32<B_, U_>), grid, dim3(64), 0, st, tasks, sg, cands); \
        break;
            SUB_SCAN_CASES(SD_CASE)
#undef SD_CASE
            default: return fail(WBX_EUNSUPPORTED, "subsequence band %d", B);
        }
    }
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

int launch_subseq_exact_cands(int kind, int B, TaskMap tasks, const SubCand *cands,
                              int64_t n_tasks, const double *S64, const int64_t *soff,
                              const int64_t *slen, const double *X64, int64_t xstride, int T,
                              double r, double *cost64, hipStream_t st) {
    if (n_tasks <= 0) return WBX_OK;
    // A wave per SIMD while it then has eight tasks or more (eight: one turn of
    // the lanes whatever their candidates), up to kCandTasks in larger launches
    // (their one or two each about fill the lanes).
    const int64_t want = (n_tasks + 1023) / 1024;
    const int per = (int)(want < 8 ? 8 : want < kCandTasks ? want : kCandTasks);
    const dim3 grid((unsigned)((n_tasks + per - 1) / per));
    switch (kind == WBX_EUCLIDEAN ? 8 : (B + 7) / 8 * 8) {
#define C_CASE(B_, U_)                                                                            \
    case B_:                                                                                      \
        hipLaunchKernelGGL(k_subseq_cand64<B_>, grid, dim3(64), 0, st, tasks, cands, n_tasks, per, \
                           S64, soff, slen, X64, xstride, T, r, kind, cost64);                    \
        break;
        SUB_DTW_CASES(C_CASE)
#undef C_CASE
        default: return fail(WBX_EUNSUPPORTED, "subsequence band %d", B);
    }
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

int launch_subseq_select(TaskMap tasks, const SubCand *cands, int64_t n_tasks,
                         const double *cost64, int64_t n_shapelets, double *dist, int64_t *idx,
                         int32_t *overflow, int *n_overflow, hipStream_t st) {
    if (n_tasks <= 0) return WBX_OK;
    hipLaunchKernelGGL(k_subseq_select, dim3((unsigned)((n_tasks + 255) / 256)), dim3(256), 0, st,
                       tasks, cands, n_tasks, cost64, n_shapelets, dist, idx, overflow, n_overflow);
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

}  // namespace wbx
