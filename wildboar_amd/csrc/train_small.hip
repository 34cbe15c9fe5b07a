// train_small.hip -- differentiable DTW of few pairs: barycenter steps (one
// mean against a cluster's series) and other calls that would leave most of
// the chip idle with one pair per lane (train.hip).
//
//  k_small_train     the forward with n = ceil(B / S) lanes per pair, S = 2 or
//                    4 band slots each, one row behind the lane before
//                    (group.hip's schedule).  Every lane writes one byte per
//                    row: which of its cells took the diagonal predecessor
//                    (low nibble) and the up (high nibble).
//  k_small_backward  one wave per pair.  Lane k loads the byte of band slot k,
//                    two compares give the row's decisions as 64-bit masks in
//                    SGPRs, and the path is walked there: the exit of a row
//                    is a count of leading zeros.  The rows' column ranges go
//                    to LDS and the 64 lanes form the gradient terms of rows,
//                    then columns (prefix sums of y, then of x, in
//                    LDS), with the arithmetic of k_lane_backtrack.
//  k_sum_pairs       dX from the per-pair rows.
//
// Bound by latency: the chain of cells of a row in the forward, the chain of
// rows in the walk.  1 x 512 pairs of 256, r = 0.1, against one pair per lane
// (8 waves): forward 221 -> 36 us, backward 334 -> 59 us.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "lane_train.h"
#include "train_small.h"

namespace wbx {

namespace {

constexpr int SU = 8;        // steps whose loads are issued together
constexpr int kSmallMaxB = 112;
constexpr int kSmallMaxLen = 2048;  // LDS of the backward
constexpr double kSmallPairs = 16384;

__device__ __forceinline__ float sshr1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x138,
                                                      0xF, 0xF, false));
}
__device__ __forceinline__ float sshl1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x130,
                                                      0xF, 0xF, false));
}

// c = min3(up, left, dg) + (x - y)^2 with the two decision bits shifted into
// pd (clear: the minimum came from diag) and pu (from up); see train_cell.
__device__ __forceinline__ float small_cell(float up, float left, float dg, float x, float y,
                                            uint32_t &pd, uint32_t &pu) {
    train_cell<false>(dg, up, left, x, y, pd, pu);
    return dg;
}

struct SmallGeo {
    int lx, ly, off, B, kf;
    int S, n, P;  // slots per lane, lanes per pair (decision bytes per row), pairs per wave
};

// Two slots per lane while every wave then has a SIMD to itself (the shorter
// chain), else four.
SmallGeo small_geo(const Band &bd, int64_t n_pairs) {
    SmallGeo g;
    g.lx = bd.lx;
    g.ly = bd.ly;
    g.off = bd.off;
    g.B = bd.B;
    g.kf = bd.ly - bd.lx + bd.off;
    g.S = 2;
    g.n = (bd.B + 1) / 2;
    g.P = 64 / g.n;
    if ((n_pairs + g.P - 1) / g.P > 1024) {
        g.S = 4;
        g.n = (bd.B + 3) / 4;
        g.P = 64 / g.n;
    }
    return g;
}

template <int S>
struct SLane {
    float row[S];
    float yw[S + SU - 1];  // yw[q] = y[yj + q]
    float l;               // last slot of the lane's last row
    int r, yj;
    bool first, last;
};

// One row of the lane; SEL keeps the state of lanes outside [0, lx).  MB: the
// place of slot B - 1 in the last lane; its up input is +inf, so whatever
// the slots past the band hold never enters it.
template <int S, int MB, bool SEL>
__device__ __forceinline__ uint32_t small_step(SLane<S> &L, int u, float x, int lx) {
    const bool act = !SEL || (unsigned)(L.r + u) < (unsigned)lx;
    float left = sshr1(L.l);
    left = L.first ? WBX_INF_F : left;
    uint32_t pd = 0, pu = 0;
    auto up_of = [&](int m, float up) { return m == MB && L.last ? WBX_INF_F : up; };
    const float c0 = small_cell(up_of(0, L.row[1]), left, L.row[0], x, L.yw[u], pd, pu);
    const float Uin = sshl1(SEL && !act ? L.row[0] : c0);
    left = c0;
#pragma unroll
    for (int m = 1; m < S; ++m) {
        const float c = small_cell(up_of(m, m == S - 1 ? Uin : L.row[m + 1]), left, L.row[m], x,
                                   L.yw[u + m], pd, pu);
        L.row[m] = SEL ? (act ? c : L.row[m]) : c;
        left = c;
    }
    L.row[0] = SEL ? (act ? c0 : L.row[0]) : c0;
    L.l = L.row[S - 1];
    // slot m at bit S - 1 - m of each nibble, set where the minimum came from
    return (pd | pu << 4) ^ ((1u << S) - 1u) * 0x11u;
}

__device__ __forceinline__ void small_loads(const float *__restrict__ X,
                                            const float *__restrict__ Y, int xr, int yc, int lx,
                                            int ly, float (&xo)[SU], float (&yo)[SU]) {
    const bool in = xr >= 0 && xr + SU <= lx && yc >= 0 && yc + SU <= ly;
    if (__ballot(!in) == 0) {  // uniform
#pragma unroll
        for (int u = 0; u < SU; u += 4) {
            const f4a a = *(const f4a *)(X + xr + u);
            const f4a b = *(const f4a *)(Y + yc + u);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                xo[u + e] = a[e];
                yo[u + e] = b[e];
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const int i = xr + u;
            xo[u] = X[i < 0 ? 0 : (i >= lx ? lx - 1 : i)];
            yo[u] = ldy(Y, yc + u, ly);
        }
    }
}

template <int S, int MB>
__global__ __launch_bounds__(64) void k_small_train(PairSpec ps, Series<float> xs,
                                                    Series<float> ys, SmallGeo g,
                                                    double *__restrict__ D,
                                                    float *__restrict__ sq,
                                                    unsigned char *__restrict__ dec) {
    const int lane = threadIdx.x;
    const int gi = lane / g.n;
    const int q = lane - gi * g.n;
    const int64_t p = (int64_t)blockIdx.x * g.P + gi;
    const bool valid = gi < g.P && p < ps.n_pairs;
    int64_t a = 0, b = 0;
    if (valid) decode_pair(ps, p, a, b);
    const float *__restrict__ X = xs.row(a);
    const float *__restrict__ Y = ys.row(b);
    const int lx = g.lx, ly = g.ly, k0 = q * S;
    constexpr int W = S + SU - 1;

    SLane<S> L;
    L.first = q == 0;
    L.last = q == g.n - 1;
#pragma unroll
    for (int m = 0; m < S; ++m) L.row[m] = k0 + m == g.off ? 0.0f : WBX_INF_F;
    L.l = L.row[S - 1];
    L.r = -q;
    L.yj = L.r + k0 - g.off;
#pragma unroll
    for (int m = 0; m < W; ++m) L.yw[m] = ldy(Y, L.yj + m, ly);
    // the wave's bytes start at its first pair; the lane's byte of row r is
    // n r further (at most 32 pairs of 2048 rows of 56 bytes)
    unsigned char *__restrict__ wout = dec + (int64_t)blockIdx.x * g.P * lx * g.n;
    uint32_t at = (uint32_t)(gi * lx * g.n + q + L.r * g.n);  // of row L.r

    const int steps = lx + g.n - 1;
    float xv[SU], yn[SU];
    small_loads(X, Y, L.r, L.yj + W, lx, ly, xv, yn);
    auto group = [&](auto edge) {
        constexpr bool E = decltype(edge)::value;
        float xb[SU], yb[SU];
        small_loads(X, Y, L.r + SU, L.yj + W + SU, lx, ly, xb, yb);
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const uint32_t bits = small_step<S, MB, E>(L, u, xv[u], lx);
            if (valid && (!E || (unsigned)(L.r + u) < (unsigned)lx))
                wout[at] = (unsigned char)bits;
            at += (uint32_t)g.n;
        }
#pragma unroll
        for (int m = 0; m < W - SU; ++m) L.yw[m] = L.yw[m + SU];
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            L.yw[W - SU + u] = yn[u];
            yn[u] = yb[u];
            xv[u] = xb[u];
        }
        L.r += SU;
        L.yj += SU;
    };
    int s = 0;
    for (; s < g.n - 1; s += SU) group(std::true_type());
    for (; s + SU <= lx; s += SU) group(std::false_type());
    for (; s < steps; s += SU) group(std::true_type());

    if (valid && g.kf >= k0 && g.kf < k0 + S) {
        float res = WBX_INF_F;
#pragma unroll
        for (int m = 0; m < S; ++m)
            if (k0 + m == g.kf) res = L.row[m];
        sq[p] = res;
        D[p] = sqrt((double)res);
    }
}

// Where a pair's gradient rows go: the output itself where it is the only
// pair of its series, else its row of the per-pair scratch.
struct SmallGrad {
    float *gx;    // gx[(one_b ? a : p) * ldgx + i]
    float *gy;    // gy[(one_a ? b : p) * ldgy + j]
    int64_t ldgx, ldgy;
    int one_b, one_a;
};

// LDS: x (lx), prefix sums of y (ly + 1, float64), the rows' column ranges
// (lx), the columns' row ranges (ly).
size_t small_lds(int lx, int ly) {
    return (size_t)((lx > ly ? lx : ly) + 1) * 8 + (size_t)(lx + ly) * 4;
}

// WIDE: bands of 65 .. 112 slots (two masks per row).
template <bool WIDE>
__global__ __launch_bounds__(64) void k_small_backward(PairSpec ps, Series<float> xs,
                                                       Series<float> ys, SmallGeo g,
                                                       const float *__restrict__ sq,
                                                       const double *__restrict__ G,
                                                       const unsigned char *__restrict__ dec,
                                                       SmallGrad out) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *pt = (double *)smem;  // pt[j] = y[0] + ... + y[j - 1], later of x
    uint32_t *rows = (uint32_t *)(pt + (g.lx > g.ly ? g.lx : g.ly) + 1);  // je << 16 | jx
    uint32_t *cols = rows + g.lx;                  // last row << 16 | first row
    const int lane = threadIdx.x;
    const int64_t p = blockIdx.x;
    int64_t a, b;
    decode_pair(ps, p, a, b);
    const float *__restrict__ X = xs.row(a);
    const float *__restrict__ Y = ys.row(b);
    const int lx = g.lx, ly = g.ly, off = g.off, B = g.B, n = g.n;
    // the walk's first rows of decisions, RB rows at a time: lane k holds the
    // byte of slot k (slots past the band read the last lane's; their bits
    // are above every slot the walk asks about)
    constexpr int RB = 16, NM = WIDE ? 2 : 1;
    const unsigned char *__restrict__ drow = dec + p * lx * n;
    int dq[NM], sh[NM];
#pragma unroll
    for (int e = 0; e < NM; ++e) {
        const int k = lane + 64 * e;
        dq[e] = k / g.S < n ? k / g.S : n - 1;
        sh[e] = g.S - 1 - k % g.S;
    }
    uint32_t cur[RB][NM], nxt[RB][NM];
    auto load = [&](uint32_t(&w)[RB][NM], int ih) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int i = ih - r < 0 ? 0 : ih - r;
#pragma unroll
            for (int e = 0; e < NM; ++e) w[r][e] = drow[(uint32_t)(i * n) + (uint32_t)dq[e]];
        }
    };
    load(cur, lx - 1);
    auto prefix = [&](const float *__restrict__ v, int len) {  // the scan of k_prefix
        if (lane == 0) pt[0] = 0.0;
        double carry = 0.0;
        for (int j0 = 0; j0 < len; j0 += 64) {
            const int j = j0 + lane;
            double s = j < len ? (double)v[j] : 0.0;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const double o = __shfl_up(s, d);
                if (lane >= d) s += o;
            }
            s += carry;
            if (j < len) pt[j + 1] = s;
            carry = __shfl(s, 63);
        }
    };
    prefix(Y, ly);

    int k = g.kf;  // the walk is uniform over the wave
    for (int ih = lx - 1; ih >= 0; ih -= RB) {
        load(nxt, ih - RB);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int i = ih - r;
            if (i < 0) break;
            const int klo = off - i > 0 ? off - i : 0;
            int khi = ly - 1 - i + off;
            if (khi > B - 1) khi = B - 1;
            if (k > khi) k = khi;
            // exit: the highest slot <= k whose decision is diag or up
            uint64_t mE[NM], mD[NM];
#pragma unroll
            for (int e = 0; e < NM; ++e) {
                const uint32_t v = cur[r][e] >> sh[e];
                mE[e] = __ballot((v & 0x11) != 0);
                mD[e] = __ballot((v & 1) != 0);
            }
            int kx = -1;
            bool isd = false;
            if constexpr (WIDE) {
                const uint64_t hi = k >= 64 ? mE[1] << (127 - k) : 0;
                const uint64_t lo = k >= 64 ? mE[0] : mE[0] << (63 - k);
                if (hi) {
                    kx = k - __builtin_clzll(hi);
                    isd = (mD[1] >> (kx - 64) & 1) != 0;
                } else if (lo) {
                    kx = (k >= 64 ? 63 : k) - __builtin_clzll(lo);
                    isd = (mD[0] >> kx & 1) != 0;
                }
            } else {
                const uint64_t t = mE[0] << (63 - k);
                if (t) {
                    kx = k - __builtin_clzll(t);
                    isd = (mD[0] >> kx & 1) != 0;
                }
            }
            // Row 0 ends at column 0 (only left moves there); the other two
            // are unreachable on a finite path and keep the walk in bounds.
            if (i == 0 || kx < klo) {
                kx = klo;
                isd = false;
            }
            if (k < kx) k = kx;
            const int je = i + k - off, jx = i + kx - off;  // in [0, ly)
            rows[i] = (uint32_t)je << 16 | (uint32_t)jx;  // every lane the same
            k = isd ? kx : kx + 1;
        }
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int e = 0; e < NM; ++e) cur[r][e] = nxt[r][e];
    }
    __syncthreads();

    const double Dp = sqrt((double)sq[p]);
    const double coefd = Dp > 0.0 ? G[p] / Dp : 0.0;
    const float coef = (float)coefd;
    float *__restrict__ gx = out.gx + (out.one_b ? a : p) * out.ldgx;
    float *__restrict__ gy = out.gy + (out.one_a ? b : p) * out.ldgy;
    for (int i = lane; i < lx; i += 64) {
        const uint32_t v = rows[i];
        const int jx = v & 0xffff, je = v >> 16;
        const float xi = X[i];
        gx[i] = (float)(coefd * ((double)(je - jx + 1) * (double)xi - (pt[je + 1] - pt[jx])));
        // Consecutive rows share at most one column (an up step), so a column
        // has its first row here unless it is the one shared with the row
        // above, its last unless shared with the row below.
        const int above = i > 0 ? (int)(rows[i - 1] >> 16) : -1;
        const int below = i + 1 < lx ? (int)(rows[i + 1] & 0xffff) : ly;
        for (int j = jx; j <= je; ++j) {
            if (j > above) ((uint16_t *)cols)[2 * j] = (uint16_t)i;
            if (j < below) ((uint16_t *)cols)[2 * j + 1] = (uint16_t)i;
        }
    }
    __syncthreads();
    prefix(X, lx);
    __syncthreads();
    // a value of x that is not finite belongs to the columns it is matched to,
    // not to all behind it
    const bool sums = fabs(pt[lx]) < WBX_INF_D;  // uniform
    for (int j = lane; j < ly; j += 64) {
        const uint32_t v = cols[j];
        const int i0 = v & 0xffff, i1 = v >> 16;
        const float cnt = (float)(i1 - i0 + 1);
        double sx = 0.0;
        if (sums)
            sx = pt[i1 + 1] - pt[i0];
        else
            for (int i = i0; i <= i1; ++i) sx += (double)X[i];
        gy[j] = __builtin_fmaf(coef * cnt, Y[j], -(coef * (float)sx));
    }
}

// dX[a][i] = sum over b of gxp[(a ny + b) lx + i]: 64 columns per block, the
// pairs split over the block's 16 waves, then the waves' sums in order.
__global__ __launch_bounds__(1024) void k_sum_pairs(const float *__restrict__ gxp, int64_t ny,
                                                    int lx, float *__restrict__ dX, int64_t ldx) {
    __shared__ float part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    const int64_t a = blockIdx.y;
    const int64_t per = (ny + 15) / 16, b0 = w * per, b1 = b0 + per < ny ? b0 + per : ny;
    float s = 0.0f;
    if (i < lx) {
        const float *src = gxp + (a * ny) * lx + i;
#pragma unroll 8
        for (int64_t b = b0; b < b1; ++b) s += src[b * lx];
    }
    part[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < lx) {
#pragma unroll
        for (int e = 1; e < 16; ++e) s += part[e][lane];
        dX[a * ldx + i] = s;
    }
}

struct SmallScratch {
    int64_t gx, gw, part, total;
};

SmallScratch small_scratch(int mode, int64_t nx, int64_t ny, int lx, int ly) {
    SmallScratch t{};
    auto al = [](int64_t v) { return (v + 255) / 256 * 256; };
    if (mode == 0) {
        t.gw = ny > 1 ? al(nx * ny * lx * 4) : 0;
        t.part = t.gw + (nx > 1 ? al(nx * ny * ly * 4) : 0);
        t.total = t.part + (nx > 1 ? al(sum_cols_part_floats(nx, ny, ly) * 4) : 0);
    }
    if (t.total == 0) t.total = 256;
    return t;
}

}  // namespace

// Pairs up to which the small form is the faster one.  Its walk takes a wave a
// pair whatever the band, the other form's time grows with the band, and its
// walk with the length at one wave per SIMD.  Where they cross, one step
// forward and backward (measured at 256 .. 32768 pairs, matrices and lists):
//   series of 64:   B <= 9 16000 pairs
//   series of 256:  B <= 9 6000, 25 8200, 49 11500, 111 13500
//   series of 1000: B <= 9 3900, 25 5200, 49 7900, 111 9500
// Matrices with many columns that are no multiple of 64 stay here: dX is a sum
// over a row's pairs in turn there, 0.11 us a column (1 x 10000 pairs of 128,
// B = 9: 191 us, 1285 us).
bool small_train_ok(int mode, int64_t nx, int64_t ny, const Band &bd) {
    if (bd.B > kSmallMaxB || bd.lx > kSmallMaxLen || bd.ly > kSmallMaxLen) return false;
    const double n_pairs = mode == 0 ? (double)nx * (double)ny : (double)nx;
    if (mode == 0 && ny % 64 != 0 && ny >= 1024) return n_pairs <= kSmallPairs;
    const double at256 = bd.B <= 49 ? 6000.0 + 137.5 * (bd.B > 9 ? bd.B - 9 : 0)
                                    : 11500.0 + 32.0 * (bd.B - 49);
    return n_pairs <=
           std::min(kSmallPairs, at256 * std::pow(256.0 / bd.lx, bd.lx < 256 ? 0.7 : 0.3));
}

static int64_t small_dec_bytes(int64_t n_pairs, const SmallGeo &g) {
    return (n_pairs * g.lx * g.n + 255) / 256 * 256;
}

void small_train_sizes(int mode, int64_t nx, int64_t ny, const Band &bd, int64_t *state_bytes,
                       int64_t *scratch_bytes) {
    const int64_t np = mode == 0 ? nx * ny : nx;
    const SmallGeo g = small_geo(bd, np);
    if (state_bytes) *state_bytes = small_dec_bytes(np, g) + (np * 4 + 255) / 256 * 256;
    if (scratch_bytes) *scratch_bytes = small_scratch(mode, nx, ny, bd.lx, bd.ly).total;
}

int small_train_forward(const PairSpec &ps, Series<float> xs, Series<float> ys, const Band &bd,
                        double *D, void *state, hipStream_t st) {
    const SmallGeo g = small_geo(bd, ps.n_pairs);
    unsigned char *dec = (unsigned char *)state;
    float *sq = (float *)(dec + small_dec_bytes(ps.n_pairs, g));
    const dim3 grid((unsigned)((ps.n_pairs + g.P - 1) / g.P));
#define WBX_SMALL_FWD(SV, MB)                                                                    \
    case SV * 8 + MB:                                                                            \
        hipLaunchKernelGGL((k_small_train<SV, MB>), grid, dim3(64), 0, st, ps, xs, ys, g, D, sq, \
                           dec);                                                                 \
        break;
    switch (g.S * 8 + (bd.B - 1) % g.S) {
        WBX_SMALL_FWD(2, 0) WBX_SMALL_FWD(2, 1) WBX_SMALL_FWD(4, 0) WBX_SMALL_FWD(4, 1)
        WBX_SMALL_FWD(4, 2) WBX_SMALL_FWD(4, 3)
        default: return fail(WBX_EUNSUPPORTED, "band %d", bd.B);
    }
#undef WBX_SMALL_FWD
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

int small_train_backward(const PairSpec &ps, Series<float> xs, Series<float> ys, const Band &bd,
                         int64_t nx, int64_t ny, const double *G, const void *state, float *dX,
                         int64_t ldx, float *dY, int64_t ldy_, void *scratch, hipStream_t st) {
    const SmallGeo g = small_geo(bd, ps.n_pairs);
    const unsigned char *dec = (const unsigned char *)state;
    const float *sq = (const float *)(dec + small_dec_bytes(ps.n_pairs, g));
    const int mode = ps.mode == PAIR_GRID ? 0 : 1;
    const SmallScratch t = small_scratch(mode, nx, ny, bd.lx, bd.ly);
    char *sc = (char *)scratch;
    SmallGrad o;
    o.one_b = mode == 1 || ny == 1;
    o.one_a = mode == 1 || nx == 1;
    o.gx = o.one_b ? dX : (float *)(sc + t.gx);
    o.ldgx = o.one_b ? ldx : bd.lx;
    o.gy = o.one_a ? dY : (float *)(sc + t.gw);
    o.ldgy = o.one_a ? ldy_ : bd.ly;
    const dim3 grid((unsigned)ps.n_pairs);
    const size_t lds = small_lds(bd.lx, bd.ly);
    if (bd.B > 64)
        hipLaunchKernelGGL(k_small_backward<true>, grid, dim3(64), lds, st, ps, xs, ys, g, sq, G,
                           dec, o);
    else
        hipLaunchKernelGGL(k_small_backward<false>, grid, dim3(64), lds, st, ps, xs, ys, g, sq, G,
                           dec, o);
    if (!o.one_b)
        hipLaunchKernelGGL(k_sum_pairs, dim3((unsigned)((bd.lx + 63) / 64), (unsigned)nx),
                           dim3(1024), 0, st, o.gx, ny, bd.lx, dX, ldx);
    if (!o.one_a)
        launch_sum_cols(o.gy, nx, ny, bd.ly, bd.ly, (float *)(sc + t.part), dY, ldy_, st);
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

}  // namespace wbx
