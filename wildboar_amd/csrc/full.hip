// full.hip -- DTW when the band covers the whole matrix (w >= min(lx, ly):
// the reference's default r = 1, DtwMetric, distance/_elastic.pyx:3126-3217),
// for calls whose pairs share one geometry, in matrix coordinates.
//
// With the whole matrix in the band there is no diagonal band to follow, so
// lanes own columns: lane q of a group owns columns [q S, q S + S) (the y
// values stay in registers for the whole pair; columns >= ly read +inf and
// never feed a column < ly) and works on row s - q at step s.  A cell needs
//   up    D(i-1, j)    -- the lane's own previous row,
//   left  D(i, j-1)    -- its previous column, or for its first column lane
//                         q-1's last column of the same row, made one step
//                         earlier (DPP wave_shr:1),
//   diag  D(i-1, j-1)  -- the previous row's left neighbour: for the first
//                         column the value lane q-1 sent one step before.
// Nothing flows right to left, so one DPP move per step suffices (the band-
// coordinate kernels need two, and half their slots lie outside the matrix
// at r = 1).  D(-1, -1) = 0 starts the path; row and column -1 are +inf.
// Groups run in lockstep; steps before a lane's row 0 and after its row
// lx - 1 keep its state (a select per cell), the steps between do not.
//
// Cell arithmetic: float32 c = fma(d, d, min3(up, left, diag)); float64 the
// reference's c = min(min(up, left), diag) + d * d, contraction off
// (bit-exact: _elastic.pyx:893-940 with w = 1).
#pragma clang fp contract(off)

#include <type_traits>

#include "wbx_internal.h"

namespace wbx {

namespace {

template <typename T>
__device__ __forceinline__ T finf();
template <>
__device__ __forceinline__ float finf<float>() {
    return WBX_INF_F;
}
template <>
__device__ __forceinline__ double finf<double>() {
    return WBX_INF_D;
}

__device__ __forceinline__ float from_left(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(WBX_INF_F), __float_as_int(v),
                                                      0x138, 0xF, 0xF, false));
}
__device__ __forceinline__ double from_left(double v) {
    const int2 b = *reinterpret_cast<const int2 *>(&v);
    int2 o;
    o.x = __builtin_amdgcn_update_dpp(0, b.x, 0x138, 0xF, 0xF, false);
    o.y = __builtin_amdgcn_update_dpp(0x7ff00000, b.y, 0x138, 0xF, 0xF, false);
    return *reinterpret_cast<const double *>(&o);
}

__device__ __forceinline__ float fcell(float up, float left, float diag, float x, float y) {
    const float d = x - y;
    return __builtin_fmaf(d, d, fminf(fminf(up, left), diag));
}
__device__ __forceinline__ double fcell(double up, double left, double diag, double x, double y) {
    const double d = x - y;
    return __builtin_fmin(__builtin_fmin(up, left), diag) + d * d;
}

template <typename T, int S>
struct FLane {
    T row[S];  // D(r - 1, c0 + m) before row r, D(r, c0 + m) after
    T yv[S];
    T dg;      // D(r - 1, c0 - 1): the left value received one step earlier
    T l;       // D(r, c0 + S - 1) of the lane's last row
    int r;
    bool first;
};

template <typename T, int S, bool SEL>
__device__ __forceinline__ void fstep(FLane<T, S> &L, T x, int lx) {
    T Lin = from_left(L.l);
    Lin = L.first ? finf<T>() : Lin;
    const bool act = !SEL || (unsigned)L.r < (unsigned)lx;
    T diag = L.dg;
    T left = Lin;
#pragma unroll
    for (int m = 0; m < S; ++m) {
        const T up = L.row[m];
        const T c = fcell(up, left, diag, x, L.yv[m]);
        diag = up;
        L.row[m] = SEL ? (act ? c : up) : c;
        left = c;
    }
    if (SEL) {
        L.dg = act ? Lin : L.dg;
    } else {
        L.dg = Lin;
    }
    L.l = L.row[S - 1];
    L.r += 1;
}

template <typename T>
__device__ __forceinline__ T fldx(const T *__restrict__ X, int i, int lx) {
    return X[i < 0 ? 0 : (i >= lx ? lx - 1 : i)];
}

// Waves per SIMD the register allocation is held to: float64 lanes of 21 to 24
// columns fit three waves' 168 registers without spills (184 otherwise).
template <typename T, int S>
constexpr int full_waves() {
    return sizeof(T) == 8 && S >= 21 && S <= 24 ? 3 : 1;
}

template <typename T, int S, int U>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(full_waves<T, S>()))) void
k_full_dtw(PairSpec ps, Series<T> xs, Series<T> ys, FullGeo g, T *__restrict__ sq) {
    const int lane = threadIdx.x;
    const int gi = lane / g.n;
    const int q = lane - gi * g.n;
    const int64_t p = (int64_t)blockIdx.x * g.P + gi;
    const bool valid = gi < g.P && p < ps.n_pairs;
    int64_t a = 0, b = 0;
    if (valid) decode_pair(ps, p, a, b);
    const T *__restrict__ X = xs.row(a);
    const T *__restrict__ Y = ys.row(b);
    const int lx = g.lx, ly = g.ly;
    const int c0 = q * S;

    FLane<T, S> L;
#pragma unroll
    for (int m = 0; m < S; ++m) {
        const int j = c0 + m;
        const T v = Y[j < ly ? j : ly - 1];
        L.yv[m] = j < ly ? v : finf<T>();
        L.row[m] = finf<T>();
    }
    L.first = q == 0;
    L.dg = q == 0 ? (T)0 : finf<T>();  // D(-1, -1) = 0
    L.l = finf<T>();
    L.r = -q;
    // Steps go in groups of U, the next group's x values loaded during the
    // current one; steps with a lane outside its rows (the first n - 1 and
    // those past row lx - 1 of lane 0) keep that lane's state through selects.
    // They go in groups too, except in the float64 lanes held to three waves
    // (whose registers that would spill): one at a time.
    constexpr bool kEdgeGroups = full_waves<T, S>() == 1;
    const int steps = lx + g.n - 1;
    int s = 0;
    if constexpr (!kEdgeGroups) {
        for (; s < g.n - 1; ++s) fstep<T, S, true>(L, fldx(X, L.r, lx), lx);
        const int rem = s < lx ? (lx - s) % U : 0;
        for (int e = 0; e < rem; ++e, ++s) fstep<T, S, false>(L, fldx(X, L.r, lx), lx);
    }
    T xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = fldx(X, L.r + u, lx);
    auto group = [&](auto edge) {
        T xn[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xn[u] = fldx(X, L.r + U + u, lx);
#pragma unroll
        for (int u = 0; u < U; ++u) fstep<T, S, decltype(edge)::value>(L, xv[u], lx);
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = xn[u];
    };
    if constexpr (kEdgeGroups)
        for (; s < g.n - 1; s += U) group(std::true_type());
    for (; s + U <= lx; s += U) group(std::false_type());
    if constexpr (kEdgeGroups)
        for (; s < steps; s += U) group(std::true_type());
    else
        for (; s < steps; ++s) fstep<T, S, true>(L, fldx(X, L.r, lx), lx);

    const int jf = ly - 1;
    if (valid && jf >= c0 && jf < c0 + S) {
        T res = finf<T>();
#pragma unroll
        for (int m = 0; m < S; ++m)
            if (c0 + m == jf) res = L.row[m];
        put_cost(ps, p, res, sq);
    }
}

constexpr int kFullS32[] = {4,  6,  8,  10, 12, 14, 15, 16, 17, 18, 19, 20,
                            21, 22, 23, 24, 25, 26, 27, 28, 30, 32};
constexpr int kFullS64[] = {4,  6,  8,  10, 12, 14, 15, 16, 17, 18, 19,
                            20, 21, 22, 23, 24, 25, 26, 27, 28};

template <typename T, int S>
void launch_full_one(const PairSpec &ps, Series<T> xs, Series<T> ys, const FullGeo &g, T *sq,
                     hipStream_t st) {
    const dim3 grid((unsigned)((ps.n_pairs + g.P - 1) / g.P));
    hipLaunchKernelGGL((k_full_dtw<T, S, (S <= 8 ? 8 : 4)>), grid, dim3(64), 0, st, ps, xs, ys, g, sq);
}

}  // namespace

// Columns per lane S and lanes per pair n = ceil(ly / S) <= 64: the compiled S
// with the smallest time for n_pairs pairs.  Large calls want the cells of a
// wave step to be matrix cells (64 / n pairs a wave, n S columns for ly, n - 1
// steps of fill and drain), small ones few columns in turn.  The figures are
// the group kernel's kind (pair_launch_ns), measured on series of 275: 50
// pairs float64 81 us at S = 24, 36 us at S = 6; 400000 pairs of 100, 844 us
// at S = 24, 707 us at S = 26.
bool full_plan(int lx, int ly, int64_t n_pairs, bool fp64, FullGeo *g) {
    const int *tab = fp64 ? kFullS64 : kFullS32;
    const int nt = fp64 ? (int)(sizeof(kFullS64) / sizeof(int))
                        : (int)(sizeof(kFullS32) / sizeof(int));
    double best = 0.0;
    for (int t = 0; t < nt; ++t) {
        const int S = tab[t];
        const int n = (ly + S - 1) / S;
        if (n > 64) continue;
        const int P = 64 / n;
        const double time =
            pair_launch_ns((n_pairs + P - 1) / P, lx + n - 1, fp64 ? 35.0 + 10.0 * S : 30.0 + 5.2 * S,
                           fp64 ? 22.0 + 9.5 * S : 17.0 + 3.25 * S);
        if (best == 0.0 || time < best) {
            best = time;
            g->S = S;
            g->n = n;
            g->P = P;
        }
    }
    g->lx = lx;
    g->ly = ly;
    return best > 0.0;
}

template <typename T>
int launch_full_dtw(const PairSpec &ps, Series<T> xs, Series<T> ys, T *sq, hipStream_t st) {
    if (ps.n_pairs <= 0) return WBX_OK;
    if (xs.lens || ys.lens) return fail(WBX_EUNSUPPORTED, "full kernel: needs one geometry");
    FullGeo g{};
    const bool dbl = std::is_same<T, double>::value;
    if (!full_plan(xs.len, ys.len, ps.n_pairs, dbl, &g))
        return fail(WBX_EUNSUPPORTED, "full kernel: %d columns", ys.len);
    switch (g.S) {
#define WBX_F(SV) \
    case SV: launch_full_one<T, SV>(ps, xs, ys, g, sq, st); break;
        WBX_F(4) WBX_F(6) WBX_F(8) WBX_F(10) WBX_F(12) WBX_F(14) WBX_F(15) WBX_F(16) WBX_F(17)
        WBX_F(18) WBX_F(19) WBX_F(20) WBX_F(21) WBX_F(22) WBX_F(23) WBX_F(24) WBX_F(25) WBX_F(26)
        WBX_F(27) WBX_F(28)
#undef WBX_F
        case 30:
        case 32:
            if constexpr (!std::is_same<T, double>::value) {
                if (g.S == 30)
                    launch_full_one<T, 30>(ps, xs, ys, g, sq, st);
                else
                    launch_full_one<T, 32>(ps, xs, ys, g, sq, st);
                break;
            }
            [[fallthrough]];
        default: return fail(WBX_EUNSUPPORTED, "full kernel: %d columns per lane", g.S);
    }
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

template int launch_full_dtw<float>(const PairSpec &, Series<float>, Series<float>, float *,
                                    hipStream_t);
template int launch_full_dtw<double>(const PairSpec &, Series<double>, Series<double>, double *,
                                     hipStream_t);

}  // namespace wbx
