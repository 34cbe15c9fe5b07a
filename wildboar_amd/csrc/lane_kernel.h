// lane_kernel.h -- FP32 DTW with one pair per lane and the band row in
// registers: the kernel template shared by the padded-band instantiations
// (lane.hip) and the exact-band ones (lane_exact.hip).
//
// For pairs that share one geometry (lx, ly, w) -- every pair of a
// pairwise/paired call on a fixed-width array, every window of one shapelet --
// each of the 64 lanes of a wave runs the whole DP of its own pair.  The row
// is kept in band coordinates (slot k <-> column j = i + k - off), where the
// three predecessors of slot k are slot k+1 of the previous row (up), slot
// k-1 of this row (left) and slot k of the previous row (diag).  Those are
// static register indices, so a fully unrolled row is BP cells of
//     d = x_i - y_j ; m = min3(up, left, diag) ; c = fma(d, d, m)
// i.e. three VALU instructions per cell and no LDS or cross-lane traffic.
//
// The y values of a row are a window y[i-off .. i-off+BP) that slides by one
// per row.  The kernel keeps a window of BP+U-1 registers, runs U rows against
// it (row u of the group reads yw[k+u]) and then shifts it by U: the shift
// costs (BP+U-1)/U moves per U*BP cells.  Columns outside [0, ly) read +inf,
// which makes their cells +inf, and the row state before row 0 is +inf with a
// 0 in slot off, which turns the first row into the reference's prefix sum.
// Padded instantiations round the band up to BP, a multiple of 8: slots >= B
// compute throw-away values and slot B is reset to +inf after every row so
// slot B-1 never sees them.  Exact instantiations (BP == B, odd B, the band
// of every pair of equal lengths) compute no padding slot and need no reset.
//
// Exact instantiations, x of a wave.  Where the 64 pairs of a wave share
// their x series (a matrix whose rows are cut into waves of 64 columns), x
// comes by scalar loads and is an SGPR operand of v_sub.  In straight-line
// rows on real data that alone is 19.6 -> 23.0e12 cells/s: one register-file
// read less per cell, which the card's power limit turns into clock (constant
// series run 17 % faster than random walks with the same instructions).
// A cell's minimum and fma are one asm block on its row register, so the row
// is updated in place; left to itself the allocator keeps a second copy of it
// (B = 75: 236 registers for 157 values) and, at B = 101, spills.
//
// WDTW (WeightedDtwMetric, distance/_elastic.pyx:3322-3341) multiplies each
// cell's squared difference by w[|i - j|]; in band coordinates |i - j| =
// |k - off| is fixed per slot, so every lane of a launch uses the same weight
// per slot: c = fma(d * d, wslot[k], m), four VALU instructions per cell.
// The per-slot weights are staged in LDS once per block and re-read every row
// (broadcast reads, no VGPRs held across rows).  Row 0 uses the reference's
// prefix-sum weights w[j - 1] (w[0] for j = 0, :893-906), a second LDS row.
#pragma once

#include <type_traits>

#include "lane_common.h"

namespace wbx {

// pen[q] is +inf for slot BP-8+q == B and -inf otherwise (uniform values), so
// max(row, pen) resets slot B without a branch.
// AD: the amercing recursion (adtw_distance, distance/_elastic.pyx:943-1008),
// m = min3(up + p, left + p, diag); row 0 runs with p = 0 (its prefix sum
// carries no penalty).
template <int BP, bool AD = false, bool WT = false>
__device__ __forceinline__ void lane_row(float (&row)[BP], const float *yw, float xi,
                                         const float (&pen)[8], float p = 0.0f,
                                         const float *wslot = nullptr) {
    float left = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < BP; ++k) {
        const float up = (k + 1 < BP) ? row[k + 1] : WBX_INF_F;
        float m;
        if constexpr (AD)
            m = fminf(fminf(up + p, left + p), row[k]);
        else
            m = fminf(fminf(up, left), row[k]);
        const float d = xi - yw[k];
        float c;
        if constexpr (WT)
            c = __builtin_fmaf(d * d, wslot[k], m);
        else
            c = __builtin_fmaf(d, d, m);
        row[k] = c;
        left = c;
    }
#pragma unroll
    for (int q = 1; q < 8; ++q) row[BP - 8 + q] = fmaxf(row[BP - 8 + q], pen[q]);
}

template <int BP, int U, bool AD = false, bool WT = false>
__device__ __forceinline__ void lane_dtw_body(PairSpec ps, Series<float> xs,
                                                 Series<float> ys, LaneGeo g, float pen_ad,
                                                 const float *__restrict__ weights,
                                                 float *__restrict__ sq) {
    constexpr int W = BP + U - 1;
    // WT: lw[0][k] row-0 weight of slot k, lw[1][k] = w[|k - off|]; slots
    // outside the band get 1 (their cells are +inf or thrown away).  A band
    // wider than the series (slopes, with the band of the series they come
    // from) has slots past the last weight; they lie outside the matrix and
    // take the last one.
    __shared__ float lw[WT ? 2 : 1][WT ? BP : 1];
    if constexpr (WT) {
        const int top = max(g.lx, g.ly) - 1;
        for (int k = threadIdx.x; k < BP; k += 64) {
            const int j = k - g.off;  // column of slot k in row 0
            lw[0][k] = (j >= 0 && k < g.B) ? weights[min(j > 0 ? j - 1 : 0, top)] : 1.0f;
            lw[1][k] = k < g.B ? weights[min(j < 0 ? -j : j, top)] : 1.0f;
        }
        __syncthreads();
    }
    const int64_t p0 = xcd_block(blockIdx.x, gridDim.x) * 64 + threadIdx.x;
    const int64_t p = p0 < ps.n_pairs ? p0 : ps.n_pairs - 1;
    int64_t a, b;
    decode_pair(ps, p, a, b);
    const float *__restrict__ X = xs.row(a);
    const float *__restrict__ Y = ys.row(b);
    const int lx = g.lx, ly = g.ly, off = g.off, B = g.B;

    float row[BP];
#pragma unroll
    for (int k = 0; k < BP; ++k) row[k] = (k == off) ? 0.0f : WBX_INF_F;
    float pen[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) pen[q] = (BP - 8 + q == B) ? WBX_INF_F : -WBX_INF_F;

    float yw[W];
#pragma unroll
    for (int m = 0; m < W; ++m) yw[m] = ldy(Y, m - off, ly);

    int i_begin = 0;
    if constexpr (WT) {
        lane_row<BP, false, true>(row, yw, X[0], pen, 0.0f, lw[0]);
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, 1 - off + W - 1, ly);
        i_begin = 1;
    }
    if constexpr (AD) {
        lane_row<BP, true, false>(row, yw, X[0], pen, 0.0f);
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, 1 - off + W - 1, ly);
        i_begin = 1;
    }
    // Leading rows one at a time so the rest is a whole number of U-groups.
    const int rem = (lx - i_begin) % U;
    for (int i = i_begin; i < i_begin + rem; ++i) {
        lane_row<BP, AD, WT>(row, yw, X[i], pen, pen_ad, WT ? lw[WT ? 1 : 0] : nullptr);
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, i + 1 - off + W - 1, ly);
    }
    if constexpr (BP >= 112 || (WT && BP > 40) || (AD && BP >= 80)) {
        // the widest class, weighted bands past 40 slots and amerced ones
        // from 80 (their weights and penalties take registers too) have none
        // left for the next group's x: each group's loads are issued at its
        // start
        for (int i0 = i_begin + rem; i0 < lx; i0 += U) {
            float xv[U], yn[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xv[u] = X[i0 + u];
                yn[u] = ldy(Y, i0 + U - off + W - U + u, ly);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if constexpr (WT) asm volatile("" ::: "memory");
                lane_row<BP, AD, WT>(row, yw + u, xv[u], pen, pen_ad,
                                         WT ? lw[WT ? 1 : 0] : nullptr);
            }
#pragma unroll
            for (int m = 0; m < W - U; ++m) yw[m] = yw[m + U];
#pragma unroll
            for (int u = 0; u < U; ++u) yw[W - U + u] = yn[u];
        }
    } else {
        // x of the current group of U rows; the loop loads the next group's
        // with the group's new window entries (columns jn .. jn + U - 1,
        // jn > 0), so nothing a row reads waits on a load issued in the same
        // group.  The lanes share the geometry: when both lie inside their
        // rows (every group but the last one or two) they are plain 16-byte
        // loads, else x is clamped into the row (never used past it) and y is
        // +inf outside it.
        static_assert(U % 4 == 0, "groups of whole 16-byte loads");
        float xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = X[min(i_begin + rem + u, lx - 1)];
        for (int i0 = i_begin + rem; i0 < lx; i0 += U) {
            float xn[U], yn[U];
            const int jn = i0 - off + W;
            if (i0 + 2 * U <= lx && jn + U <= ly) {
#pragma unroll
                for (int u = 0; u < U; u += 4) {
                    const f4a a = *(const f4a *)(X + i0 + U + u);
                    const f4a b = *(const f4a *)(Y + jn + u);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        xn[u + q] = a[q];
                        yn[u + q] = b[q];
                    }
                }
            } else {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    xn[u] = X[min(i0 + U + u, lx - 1)];
                    yn[u] = ldy(Y, jn + u, ly);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // the weights are re-read from LDS every row rather than held
                // in registers across the loop (the band row and y window
                // fill them)
                if constexpr (WT) asm volatile("" ::: "memory");
                lane_row<BP, AD, WT>(row, yw + u, xv[u], pen, pen_ad,
                                         WT ? lw[WT ? 1 : 0] : nullptr);
            }
#pragma unroll
            for (int m = 0; m < W - U; ++m) yw[m] = yw[m + U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                yw[W - U + u] = yn[u];
                xv[u] = xn[u];
            }
        }
    }

    float res = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < BP; ++k)
        if (k == g.kf) res = row[k];
    if (p0 < ps.n_pairs) put_cost(ps, p0, res, sq);
}

// Plain DTW on padded bands is held to two waves per SIMD like the exact
// kernels (at 104 and 112 slots the allocator would take one wave's worth);
// the weighted and amerced variants need more registers than two waves have.
template <int BP, int U, bool AD = false, bool WT = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(AD || WT ? 1 : 2))) void
k_lane_dtw(PairSpec ps, Series<float> xs, Series<float> ys, LaneGeo g, float pen_ad,
           const float *__restrict__ weights, float *__restrict__ sq) {
    lane_dtw_body<BP, U, AD, WT>(ps, xs, ys, g, pen_ad, weights, sq);
}

// One row of an exact band (m = min3(up, left, diag), c = fma(d, d, m)
// in the row register itself; the outermost slots lack one input).
template <int B>
__device__ __forceinline__ void exact_row(float (&row)[B], const float *yw, float xi) {
    float left = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < B; ++k) {
        const float d = xi - yw[k];
        if (k == 0)
            asm("v_min_f32 %0, %1, %0\n\tv_fmac_f32 %0, %2, %2"
                : "+v"(row[k])
                : "v"(row[1]), "v"(d));
        else if (k + 1 < B)
            asm("v_min3_f32 %0, %1, %2, %0\n\tv_fmac_f32 %0, %3, %3"
                : "+v"(row[k])
                : "v"(row[k + 1]), "v"(left), "v"(d));
        else
            asm("v_min_f32 %0, %1, %0\n\tv_fmac_f32 %0, %2, %2"
                : "+v"(row[k])
                : "v"(left), "v"(d));
        left = row[k];
    }
}

// The same for WDTW between series of equal length: slot k weighs w[|k - off|]
// with off = (B - 1) / 2, the same for every lane and row, so the (B + 1) / 2
// weights sit in SGPRs and the cell is c = fma(w, d * d, m), four VALU
// instructions.  ROW0: the prefix sum's weights, w[j - 1] at column j > 0,
// w[0] at column 0 (columns below 0 are +inf whatever their weight).
template <int B, bool ROW0>
__device__ __forceinline__ void exact_row_w(float (&row)[B], const float *yw, float xi,
                                            const float (&w)[(B + 1) / 2]) {
    constexpr int off = (B - 1) / 2;
    float left = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < B; ++k) {
        constexpr int top = (B + 1) / 2 - 1;
        const int a = k < off ? off - k : k - off;
        const int e = !ROW0 ? a : (k > off ? a - 1 : 0);
        const float wk = w[e < top ? e : top];
        float d = xi - yw[k];
        if (k == 0)
            asm("v_min_f32 %0, %2, %0\n\tv_mul_f32 %1, %1, %1\n\tv_fmac_f32 %0, %3, %1"
                : "+v"(row[k]), "+v"(d)
                : "v"(row[1]), "s"(wk));
        else if (k + 1 < B)
            asm("v_min3_f32 %0, %2, %3, %0\n\tv_mul_f32 %1, %1, %1\n\tv_fmac_f32 %0, %4, %1"
                : "+v"(row[k]), "+v"(d)
                : "v"(row[k + 1]), "v"(left), "s"(wk));
        else
            asm("v_min_f32 %0, %2, %0\n\tv_mul_f32 %1, %1, %1\n\tv_fmac_f32 %0, %3, %1"
                : "+v"(row[k]), "+v"(d)
                : "v"(left), "s"(wk));
        left = row[k];
    }
}

// x of a wave that shares one series: constant address space, so the loads
// are scalar.
typedef const float __attribute__((address_space(4))) *cfloat;

// Exact bands, plain DTW.  XU: grid pairs, wave blk runs row blk / nb against
// columns 64 (blk % nb) .. + 63, nb = ceil(ny / 64); else wave blk runs pairs
// 64 blk .. + 63 of any kind, x per lane.  Two waves per SIMD (at most 256
// registers) keep the VALU busy -- one wave issues about half as often.
// Bound by VALU issue and the clock that power allows; groups of 8 rows move
// the window half as often as groups of 4 (13 instead of 26 moves a row at
// B = 101), longer groups gain nothing.  2000 x 2000 x 512 on one box, x per
// lane -> XU: B = 23 2.92 -> 2.67 ms, B = 49 5.52 -> 5.23, B = 75 8.83 -> 8.10,
// B = 101 12.02 -> 10.73, B = 111 13.05 -> 11.70.
// WT: WDTW (equal lengths, XU; weights: at least (B + 1) / 2 values, which
// lane_exact_w_waves sees to).  1000 x 1000 x 256, B = 49: 1205 us on the
// group kernel, 873 us.
template <int B, int U, bool XU, bool WT = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_lane_dtw_exact(
    PairSpec ps, Series<float> xs, Series<float> ys, LaneGeo g,
    const float *__restrict__ weights, float *__restrict__ sq) {
    constexpr int W = B + U - 1;
    static_assert(U % 4 == 0, "groups of whole 16-byte loads");
    const int lane = threadIdx.x;
    const int lx = g.lx, ly = g.ly, off = g.off;
    int64_t a, b, p0;
    bool live;
    if constexpr (XU) {
        const unsigned ny = (unsigned)ps.ny, nb = (ny + 63) / 64;
        const unsigned blk = (unsigned)xcd_block(blockIdx.x, gridDim.x);
        const unsigned ra = (unsigned)__builtin_amdgcn_readfirstlane((int)(blk / nb));
        const unsigned j = (blk - ra * nb) * 64 + lane;
        live = j < ny;
        a = ra;
        b = live ? j : ny - 1;
        p0 = a * ps.ny + j;
    } else {
        p0 = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
        live = p0 < ps.n_pairs;
        decode_pair(ps, live ? p0 : ps.n_pairs - 1, a, b);
    }
    using XP = typename std::conditional<XU, cfloat, const float *>::type;
    const XP X = (XP)xs.row(a);
    const float *__restrict__ Y = ys.row(b);

    float row[B];
#pragma unroll
    for (int k = 0; k < B; ++k) row[k] = (k == off) ? 0.0f : WBX_INF_F;
    // the first window, 8 loads at a time: all of them in flight would need
    // an address register pair each
    float yw[W];
#pragma unroll
    for (int m = 0; m < W; ++m) {
        yw[m] = ldy(Y, m - off, ly);
        if ((m & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    float w[WT ? (B + 1) / 2 : 1];
    if constexpr (WT) {
        const cfloat ws = (cfloat)weights;
#pragma unroll
        for (int q = 0; q < (B + 1) / 2; ++q) w[q] = ws[q];
    }
    auto one_row = [&](const float *y, float xi, auto row0) {
        if constexpr (WT)
            exact_row_w<B, decltype(row0)::value>(row, y, xi, w);
        else
            exact_row<B>(row, y, xi);
    };
    // leading rows one at a time so the rest is a whole number of groups
    // (WDTW: row 0 among them, its weights differ)
    int i_begin = 0;
    if constexpr (WT) {
        one_row(yw, X[0], std::true_type());
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, 1 - off + W - 1, ly);
        i_begin = 1;
    }
    const int rem = i_begin + (lx - i_begin) % U;
    for (int i = i_begin; i < rem; ++i) {
        one_row(yw, X[i], std::false_type());
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, i + 1 - off + W - 1, ly);
    }
    // x of the current group; the loop loads the next group's with the
    // group's new window entries (columns jn .. jn + U - 1, jn > 0) before
    // the rows run.  The lanes share the geometry: when both lie inside their
    // rows (every group but the last one or two) they are plain loads, else x
    // is clamped into the row (never used past it) and y is +inf outside it.
    float xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = X[min(rem + u, lx - 1)];
    // the loads above are waited for here: left in flight, the wait for them
    // inside the loop would cover the group's own loads too
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    for (int i0 = rem; i0 < lx; i0 += U) {
        float xn[U], yn[U];
        const int jn = i0 - off + W;
        if (i0 + 2 * U <= lx && jn + U <= ly) {
#pragma unroll
            for (int u = 0; u < U; u += 4) {
                const f4a bv = *(const f4a *)(Y + jn + u);
                if constexpr (XU) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) xn[u + q] = X[i0 + U + u + q];
                } else {
                    const f4a av = *(const f4a *)(X + i0 + U + u);
#pragma unroll
                    for (int q = 0; q < 4; ++q) xn[u + q] = av[q];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) yn[u + q] = bv[q];
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xn[u] = X[min(i0 + U + u, lx - 1)];
                yn[u] = ldy(Y, jn + u, ly);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) one_row(yw + u, xv[u], std::false_type());
#pragma unroll
        for (int m = 0; m < W - U; ++m) yw[m] = yw[m + U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            yw[W - U + u] = yn[u];
            xv[u] = xn[u];
        }
    }
    float res = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k == g.kf) res = row[k];
    if (live) put_cost(ps, p0, res, sq);
}

}  // namespace wbx
