// lane_train.h -- the lane-per-pair forward of the differentiable DTW: the
// kernel template shared by the padded-band instantiations (train.hip) and
// the exact-band ones (train_exact.hip).
#pragma once

#include <type_traits>

#include "lane_common.h"

namespace wbx {

// One cell, on its row register, which holds the diagonal before and the cost
// after (so the row is updated in place; as separate values the allocator
// keeps a second copy of it):
//   m = min3(up, left, diag)
//   m - diag, m - up                 negative unless equal, then +0
//   c = fma(x - y, x - y, m)
//   pd = 2 pd + sign, pu = 2 pu + sign   alignbit shifts each sign bit in
// so a clear bit says that the minimum came from there.  Seven VALU
// instructions, three of them subtractions that issue beside another wave's
// minimum or shift: 17.1 cycles a cell with x in an SGPR, 22.5 with two
// compares into SGPR masks and two add-with-carry (x in a VGPR 17.9).
// Costs that are not finite (then neither is the distance, and the gradient 0 or
// NaN) are not equal even to themselves here: +inf - +inf has its sign set.  The
// walk stays inside the band without their bits.
// The two shifts stay last: gfx950 wants two instructions between the fma and a
// DPP move that reads c (the strips of train_small.hip), and the compiler
// does not look into the block.
// XU: x is the same for the whole wave, an SGPR operand.
#define WBX_TRAIN_CELL(X)                                                                    \
    asm("v_min3_f32 %[t], %[up], %[left], %[c]\n\t"                                          \
        "v_sub_f32_e32 %[a], %[t], %[c]\n\t"                                                 \
        "v_sub_f32_e32 %[b], %[t], %[up]\n\t"                                                \
        "v_sub_f32_e32 %[d], %[x], %[y]\n\t"                                                 \
        "v_fma_f32 %[c], %[d], %[d], %[t]\n\t"                                               \
        "v_alignbit_b32 %[pd], %[pd], %[a], 31\n\t"                                          \
        "v_alignbit_b32 %[pu], %[pu], %[b], 31"                                              \
        : [c] "+v"(c), [pd] "+v"(pd), [pu] "+v"(pu), [d] "=&v"(d), [t] "=&v"(t), [a] "=&v"(a), \
          [b] "=&v"(b)                                                                       \
        : [left] "v"(left), [up] "v"(up), [x] X(x), [y] "v"(y))
template <bool XU>
__device__ __forceinline__ void train_cell(float &c, float up, float left, float x, float y,
                                           uint32_t &pd, uint32_t &pu) {
    float d, t, a, b;
    if constexpr (XU)
        WBX_TRAIN_CELL("s");
    else
        WBX_TRAIN_CELL("v");
}
#undef WBX_TRAIN_CELL

// EX: the band is exactly BP slots, none needs a reset after the row.
template <int BP, bool EX, bool XU>
__device__ __forceinline__ void train_row(float (&row)[BP], const float *yw, float xi,
                                          const float (&pen)[8], uint32_t *pd, uint32_t *pu) {
    float left = WBX_INF_F;
#pragma unroll
    for (int k = 0; k < BP; ++k) {
        const float up = (k + 1 < BP) ? row[k + 1] : WBX_INF_F;
        train_cell<XU>(row[k], up, left, xi, yw[k], pd[k >> 5], pu[k >> 5]);
        left = row[k];
    }
    if constexpr (!EX) {
#pragma unroll
        for (int q = 1; q < 8; ++q) row[BP - 8 + q] = fmaxf(row[BP - 8 + q], pen[q]);
    }
}

// Plane words of wave v, row i, lane l: 2 NW words starting at
// dirs[((v * lx + i) * 64 + l) * 2 NW], as (diag word w, up word w) pairs, so a
// lane's row is one contiguous piece and a wave's row is 64 of them in a row.
__device__ __forceinline__ int64_t plane_base(int64_t wave, int lx, int i, int nw2, int lane) {
    return (((int64_t)wave * lx + i) * 64 + lane) * nw2;
}

template <int BP>
__device__ __forceinline__ void store_planes(uint32_t *__restrict__ dirs, int64_t wave, int lane,
                                             int lx, int i, uint32_t (&pd)[(BP + 31) / 32],
                                             uint32_t (&pu)[(BP + 31) / 32]) {
    constexpr int NW = (BP + 31) / 32;
    uint2 *d = (uint2 *)(dirs + plane_base(wave, lx, i, 2 * NW, lane));
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        // as "came from there" bits: the clear ones of the word's slots
        constexpr int last = BP - 32 * (NW - 1);
        const uint32_t mask = w + 1 < NW || last == 32 ? ~0u : (1u << last) - 1u;
        d[w] = make_uint2(pd[w] ^ mask, pu[w] ^ mask);
        pd[w] = 0u;
        pu[w] = 0u;
    }
}

// Waves per SIMD that the registers (row and window: 2 BP, and x where it is
// not an SGPR) reach without spills.
constexpr int train_waves(int slots) {
    return slots <= 49 ? 4 : slots <= 63 ? 3 : slots <= 99 ? 2 : 1;
}

// One pair per lane, wave v runs pairs 64 v .. + 63.  EX: band of exactly BP
// slots; XU: the pairs of every wave share their x series (a matrix whose
// column count is a multiple of 64), read by scalar loads.  262,144 pairs of
// 256, B = 49: 711 us padded to 56 slots with compares, 600 us exact, 513 us
// with the sign-bit cell and a shared x.
template <int BP, int U, bool EX, bool XU>
__global__ __launch_bounds__(64) __attribute__((
    amdgpu_waves_per_eu(train_waves(XU ? BP : BP + 4)))) void
k_lane_train(PairSpec ps, Series<float> xs, Series<float> ys, LaneGeo g, float *__restrict__ sq,
             uint32_t *__restrict__ dirs) {
    constexpr int W = BP + U - 1;
    constexpr int NW = (BP + 31) / 32;
    const int lane = threadIdx.x;
    const int64_t wave = blockIdx.x;
    const int64_t p0 = wave * 64 + lane;
    const int64_t p = p0 < ps.n_pairs ? p0 : ps.n_pairs - 1;
    int64_t a, b;
    decode_pair(ps, p, a, b);
    typedef const float __attribute__((address_space(4))) *cfp;
    using XP = typename std::conditional<XU, cfp, const float *>::type;
    const XP X = (XP)xs.row(XU ? __builtin_amdgcn_readfirstlane((int)a) : a);
    const float *__restrict__ Y = ys.row(b);
    const int lx = g.lx, ly = g.ly, off = g.off, B = g.B;

    float row[BP];
#pragma unroll
    for (int k = 0; k < BP; ++k) row[k] = (k == off) ? 0.0f : WBX_INF_F;
    float pen[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) pen[q] = (BP - 8 + q == B) ? WBX_INF_F : -WBX_INF_F;
    uint32_t pd[NW], pu[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) pd[w] = pu[w] = 0u;
    float yw[W];
#pragma unroll
    for (int m = 0; m < W; ++m) {
        yw[m] = ldy(Y, m - off, ly);
        if ((m & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);

    const int rem = lx % U;
    for (int i = 0; i < rem; ++i) {
        train_row<BP, EX, XU>(row, yw, X[i], pen, pd, pu);
        store_planes<BP>(dirs, wave, lane, lx, i, pd, pu);
#pragma unroll
        for (int m = 0; m < W - 1; ++m) yw[m] = yw[m + 1];
        yw[W - 1] = ldy(Y, i + 1 - off + W - 1, ly);
    }
    float xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = X[rem + u < lx ? rem + u : lx - 1];
    for (int i0 = rem; i0 < lx; i0 += U) {
        float xn[U], yn[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int inext = i0 + U + u;
            xn[u] = X[inext < lx ? inext : lx - 1];
            yn[u] = ldy(Y, i0 + U - off + W - U + u, ly);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            train_row<BP, EX, XU>(row, yw + u, xv[u], pen, pd, pu);
            store_planes<BP>(dirs, wave, lane, lx, i0 + u, pd, pu);
        }
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
    for (int k = 0; k < BP; ++k)
        if (k == g.kf) res = row[k];
    if (p0 < ps.n_pairs) sq[p0] = res;
}

// Exact bands (train_exact.hip, odd B = 9 .. 111).
int launch_lane_train_exact(const PairSpec &ps, Series<float> xs, Series<float> ys,
                            const LaneGeo &g, float *sq, uint32_t *dirs, hipStream_t st);

}  // namespace wbx
