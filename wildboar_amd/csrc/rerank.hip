// rerank.hip -- certified selection of the pairs an FP32 result cannot decide.
//
// An FP32 cell is c = fl(fma(d, d, m)) with d = fl(x - y) (or fl(fl(d*d)*w)+m
// in the plain FP32 kernel).  All terms are non-negative and min is exact, so
// by induction over the DP every computed cost satisfies
//     (1-u)^K C - A  <=  c  <=  (1+u)^K C + A,    K = lx + ly + 2 (+2 WDTW)
// with u = 2^-24, C the exact real cost and A = P * 4 u M^2 (1+u)^K the
// contribution of rounding float64 inputs to float32 (M = max |input|,
// P = lx + ly - 1 path cells; A = 0 when the inputs already are float32).
// The reference's float64 value obeys the same bound with u = 2^-53.  This
// gives for every pair an interval [lo, hi] that contains the reference's
// sqrt'ed float64 distance.
//
// argmin (heap replay of _ArgMinBatch, distance/_cdistance.pyx:1318-1345):
// pair j can be pushed only if d_j < T_j, where T_j is the k-th smallest of
// d_0..d_{j-1}; T_j <= the k-th smallest hi over j' < j.  So every j with
// lo_j < that running k-th smallest hi is a candidate and nothing else can be
// pushed.  Candidates are re-evaluated exactly in FP64 and the replay runs over
// each row's candidates in column order; the others are never pushed.
#include "wbx_internal.h"

namespace wbx {

ErrBound make_err_bound(int lx, int ly, int weighted, double absmax, int inputs_exact) {
    const double u = 5.9604644775390625e-08;  // 2^-24
    const double u64 = 1.1102230246251565e-16;
    const int P = lx + ly - 1;
    const double K = (double)P + 3.0 + (weighted ? 2.0 : 0.0);
    ErrBound eb;
    eb.e_up = exp(K * log1p(u)) * (1.0 + 1e-12);
    eb.e_dn = exp(K * log1p(-u)) * (1.0 - 1e-12);
    eb.A = inputs_exact ? 0.0 : (double)P * 4.0 * u * absmax * absmax * eb.e_up * (1.0 + 1e-12);
    eb.e64 = (K + 8.0) * u64 * 1.01;
    return eb;
}

__device__ __forceinline__ void dist_bounds(float c, const ErrBound &eb, double &lo, double &hi) {
    if (!(c < WBX_INF_F)) {
        lo = 0.0;
        hi = WBX_INF_D;
        return;
    }
    const double cd = (double)c;
    double clo = cd - eb.A;
    clo = clo > 0.0 ? clo / eb.e_up : 0.0;
    const double chi = (cd + eb.A) / eb.e_dn;
    lo = sqrt(clo * (1.0 - eb.e64)) * (1.0 - 4.4e-16);
    hi = sqrt(chi * (1.0 + eb.e64)) * (1.0 + 4.4e-16);
}

constexpr int KMAX = 32;

__device__ __forceinline__ double lane_value(double v, int q) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, q);
    const uint64_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), q);
    return __builtin_bit_cast(double, hi << 32 | lo);
}

// One wave per x row.  The k smallest hi values so far sit in lanes 0 .. k - 1
// in ascending order (+inf where there are fewer), T is the k-th.  64 costs
// are read together; T only falls, so a cost whose lo is not below the T at
// the start of its 64 can neither be a candidate nor change T (hi >= lo), and
// one comparison with the cost at which lo reaches T drops it.  The others
// are taken in column order, which selects what a scan of the row selects.
// A row's candidates are one bit per column in `words` (the lane that stores a
// word reads it back).  When the `per` rows of a wave are done it reserves
// their places in the pair list with one atomic and writes them there, each
// row's in column order (the order of the rows in the list is free).
//
// Bound by the latency of the loads and of the selection steps (a row needs
// about k ln(ny / k) of them).  500 rows of 4000, k = 5: 40 us.  One lane per
// row, in two passes with a division and a square root for every cost, took 2 x
// 2390 us there: 8 waves, their loads ny floats apart.  The atomics of a launch
// run one after the other, 13 ns each: with one per row 100000 rows of 10
// took 1.3 ms for them alone.
__global__ __launch_bounds__(64) void k_argmin_candidates(
    const float *__restrict__ sq, int64_t nx, int64_t ny, int k, int per, ErrBound eb,
    const unsigned *__restrict__ absmax_bits, uint64_t *words, int64_t *__restrict__ offs,
    int64_t *__restrict__ counts, unsigned long long *__restrict__ total,
    int32_t *__restrict__ pa, int32_t *__restrict__ pb) {
    const int64_t i0 = (int64_t)blockIdx.x * per;
    const int rows = (int)(nx - i0 < per ? nx - i0 : per);
    const int lane = threadIdx.x;
    if (absmax_bits) {  // A was made for |x| <= 1
        const double m = (double)__uint_as_float(*absmax_bits);
        eb.A *= m * m;
    }
    const int64_t nw = (ny + 63) / 64;
    int64_t own_cnt = 0;  // of row i0 + lane
    for (int e = 0; e < rows; ++e) {
        const float *__restrict__ row = sq + (i0 + e) * ny;
        uint64_t *wrow = words + (i0 + e) * nw;
        // the starting +inf goes through a vector register: as a constant in a
        // scalar pair the compiler writes it with one 32-bit literal, which is 0
        double top = WBX_INF_D;
        asm volatile("" : "+v"(top));
        double T = lane_value(top, 0), cth = T;
        int64_t cnt = 0;
        constexpr int UC = 4;  // groups of 64 costs in flight
        for (int64_t w0 = 0; w0 < nw; w0 += UC) {
            float cv[UC];
#pragma unroll
            for (int u = 0; u < UC; ++u) {
                const int64_t j = (w0 + u) * 64 + lane;
                cv[u] = j < ny ? row[j] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < UC; ++u) {
                const int64_t j = (w0 + u) * 64 + lane;
                if (w0 + u >= nw) break;  // uniform
                const float c = cv[u];
                // a cost that is not finite has lo = 0
                uint64_t mask = __ballot(j < ny && (!(c < WBX_INF_F) || (double)c < cth));
                uint64_t word = 0;
                if (mask) {
                    double lo, hi;
                    dist_bounds(c, eb, lo, hi);
                    while (mask) {
                        const int q = __builtin_ctzll(mask);
                        mask &= mask - 1;
                        if (lane_value(lo, q) < T) word |= (uint64_t)1 << q;
                        const double hq = lane_value(hi, q);
                        if (hq < T) {
                            const int pos =
                                __popcll(__ballot(lane < k && top <= hq));
                            const double below = __shfl_up(top, 1);
                            top = lane < pos ? top : lane == pos ? hq : below;
                            T = lane_value(top, k - 1);
                        }
                    }
                    // lo(c) < T only if c is below this
                    cth = (T * T / (1.0 - eb.e64) * eb.e_up + eb.A) * (1.0 + 1e-9);
                    cnt += __popcll(word);
                }
                if (lane == (int)((w0 + u) & 63)) wrow[w0 + u] = word;
            }
        }
        if (lane == e) own_cnt = cnt;
    }
    int64_t inc = own_cnt;  // inclusive scan over the rows
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    unsigned long long base = 0;
    if (lane == 63) base = atomicAdd(total, (unsigned long long)inc);
    base = (unsigned long long)__shfl((long long)base, 63);
    if (lane < rows) {
        offs[i0 + lane] = (int64_t)base + inc - own_cnt;
        counts[i0 + lane] = own_cnt;
    }
    for (int e = 0; e < rows; ++e) {
        const uint64_t *wrow = words + (i0 + e) * nw;
        for (int64_t w0 = 0; w0 < nw; w0 += 64) {
            const int64_t wi = w0 + lane;
            uint64_t word = wi < nw ? wrow[wi] : 0;  // stored by this lane
            const int own = __popcll(word);
            int pre = own;  // inclusive scan over the lanes
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(pre, d);
                if (lane >= d) pre += o;
            }
            unsigned long long q = base + (unsigned long long)(pre - own);
            while (word) {
                const int z = __builtin_ctzll(word);
                word &= word - 1;
                pa[q] = (int32_t)(i0 + e);
                pb[q] = (int32_t)(wi * 64 + z);
                ++q;
            }
            base += (unsigned long long)__shfl(pre, 63);
        }
    }
}

size_t argmin_words_bytes(int64_t nx, int64_t ny) {
    return (size_t)nx * (size_t)((ny + 63) / 64) * 8;
}

int launch_argmin_candidates(const float *sq, int64_t nx, int64_t ny, int k, const ErrBound &eb,
                             const unsigned *absmax_bits, void *words, int64_t *offs,
                             int64_t *counts, unsigned long long *total, int32_t *pa, int32_t *pb,
                             int64_t *total_host, hipStream_t st) {
    if (k > KMAX) return fail(WBX_EUNSUPPORTED, "certified argmin supports k <= %d", KMAX);
    int rc = launch_fill_i32((int *)total, 2, 0, st);
    if (rc) return rc;
    // a row a wave while four waves per SIMD do, at most 64 (a lane has a row's
    // count)
    const int64_t want = (nx + 4095) / 4096;
    const int per = (int)(want < 64 ? want : 64);
    hipLaunchKernelGGL(k_argmin_candidates, dim3((unsigned)((nx + per - 1) / per)), dim3(64), 0,
                       st, sq, nx, ny, k, per, eb, absmax_bits, (uint64_t *)words, offs, counts,
                       total, pa, pb);
    WBX_HIP_CHECK(hipGetLastError());
    WBX_HIP_CHECK(hipMemcpyAsync(total_host, total, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    WBX_HIP_CHECK(hipStreamSynchronize(st));
    return WBX_OK;
}

}  // namespace wbx
