// train.hip -- differentiable DTW: forward that records backtrack decisions,
// row-lockstep backtrack, and gradient reductions.
//
// The gradient of D = sqrt(C) along the optimal path P (dtw_mapping's
// backtrack, distance/dtw.py:395-423: from (n-1, m-1) step to
// argmin([diag, up, left]), the first minimum winning) is
//     dD/dx_i = sum_{(i,j) in P} (x_i - y_j) / D,   dD/dy_j = -sum ... / D
// (0 when D == 0).  The step taken out of cell (i, j) by the backtrack is the
// argmin over the same three predecessor costs the forward DP minimised at
// (i, j), so the forward records it: for every cell two bits, "min came from
// diag" and "min came from up" (diag before up before left on ties).
//
//  k_lane_train      the lane-per-pair kernel of lane.hip plus the two bit
//                    planes, one 32-bit word per 32 band slots per row, stored
//                    [wave][row][plane word][lane] so every store and load of
//                    a wave is one contiguous 256-byte line.
//  k_lane_backtrack  one pair per lane, all lanes of a wave on the same row,
//                    rows from the last to the first.  Within row i the path
//                    enters at slot k and moves left until the first cell
//                    whose decision is diag or up; that exit is a bit scan of
//                    (diag | up) over the row's words, which sit at addresses
//                    independent of the path and are fetched rows ahead.
//                    The row's sum of (x_i - y_j) G / D comes from prefix
//                    sums of y at once, a column's from prefix sums of x as
//                    soon as no lane's path can reach it any more.
//  k_sum_*           fixed-order sums of per-pair gradients into dX, dY
//                    (the backward is bitwise deterministic).
#include "lane_train.h"
#include "train_small.h"

namespace wbx {

// Sum over the 64 lanes in a fixed order: a running sum within each row of 16
// lanes (DPP row_shr 1, 2, 4, 8), then rows folded in with row_bcast 15 and
// 31, which leaves the total in lane 63.  Every lane returns that total.
#define WBX_DPP(v, ctrl, rmask) \
    __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rmask, 0xF, false))
__device__ __forceinline__ float wave_sum(float v) {
    v += WBX_DPP(v, 0x111, 0xF);  // row_shr:1
    v += WBX_DPP(v, 0x112, 0xF);  // row_shr:2
    v += WBX_DPP(v, 0x114, 0xF);  // row_shr:4
    v += WBX_DPP(v, 0x118, 0xF);  // row_shr:8
    v += WBX_DPP(v, 0x142, 0xA);  // row_bcast:15 into rows 1, 3
    v += WBX_DPP(v, 0x143, 0xC);  // row_bcast:31 into rows 2, 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
#undef WBX_DPP

// Where the per-pair gradients go.  Column j of pair (a, b) has the one term
// dD/dy_j = y_j u - v, u = coef * (number of path cells in column j) and
// v = coef * (sum of x_i over those cells), written 8 columns at a time.
struct GradOut {
    int mode;          // 0: GRID pairs, 1: DIAG (paired) pairs
    int xred;          // GRID with ny % 64 == 0: a wave's lanes share one x row
    int64_t nx, ny, nbc;  // nbc = ny / 64 when xred
    float *dX;         // DIAG, and GRID xred with nbc == 1: written directly
    int64_t ldx;
    float *xpart;      // GRID xred, nbc > 1: [a][bchunk][i]
    float *gxp;        // GRID without lane sharing: per-pair rows [wave][i][lane]
    float *gw;         // per-pair column terms, pair-major rows of lyp floats
    int lyp;           // ly rounded up to a multiple of 8 (rows stay 32-byte aligned)
    const float *YP;   // y_b in rows of lyp floats, zero past ly
    // X transposed (XT[i * nx + a]) and prefix sums of Y transposed
    // (PT[j * ny + b] = y_b[0] + ... + y_b[j-1], j in [0, ly], float64): the
    // lanes of a wave hold neighbouring pairs, so their loads coalesce
    const float *XT;
    const double *PT;
    // prefix sums of X, PX[i * pxi + a * pxa]: rows of one series where the
    // lanes of a wave share it, else transposed like PT
    const double *PX;
    int64_t pxi, pxa;
};

// Prefix sums P_b[j] = y_b[0] + ... + y_b[j - 1] in float64, j in [0, ly]; one
// wave per series, 64 columns at a time with a shuffle scan (the sum order is
// fixed: the result is deterministic).  ROWS: out[b * (ly + 1) + j]; else
// transposed, out[j * n + b], through an LDS tile so that a block's 16 series
// write whole lines (a scattered store per sum took 116 us longer for twice
// 65,536 series of 64).
// YP[b * lyp + j] = y_b[j], zero for ly <= j < lyp (lyp 0: not wanted).
template <bool ROWS>
__global__ __launch_bounds__(1024) void k_prefix(const float *__restrict__ Y, int64_t n, int ly,
                                                 int64_t stride, double *__restrict__ out,
                                                 float *__restrict__ YP, int lyp) {
    __shared__ double tile[16][65];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t b0 = (int64_t)blockIdx.x * 16, b = b0 + w;
    const bool mine = b < n;
    const float *y = Y + (mine ? b : n - 1) * stride;
    if (ROWS) {
        if (mine && lane == 0) out[b * (ly + 1)] = 0.0;
    } else if (threadIdx.x < 16 && b0 + threadIdx.x < n) {
        out[b0 + threadIdx.x] = 0.0;
    }
    if (mine)
        for (int j = lane; j < lyp; j += 64) YP[b * lyp + j] = j < ly ? y[j] : 0.0f;
    double carry = 0.0;
    for (int j0 = 0; j0 < ly; j0 += 64) {
        const int j = j0 + lane;
        double s = j < ly ? (double)y[j] : 0.0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const double o = __shfl_up(s, d);
            if (lane >= d) s += o;
        }
        s += carry;
        carry = __shfl(s, 63);
        if (ROWS) {
            if (mine && j < ly) out[b * (ly + 1) + j + 1] = s;
        } else {
            tile[w][lane] = s;
            __syncthreads();
            const int q = threadIdx.x & 15, c = threadIdx.x >> 4;
            if (b0 + q < n && j0 + c < ly) out[(j0 + c + 1) * n + b0 + q] = tile[q][c];
            __syncthreads();
        }
    }
}

// dst[c * n + r] = src[r * stride + c] through a 32 x 32 LDS tile.
__global__ __launch_bounds__(256) void k_transpose(const float *__restrict__ src, int64_t n,
                                                   int len, int64_t stride,
                                                   float *__restrict__ dst) {
    __shared__ float tile[32][33];
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // ty in [0, 8)
#pragma unroll
    for (int q = 0; q < 32; q += 8) {
        const int64_t r = r0 + ty + q, c = c0 + tx;
        if (r < n && c < len) tile[ty + q][tx] = src[r * stride + c];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 32; q += 8) {
        const int64_t c = c0 + ty + q, r = r0 + tx;
        if (r < n && c < len) dst[c * n + r] = tile[tx][ty + q];
    }
}

// Bit of slot k in its plane word: slots are shifted in from the low end, so
// slot k of word w sits at bit (count_w - 1 - (k - 32 w)); the last word holds
// the lastc slots that the forward computed past the others.
template <int BP, int NV>
__global__ __launch_bounds__(64 * NV) __attribute__((
    amdgpu_waves_per_eu(BP > 64 ? 2 : NV == 1 ? 3 : 4))) void k_lane_backtrack(PairSpec ps, LaneGeo g,
                                                       const float *__restrict__ sq,
                                                       const double *__restrict__ G,
                                                       const uint32_t *__restrict__ dirs,
                                                       int lastc, GradOut go) {
    constexpr int NW = (BP + 31) / 32;
    const int lane = threadIdx.x & 63, wv = NV == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t wave = blockIdx.x;
    bool mine = true;  // this wave is not a block's filling
    if constexpr (NV > 1) {
        const int64_t r = blockIdx.x / go.nbc * NV + wv;
        mine = r < go.nx;
        wave = (mine ? r : go.nx - 1) * go.nbc + blockIdx.x % go.nbc;
    }
    const int64_t p0 = wave * 64 + lane;
    const bool active = mine && p0 < ps.n_pairs;
    const int64_t p = p0 < ps.n_pairs ? p0 : ps.n_pairs - 1;
    int64_t a, b;
    decode_pair(ps, p, a, b);
    if constexpr (NV > 1) a = __builtin_amdgcn_readfirstlane((int)a);  // the wave's series
    const float *__restrict__ XT = go.XT + a;   // x_i = XT[i * nx]
    const double *__restrict__ PT = go.PT + b;  // prefix of y_b up to j: PT[j * ny]
    const int64_t nxs = go.nx, nys = go.ny;
    const int lx = g.lx, ly = g.ly, off = g.off, B = g.B;
    const double D = sqrt((double)sq[p]);
    const double coefd = (active && D > 0.0) ? G[p] / D : 0.0;
    const float coef = (float)coefd;
    // A column's terms need its first and last path row.  The walk of a row
    // notes its slot at the column where the row ends (one LDS write; of
    // several rows ending in a column the topmost stays) and how the column
    // was entered, and columns that no later row can reach are finished by all
    // lanes together, CG at a time from the right: rows of a column are
    // contiguous and one row's columns too, so the last note seen gives both
    // rows, and the sum of x over them is a difference of prefix sums.
    // Finishing each row's columns as the row leaves them runs every wave as
    // long as the longest horizontal run among its 64 paths, row after row:
    // 953 us at 262,144 pairs of 256, B = 49; 769 us this way.
    // NV > 1: the block's waves have the same lanes of y series and walk the
    // same rows, so the prefix sums of y come from a window in LDS, advanced by
    // RB columns a batch (see share_prefix): 519 us.
    constexpr int CG = 8;
    // Rows are taken RB at a time: first the path through the RB rows (bits
    // only, already in registers) while every x and prefix load those rows need
    // is issued, then the sums; the next RB rows' bits are fetched in between.
    // More rows per batch are fewer memory round trips per pair: with NV = 1,
    // 8 rows in 165 registers (three waves per SIMD) 769 us, 4 rows in 125
    // (four) 838 us; with the sums in LDS 4 rows keep four waves.
    constexpr int RB = NV == 1 && BP <= 64 ? 8 : 4;
    // columns with notes at a time: the band, a batch of rows, a partial group
    constexpr int W = BP + RB + CG - 2;
    // column mod W: the row's slot there + 1, bit 7: the column is entered by a
    // diagonal step; 0: no row ends there
    __shared__ uint8_t notes[NV][W][64];
    uint8_t(*note)[64] = notes[wv];
#pragma unroll
    for (int e = 0; e < W; ++e) note[e][lane] = 0;
    // the prefix sums of y that the rows of a batch and of the next one need
    constexpr int RW = NV > 1 ? BP + 2 * RB : 1;
    __shared__ double ring[RW][64];  // column mod RW
    if constexpr (NV > 1) {
        for (int j = lx - RB - off + wv; j <= lx - 1 + B - off; j += NV)
            if (j >= 0 && j <= ly) ring[j % RW][lane] = PT[j * nys];
        __syncthreads();
    }
    typedef float fcg __attribute__((ext_vector_type(CG)));
    fcg *__restrict__ gww = (fcg *)(go.gw + p * go.lyp);
    const fcg *__restrict__ ypw = (const fcg *)(go.YP + b * go.lyp);
    const double *__restrict__ PX = go.PX + a * go.pxa;
    const int64_t pxi = go.pxi;
    int jg = (ly - 1) / CG * CG;  // the next group of columns
    int sg = jg % W;
    int is = lx - 1;  // topmost row of the last column done
    // A value of x that is not finite belongs to the columns it is matched to,
    // not to all behind it: the lanes of such series (whose total is not finite
    // either) add the column's values up instead.
    const bool odd = !(fabs(PX[lx * pxi]) < WBX_INF_D);
    const bool any_odd = __ballot(odd) != 0;
    auto finish_group = [&](auto odd_lanes) {
        double hi[CG], lo[CG];
        float cnt[CG];
        const fcg yv_ = ypw[jg / CG];
#pragma unroll
        for (int e = CG - 1; e >= 0; --e) {
            const int j = jg + e;
            const int sl = sg + e < W ? sg + e : sg + e - W;
            const uint32_t v = note[sl][lane];
            note[sl][lane] = 0;
            const int last = is - (int)(v >> 7);
            if (v) is = j + off + 1 - (int)(v & 127u);
            cnt[e] = (float)(last - is + 1);
            hi[e] = PX[(last + 1) * pxi];
            lo[e] = PX[is * pxi];
            if constexpr (decltype(odd_lanes)::value) {
                if (odd) {
                    hi[e] = lo[e] = 0.0;
                    for (int i = is; i <= last; ++i) hi[e] += (double)XT[(int64_t)i * nxs];
                }
            }
        }
        fcg o;
#pragma unroll
        for (int e = 0; e < CG; ++e) {
            const float c = jg + e < ly ? coef : 0.0f;  // zeros past the series
            o[e] = __builtin_fmaf(c * cnt[e], yv_[e], -(c * (float)(hi[e] - lo[e])));
        }
        if (active) gww[jg / CG] = o;
        jg -= CG;
        sg = sg >= CG ? sg - CG : sg - CG + W;
    };

    uint32_t wd[RB][NW], wu[RB][NW];
    auto load_bits = [&](int ih) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int i = ih - r < 0 ? 0 : ih - r;
            const uint2 *src = (const uint2 *)(dirs + plane_base(wave, lx, i, 2 * NW, lane));
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const uint2 v = src[w];
                wd[r][w] = v.x;
                wu[r][w] = v.y;
            }
        }
    };
    load_bits(lx - 1);
    int k = g.kf;
    int sb = (lx - 1 - off) % W;  // slot 0 of the row, as a note's place
    if (sb < 0) sb += W;
    int rb = (lx - 1 - off) % RW;  // and as a place in the ring
    if (rb < 0) rb += RW;
    uint32_t ent = 0;  // the column the row ends in: 128 if entered by a diagonal step
    for (int ih = lx - 1; ih >= 0; ih -= RB) {
        const int jn = ih - 2 * RB + 1 - off + wv;  // this wave's new column of the next batch
        double pn = 0.0;
        if (NV > 1 && wv < RB && jn >= 0) pn = PT[jn * nys];
        int nr[RB];  // cells of the row
        float xr[RB];
        double ph[RB], pl[RB];
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int i = ih - r;
            if (i < 0) break;  // uniform
            const int klo = off - i > 0 ? off - i : 0;
            int khi = ly - 1 - i + off;
            if (khi > B - 1) khi = B - 1;
            if (k > khi) k = khi;
            // exit: the highest slot <= k whose decision is diag or up
            const int wk = k >> 5;
            int kx = -1;
            bool isd = false;
#pragma unroll
            for (int w = NW - 1; w >= 0; --w) {
                const int cnt_w = (w == NW - 1) ? lastc : 32;
                uint32_t msk = wd[r][w] | wu[r][w];
                if (w > wk) msk = 0u;
                if (w == wk) msk &= ~0u << (cnt_w - 1 - (k - 32 * w));
                if (kx < 0 && msk != 0u) {
                    const int q = __builtin_ctz(msk);
                    kx = 32 * w + cnt_w - 1 - q;
                    isd = ((wd[r][w] >> q) & 1u) != 0u;
                }
            }
            // Row 0 always ends at column 0 (only left moves there, dtw.py:404-406);
            // kx < klo is unreachable on a finite path and keeps the walk in bounds.
            if (i == 0 || kx < klo) {
                kx = klo;
                isd = false;
            }
            if (k < kx) k = kx;  // likewise unreachable; keeps je >= jx
            const int je = i + k - off, jx = i + kx - off;  // in [0, ly)
            const int sl = sb + k;
            note[sl < W ? sl : sl - W][lane] = (uint8_t)(ent | (uint32_t)(k + 1));
            sb = sb == 0 ? W - 1 : sb - 1;
            ent = isd ? 128u : kx == k ? ent : 0u;
            nr[r] = k - kx + 1;
            xr[r] = XT[(int64_t)i * nxs];
            if constexpr (NV > 1) {
                const int sh = rb + k + 1, sx = rb + kx;
                ph[r] = ring[sh < RW ? sh : sh - RW][lane];
                pl[r] = ring[sx < RW ? sx : sx - RW][lane];
                rb = rb == 0 ? RW - 1 : rb - 1;
            } else {
                ph[r] = PT[(int64_t)(je + 1) * nys];
                pl[r] = PT[(int64_t)jx * nys];
            }
            k = isd ? kx : kx + 1;
        }
        if (ih - RB >= 0) load_bits(ih - RB);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int i = ih - r;
            if (i < 0) break;  // uniform
            const float xi = xr[r];
            // dD/dx_i: coef * sum over the row's cells of (x_i - y_j)
            const float gx = (float)(coefd * ((double)nr[r] * (double)xi - (ph[r] - pl[r])));
            if (go.mode == 1) {
                if (active) go.dX[p * go.ldx + i] = gx;
            } else if (go.xred) {
                const float tot = wave_sum(gx);
                if (lane == 0 && mine) {
                    const int64_t bc = (wave * 64 - a * go.ny) / 64;
                    if (go.nbc == 1)
                        go.dX[a * go.ldx + i] = tot;
                    else
                        go.xpart[(a * go.nbc + bc) * lx + i] = tot;
                }
            } else {
                go.gxp[(wave * lx + i) * 64 + lane] = gx;
            }
        }
        if constexpr (NV > 1) {
            if (wv < RB && jn >= 0) ring[jn % RW][lane] = pn;
            __syncthreads();
        }
        // rows up to ih - RB reach columns below ih - RB + B - off
        while (jg >= 0 && (ih < RB || jg >= ih - RB + B - off)) {
            if (any_odd)
                finish_group(std::true_type());
            else
                finish_group(std::false_type());
        }
    }
}

__device__ __forceinline__ int64_t pair_slot(int64_t p, int len, int idx) {
    return ((p >> 6) * len + idx) * 64 + (p & 63);
}

// dX[a][i] = sum_b gxp[pair (a, b)][i], b in order (GRID without lane sharing)
__global__ __launch_bounds__(256) void k_sum_rows(const float *__restrict__ gxp, int64_t nx,
                                                  int64_t ny, int lx, float *__restrict__ dX,
                                                  int64_t ldx) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= nx * lx) return;
    const int64_t a = q / lx;
    const int i = (int)(q - a * lx);
    float s = 0.0f;
    for (int64_t b = 0; b < ny; ++b) s += gxp[pair_slot(a * ny + b, lx, i)];
    dX[a * ldx + i] = s;
}

// dX[a][i] = sum over b-chunks c of xpart[a][c][i]
__global__ __launch_bounds__(256) void k_sum_xpart(const float *__restrict__ xpart, int64_t nx,
                                                   int64_t nbc, int lx, float *__restrict__ dX,
                                                   int64_t ldx) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= nx * lx) return;
    const int64_t a = q / lx;
    const int i = (int)(q - a * lx);
    float s = 0.0f;
    for (int64_t c = 0; c < nbc; ++c) s += xpart[(a * nbc + c) * lx + i];
    dX[a * ldx + i] = s;
}

// part[c][b][j]: sums over a in chunk c of the column terms of pair (a, b),
// a in order
__global__ __launch_bounds__(256) void k_sum_cols_partial(const float *__restrict__ gw, int64_t nx,
                                                          int64_t ny, int ly, int lyp, int chunk,
                                                          float *__restrict__ part) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t per = ny * ly;
    const int c = blockIdx.y;
    if (q >= per) return;
    const int64_t b = q / ly;
    const int j = (int)(q - b * ly);
    const int64_t a0 = (int64_t)c * chunk;
    const int64_t a1 = a0 + chunk < nx ? a0 + chunk : nx;
    float s = 0.0f;
#pragma unroll 8
    for (int64_t a = a0; a < a1; ++a) s += gw[(a * ny + b) * lyp + j];
    part[(int64_t)c * per + q] = s;
}

// dY[b][j] = sum of the chunk partials, chunks in order
__global__ __launch_bounds__(256) void k_sum_cols_final(const float *__restrict__ part, int nc,
                                                        int64_t ny, int ly, float *__restrict__ dY,
                                                        int64_t ldy_) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t per = ny * ly;
    if (q >= per) return;
    float s = 0.0f;
    for (int c = 0; c < nc; ++c) s += part[(int64_t)c * per + q];
    const int64_t b = q / ly;
    const int j = (int)(q - b * ly);
    dY[b * ldy_ + j] = s;
}

// Paired pairs: dY[p][j] is pair p's column term.
__global__ __launch_bounds__(256) void k_dy_paired(const float *__restrict__ gw, int64_t n, int ly,
                                                   int lyp, float *__restrict__ dY, int64_t ldy_) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= n * ly) return;
    const int64_t p = q / ly;
    const int j = (int)(q - p * ly);
    const int64_t o = p * lyp + j;
    dY[p * ldy_ + j] = gw[o];
}

constexpr int TRAIN_MAX_BP = 112;
constexpr int COL_CHUNK = 256;  // x series per column partial: 16 partials for 4096

int64_t sum_cols_part_floats(int64_t nx, int64_t ny, int64_t ly) {
    return (nx + COL_CHUNK - 1) / COL_CHUNK * ny * ly;
}

void launch_sum_cols(const float *gw, int64_t nx, int64_t ny, int ly, int lyp, float *part,
                     float *dY, int64_t ldy_, hipStream_t st) {
    const unsigned blocks = (unsigned)((ny * ly + 255) / 256);
    const int nc = (int)((nx + COL_CHUNK - 1) / COL_CHUNK);
    hipLaunchKernelGGL(k_sum_cols_partial, dim3(blocks, (unsigned)nc), dim3(256), 0, st, gw, nx,
                       ny, ly, lyp, COL_CHUNK, part);
    hipLaunchKernelGGL(k_sum_cols_final, dim3(blocks), dim3(256), 0, st, part, nc, ny, ly, dY,
                       ldy_);
}

// Whether 8 waves (8 x series, the same 64 y series) share a block's window of
// y prefix sums.  The gathers it replaces touch about 45 lines each, so that a
// full chip waits for the vector caches (262,144 pairs of 256, B = 49: 769 ->
// 519 us); at few waves there is no queue and the blocks' barriers cost more.
// Alone, waves run 3 to a SIMD (2 past 64 slots); the line is where they need
// a second pass.  One step, alone and shared: 256 blocks, B = 49 678 and 733
// us, B = 103 1026 and 918; 512 blocks, B = 49 1280 and 1029.
static bool share_prefix(int BP, int64_t blocks) { return blocks >= (BP > 64 ? 256 : 385); }

static int train_bp(int B) { return (B + 7) / 8 * 8; }

template <int BP, int U>
static void train_fwd_one(const PairSpec &ps, Series<float> xs, Series<float> ys, LaneGeo g,
                          float *sq, uint32_t *dirs, hipStream_t st) {
    hipLaunchKernelGGL((k_lane_train<BP, U, false, false>), dim3((unsigned)((ps.n_pairs + 63) / 64)), dim3(64), 0,
                       st, ps, xs, ys, g, sq, dirs);
}

template <int BP>
static void train_bwd_one(const PairSpec &ps, LaneGeo g, const float *sq, const double *G,
                          const uint32_t *dirs, GradOut go, hipStream_t st) {
    const int slots = lane_exact_supported(g.B) ? g.B : BP;  // as the forward computed
    const int lastc = slots - 32 * ((BP + 31) / 32 - 1);
    if (go.xred && share_prefix(BP, (go.nx + 7) / 8 * go.nbc))
        hipLaunchKernelGGL((k_lane_backtrack<BP, 8>), dim3((unsigned)((go.nx + 7) / 8 * go.nbc)),
                           dim3(512), 0, st, ps, g, sq, G, dirs, lastc, go);
    else
        hipLaunchKernelGGL((k_lane_backtrack<BP, 1>), dim3((unsigned)((ps.n_pairs + 63) / 64)),
                           dim3(64), 0, st, ps, g, sq, G, dirs, lastc, go);
}

#define TRAIN_CASES(X)                                                                          \
    X(8, 4) X(16, 4) X(24, 4) X(32, 4) X(40, 4) X(48, 4) X(56, 4) X(64, 4) X(72, 4) X(80, 4)    \
        X(88, 4) X(96, 4) X(104, 4) X(112, 4)

struct TrainGeo {
    LaneGeo g;
    int BP, NW;
};

#define RCT(x)               \
    do {                     \
        int _rc = (x);       \
        if (_rc) return _rc; \
    } while (0)

// Which form serves a call: the decision planes of the lane kernels (DTW,
// bands up to TRAIN_MAX_BP slots) or the band checkpoints of train_seg.hip
// (WDTW, wider bands, and every call with mode bit 1 set).
static int train_route(const wbx_metric *m, int mode, int64_t tx, int64_t ty, bool *seg) {
    if (mode < 0 || mode > 3) return fail(WBX_EINVAL, "mode %d (0..3)", mode);
    if (m->kind != WBX_DTW && m->kind != WBX_WDTW)
        return fail(WBX_EUNSUPPORTED, "differentiable DTW supports metrics dtw and wdtw");
    if (m->precision != WBX_FP32)
        return fail(WBX_EUNSUPPORTED, "differentiable DTW runs in FP32");
    if (tx < 1 || ty < 1 || tx > (1 << 24) || ty > (1 << 24))
        return fail(WBX_EINVAL, "series lengths (%lld, %lld)", (long long)tx, (long long)ty);
    const Band bd = make_band((int)tx, (int)ty, m->r);
    // the checkpointed form splits the band over lanes of at least two slots;
    // a one-slot DTW band (the diagonal) takes the planes
    if (bd.B < 2) {
        if (m->kind == WBX_WDTW)
            return fail(WBX_EUNSUPPORTED, "differentiable WDTW needs a band of 2 slots or more");
        *seg = false;
        return WBX_OK;
    }
    *seg = (mode & 2) != 0 || m->kind == WBX_WDTW || bd.B > TRAIN_MAX_BP;
    return WBX_OK;
}

static int train_geo(const wbx_metric *m, int64_t tx, int64_t ty, TrainGeo *out) {
    if (m->kind != WBX_DTW)
        return fail(WBX_EUNSUPPORTED, "differentiable DTW supports metric dtw only");
    if (m->precision != WBX_FP32)
        return fail(WBX_EUNSUPPORTED, "differentiable DTW runs in FP32");
    const Band bd = make_band((int)tx, (int)ty, m->r);
    if (bd.B > TRAIN_MAX_BP)
        return fail(WBX_EUNSUPPORTED, "differentiable DTW: band of %d slots exceeds %d", bd.B,
                    TRAIN_MAX_BP);
    out->g = LaneGeo{bd.lx, bd.ly, bd.off, bd.B, bd.ly - bd.lx + bd.off};
    out->BP = train_bp(bd.B);
    out->NW = (out->BP + 31) / 32;
    return WBX_OK;
}

// Backward scratch (GRID only): per-pair y rows, per-pair x rows when the
// lanes of a wave do not share an x row, x partials per 64-column chunk, and
// the column partials.
struct TrainScratch {
    bool xred;
    int64_t nbc, xt, pt, px, gw, yp, gx, xpart, part, total;  // byte offsets / sizes
};

static TrainScratch train_scratch(int mode, int64_t nx, int64_t ny, int64_t tx, int64_t ty) {
    TrainScratch t{};
    auto al = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t np = mode == 0 ? nx * ny : nx, waves = (np + 63) / 64;
    int64_t o = 0;
    t.xt = o;
    o += al(nx * tx * 4);
    t.pt = o;
    o += al((ty + 1) * ny * 8);
    t.px = o;
    o += al((tx + 1) * nx * 8);
    const int64_t lyp = (ty + 7) / 8 * 8;
    t.gw = o;
    o += al(np * lyp * 4);
    t.yp = o;
    o += al(ny * lyp * 4);
    t.gx = t.xpart = t.part = o;
    if (mode != 0) {
        t.total = o;
        return t;
    }
    t.xred = ny % 64 == 0;
    t.nbc = t.xred ? ny / 64 : 0;
    t.gx = o;
    if (!t.xred) o += al(waves * tx * 64 * 4);
    t.xpart = o;
    if (t.xred && t.nbc > 1) o += al(nx * t.nbc * tx * 4);
    t.part = o;
    o += al(sum_cols_part_floats(nx, ny, ty) * 4);
    t.total = o;
    return t;
}

}  // namespace wbx

using namespace wbx;

extern "C" {

// Sizes of the state kept from forward to backward (decision planes + the
// squared costs) and of the backward's scratch (per-pair gradients).
int wbx_dtw_train_sizes(const wbx_metric *metric, int mode, int64_t nx, int64_t ny, int64_t tx,
                        int64_t ty, int64_t *state_bytes, int64_t *scratch_bytes) {
    if (!metric) return fail(WBX_EINVAL, "metric is NULL");
    bool seg;
    RCT(train_route(metric, mode, tx, ty, &seg));
    if (seg)
        return seg_train_sizes(metric, mode & 1, nx, ny, tx, ty, state_bytes, scratch_bytes);
    TrainGeo tg;
    int rc = train_geo(metric, tx, ty, &tg);
    if (rc) return rc;
    const int64_t np = mode == 0 ? nx * ny : nx;
    const Band bd = make_band((int)tx, (int)ty, metric->r);
    if (small_train_ok(mode, nx, ny, bd)) {
        small_train_sizes(mode, nx, ny, bd, state_bytes, scratch_bytes);
        return WBX_OK;
    }
    const int64_t waves = (np + 63) / 64;
    const int64_t planes = waves * tx * 2 * tg.NW * 64 * 4;
    if (state_bytes) *state_bytes = planes + ((np * 4 + 255) / 256) * 256;
    if (scratch_bytes) *scratch_bytes = train_scratch(mode, nx, ny, tx, ty).total;
    return WBX_OK;
}

// mode 0: all (x, y) pairs of X (nx) and Y (ny), D is (nx, ny);
// mode 1: D[p] = DTW(X[p], Y[p]) for p < nx (ny must equal nx).
int wbx_dev_dtw_train_forward(const wbx_metric *metric, int mode, const float *X, int64_t nx,
                              int64_t x_stride, int64_t tx, const float *Y, int64_t ny,
                              int64_t y_stride, int64_t ty, double *D, void *state, void *stream) {
    if (!metric || !X || !Y || !D || !state) return fail(WBX_EINVAL, "NULL argument");
    if (nx < 1 || ny < 1 || tx < 1 || ty < 1) return fail(WBX_EINVAL, "empty input");
    if ((mode & 1) && nx != ny) return fail(WBX_EINVAL, "paired mode needs nx == ny");
    bool seg;
    RCT(train_route(metric, mode, tx, ty, &seg));
    if (seg)
        return seg_train_forward(metric, mode & 1, X, nx, x_stride, tx, Y, ny, y_stride, ty, D,
                                 state, (hipStream_t)stream);
    TrainGeo tg;
    int rc = train_geo(metric, tx, ty, &tg);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    PairSpec ps{mode == 0 ? PAIR_GRID : PAIR_DIAG, mode == 0 ? nx * ny : nx, mode == 0 ? ny : nx,
                nullptr, nullptr};
    const int64_t waves = (ps.n_pairs + 63) / 64;
    uint32_t *dirs = (uint32_t *)state;
    float *sq = (float *)((char *)state + waves * tx * 2 * tg.NW * 64 * 4);
    Series<float> xs{X, x_stride, (int)tx, nullptr}, ys{Y, y_stride, (int)ty, nullptr};
    const Band bd = make_band((int)tx, (int)ty, metric->r);
    if (small_train_ok(mode, nx, ny, bd)) return small_train_forward(ps, xs, ys, bd, D, state, st);
    if (lane_exact_supported(tg.g.B)) {
        RCT(launch_lane_train_exact(ps, xs, ys, tg.g, sq, dirs, st));
        return launch_finish<float>(ps, sq, D, ny, st);
    }
    switch (tg.BP) {
#define FWD_CASE(BPV, UV) \
    case BPV: train_fwd_one<BPV, UV>(ps, xs, ys, tg.g, sq, dirs, st); break;
        TRAIN_CASES(FWD_CASE)
#undef FWD_CASE
        default: return fail(WBX_EUNSUPPORTED, "band %d", tg.g.B);
    }
    WBX_HIP_CHECK(hipGetLastError());
    return launch_finish<float>(ps, sq, D, ny, st);
}

// G: upstream gradient dL/dD, same layout as D.  dX (nx, tx) and dY (ny, ty)
// float32 with row strides ldx / ldy are overwritten.
int wbx_dev_dtw_train_backward(const wbx_metric *metric, int mode, const float *X, int64_t nx,
                               int64_t x_stride, int64_t tx, const float *Y, int64_t ny,
                               int64_t y_stride, int64_t ty, const double *G, const void *state,
                               float *dX, int64_t ldx, float *dY, int64_t ldy_, void *scratch,
                               void *stream) {
    if (!metric || !X || !Y || !G || !state || !dX || !dY || !scratch)
        return fail(WBX_EINVAL, "NULL argument");
    if (nx < 1 || ny < 1 || tx < 1 || ty < 1) return fail(WBX_EINVAL, "empty input");
    if ((mode & 1) && nx != ny) return fail(WBX_EINVAL, "paired mode needs nx == ny");
    bool seg;
    RCT(train_route(metric, mode, tx, ty, &seg));
    if (seg)
        return seg_train_backward(metric, mode & 1, X, nx, x_stride, tx, Y, ny, y_stride, ty, G,
                                  state, dX, ldx, dY, ldy_, scratch, (hipStream_t)stream);
    TrainGeo tg;
    int rc = train_geo(metric, tx, ty, &tg);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    PairSpec ps{mode == 0 ? PAIR_GRID : PAIR_DIAG, mode == 0 ? nx * ny : nx, mode == 0 ? ny : nx,
                nullptr, nullptr};
    const Band bd = make_band((int)tx, (int)ty, metric->r);
    if (small_train_ok(mode, nx, ny, bd))
        return small_train_backward(ps, Series<float>{X, x_stride, (int)tx, nullptr},
                                    Series<float>{Y, y_stride, (int)ty, nullptr}, bd, nx, ny, G,
                                    state, dX, ldx, dY, ldy_, scratch, st);
    const int64_t waves = (ps.n_pairs + 63) / 64;
    const uint32_t *dirs = (const uint32_t *)state;
    const float *sq = (const float *)((const char *)state + waves * tx * 2 * tg.NW * 64 * 4);
    const TrainScratch ts = train_scratch(mode, nx, ny, tx, ty);
    char *sc = (char *)scratch;
    GradOut go{};
    go.mode = mode;
    go.xred = ts.xred ? 1 : 0;
    go.nx = nx;
    go.ny = ny;
    go.nbc = ts.nbc;
    go.dX = dX;
    go.ldx = ldx;
    go.gxp = (float *)(sc + ts.gx);
    go.xpart = (float *)(sc + ts.xpart);
    go.gw = (float *)(sc + ts.gw);
    go.lyp = (int)((ty + 7) / 8 * 8);
    float *yp = (float *)(sc + ts.yp);
    go.YP = yp;
    float *part = (float *)(sc + ts.part);
    float *xt = (float *)(sc + ts.xt);
    double *pt = (double *)(sc + ts.pt);
    hipLaunchKernelGGL(k_transpose, dim3((unsigned)((tx + 31) / 32), (unsigned)((nx + 31) / 32)),
                       dim3(256), 0, st, X, nx, (int)tx, x_stride, xt);
    hipLaunchKernelGGL(k_prefix<false>, dim3((unsigned)((ny + 15) / 16)), dim3(1024), 0, st, Y, ny,
                       (int)ty, y_stride, pt, yp, go.lyp);
    double *px = (double *)(sc + ts.px);
    go.pxi = ts.xred ? 1 : nx;
    go.pxa = ts.xred ? tx + 1 : 1;
    go.PX = px;
    hipLaunchKernelGGL(ts.xred ? k_prefix<true> : k_prefix<false>,
                       dim3((unsigned)((nx + 15) / 16)), dim3(1024), 0, st, X, nx, (int)tx,
                       x_stride, px, (float *)nullptr, 0);
    go.XT = xt;
    go.PT = pt;
    switch (tg.BP) {
#define BWD_CASE(BPV, UV) \
    case BPV: train_bwd_one<BPV>(ps, tg.g, sq, G, dirs, go, st); break;
        TRAIN_CASES(BWD_CASE)
#undef BWD_CASE
        default: return fail(WBX_EUNSUPPORTED, "band %d", tg.g.B);
    }
    WBX_HIP_CHECK(hipGetLastError());
    const unsigned gy_blocks = (unsigned)((ny * ty + 255) / 256);
    if (mode == 0) {
        const unsigned gx_blocks = (unsigned)((nx * tx + 255) / 256);
        if (!ts.xred)
            hipLaunchKernelGGL(k_sum_rows, dim3(gx_blocks), dim3(256), 0, st, go.gxp, nx, ny,
                               (int)tx, dX, ldx);
        else if (ts.nbc > 1)
            hipLaunchKernelGGL(k_sum_xpart, dim3(gx_blocks), dim3(256), 0, st, go.xpart, nx, ts.nbc,
                               (int)tx, dX, ldx);
        launch_sum_cols(go.gw, nx, ny, (int)ty, go.lyp, part, dY, ldy_, st);
    } else {
        hipLaunchKernelGGL(k_dy_paired, dim3(gy_blocks), dim3(256), 0, st, go.gw, ny, (int)ty,
                           go.lyp, dY, ldy_);
    }
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

}  // extern "C"
