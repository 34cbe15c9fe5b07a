// lane_exact_w.hip -- the exact-band lane kernel (lane_kernel.h) for WDTW
// matrices of series of equal length, compiled for every odd band width
// B = 9 .. 111 with the weights of a row in SGPRs.
#include "lane_kernel.h"

namespace wbx {

// The kernel reads (B + 1) / 2 weights of the max(lx, ly) there are.  The slopes
// of a derivative metric keep the band of the longer series they come from,
// which can be wider than the slopes are long: those calls take the kernels
// that clamp the index.
int64_t lane_exact_w_waves(const PairSpec &ps, int lx, int ly, int B) {
    if (ps.mode != PAIR_GRID || lx != ly || (B + 1) / 2 > lx || !lane_exact_supported(B)) return 0;
    const int64_t waves = ps.n_pairs / ps.ny * ((ps.ny + 63) / 64);
    return waves <= INT32_MAX ? waves : 0;
}

int launch_lane_exact_w(const PairSpec &ps, Series<float> xs, Series<float> ys, const LaneGeo &g,
                        const float *weights, float *sq, hipStream_t st) {
    const int64_t waves = lane_exact_w_waves(ps, xs.len, ys.len, g.B);
    if (!waves) return fail(WBX_EUNSUPPORTED, "weighted lane kernel: unsupported geometry");
    const dim3 grid((unsigned)waves);
    switch (g.B) {
#define WBX_EXACT(b)                                                                          \
    case b:                                                                                   \
        hipLaunchKernelGGL((k_lane_dtw_exact<b, b <= 88 ? 8 : 4, true, true>), grid, dim3(64), \
                           0, st, ps, xs, ys, g, weights, sq);                                \
        break;
        WBX_EXACT(9) WBX_EXACT(11) WBX_EXACT(13) WBX_EXACT(15) WBX_EXACT(17) WBX_EXACT(19)
        WBX_EXACT(21) WBX_EXACT(23) WBX_EXACT(25) WBX_EXACT(27) WBX_EXACT(29) WBX_EXACT(31)
        WBX_EXACT(33) WBX_EXACT(35) WBX_EXACT(37) WBX_EXACT(39) WBX_EXACT(41) WBX_EXACT(43)
        WBX_EXACT(45) WBX_EXACT(47) WBX_EXACT(49) WBX_EXACT(51) WBX_EXACT(53) WBX_EXACT(55)
        WBX_EXACT(57) WBX_EXACT(59) WBX_EXACT(61) WBX_EXACT(63) WBX_EXACT(65) WBX_EXACT(67)
        WBX_EXACT(69) WBX_EXACT(71) WBX_EXACT(73) WBX_EXACT(75) WBX_EXACT(77) WBX_EXACT(79)
        WBX_EXACT(81) WBX_EXACT(83) WBX_EXACT(85) WBX_EXACT(87) WBX_EXACT(89) WBX_EXACT(91)
        WBX_EXACT(93) WBX_EXACT(95) WBX_EXACT(97) WBX_EXACT(99) WBX_EXACT(101) WBX_EXACT(103)
        WBX_EXACT(105) WBX_EXACT(107) WBX_EXACT(109) WBX_EXACT(111)
#undef WBX_EXACT
    }
    WBX_HIP_CHECK(hipGetLastError());
    return WBX_OK;
}

}  // namespace wbx
