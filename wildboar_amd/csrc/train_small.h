// train_small.h -- differentiable DTW of few pairs (train_small.hip).
#pragma once

#include "lane_common.h"

namespace wbx {

// Whether the small form serves a DTW call of all (mode 0) or paired (1) series
// (decided by the sizes alone: forward, backward and the size query agree).
bool small_train_ok(int mode, int64_t nx, int64_t ny, const Band &bd);
// Bytes of the state (decisions, squared costs) and of the backward's scratch.
void small_train_sizes(int mode, int64_t nx, int64_t ny, const Band &bd, int64_t *state_bytes,
                       int64_t *scratch_bytes);
int small_train_forward(const PairSpec &ps, Series<float> xs, Series<float> ys, const Band &bd,
                        double *D, void *state, hipStream_t st);
int small_train_backward(const PairSpec &ps, Series<float> xs, Series<float> ys, const Band &bd,
                         int64_t nx, int64_t ny, const double *G, const void *state, float *dX,
                         int64_t ldx, float *dY, int64_t ldy_, void *scratch, hipStream_t st);

// dY[b][j] = sum over a of gw[(a ny + b) lyp + j], in order within chunks of
// x series and over the chunks (train.hip); part: chunks * ny * ly floats.
int64_t sum_cols_part_floats(int64_t nx, int64_t ny, int64_t ly);
void launch_sum_cols(const float *gw, int64_t nx, int64_t ny, int ly, int lyp, float *part,
                     float *dY, int64_t ldy_, hipStream_t st);

}  // namespace wbx
