// Launchers of the warm-start U-Net kernels (unet_kernels.hip).  Tensors are
// channels-last at their level's resolution: activations BF16 bit patterns
// (uint16_t), gradients FP32 or, as operands of the products, BF16.  FP32
// master weights are [27][ci][co]; weights_bf16 makes the copies the products
// read.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace artss {
namespace nn {

struct Dims {
    int X, Y, Z;  // voxels along x, y, z
};

// 3x3x3 convolution with ci, co in {16,32,64} (MFMA); Wt: the layer's `fwd`
// copy; up: the input is at half resolution and read nearest-upsampled; pre
// (may be null): pre-activation; skip (may be null): added after the activation
void conv_fwd(hipStream_t s, int ci, int co, bool up, Dims D, const uint16_t *in, const uint16_t *Wt,
              const float *bias, uint16_t *out, uint16_t *pre, const uint16_t *skip, bool relu);
// first layer 2 -> 16 (FP32 input, ReLU) and last layer 16 -> 1 (no activation)
void conv_in(hipStream_t s, Dims D, const float *x, const float *W, const float *bias, uint16_t *out);
void conv_out(hipStream_t s, Dims D, const uint16_t *in, const float *W, const float *bias, float *y);
// 2x2x2 mean (Dc: coarse dims)
void down(hipStream_t s, int c, Dims Dc, const uint16_t *in, uint16_t *out);

// ---- backward.  `part` receives one row of partial sums per workgroup, as
// many rows as the matching *_rows call says; sum_rows adds them.
// data gradient of a layer that is not upsampled, zero where act (may be
// null) is not positive; W: the layer's `bwd` copy
void conv_dgrad(hipStream_t s, int ci, int co, Dims D, const uint16_t *g, const uint16_t *W, const uint16_t *act,
                float *gin);
// data gradient of an upsampling layer at its coarse input (Dc): gskip (may be
// null) the gradient, gmask its BF16 form where act > 0, rows of ci sums of that
int up_dgrad_rows(int ci, int co, Dims Dc);
void conv_up_dgrad(hipStream_t s, int ci, int co, Dims Dc, const uint16_t *g, const uint16_t *Wd,
                   const uint16_t *act, float *gskip, uint16_t *gmask, float *part);
// weight gradient, rows of 27 ci co
int wgrad_rows(int ci, int co, Dims D);
void conv_wgrad(hipStream_t s, int ci, int co, bool up, Dims D, const uint16_t *in, const uint16_t *g, float *part);
// end layers: rows of 54 x 16 weight and 16 bias sums (first), 27 x 16 (last)
int end_wgrad_rows(Dims D);
void conv_in_wgrad(hipStream_t s, Dims D, const float *x, const float *g, float *part);
void conv_out_wgrad(hipStream_t s, Dims D, const uint16_t *in, const float *gy, float *part);
// rows of the elementwise kernels over `voxels` with `groups` items per voxel
int elementwise_rows(long long voxels, int groups);
// last layer's data gradient as conv_up_dgrad's outputs, rows of 16
int end_dgrad_rows(Dims D);
void conv_out_dgrad(hipStream_t s, Dims D, const float *W, const float *gy, const uint16_t *act, float *gskip,
                    uint16_t *gmask, float *part);
// gskip + the spread mean gradient gc of the next coarser level, BF16 where
// act > 0 (groups c / 4, rows of c)
void enc_grad(hipStream_t s, int c, Dims D, const float *gskip, const float *gc, const uint16_t *act, uint16_t *gmask,
              float *part);
// gy = d (mean squared error) / dy (groups 1, rows of 4: sum of squares, sum of gy)
void mse(hipStream_t s, long long n, const float *y, const float *target, float *gy, float *part);

struct SumJob {
    const float *part;
    int rows, stride, n;  // n columns of rows that are `stride` apart
    float scale;
    float *out;
};
constexpr int kMaxSumJobs = 24;
struct SumJobs {
    int count;
    SumJob job[kMaxSumJobs];
};
// out[c] = scale * sum over the rows, in a fixed order, for every job
void sum_rows(hipStream_t s, const SumJobs &jobs);

void adam(hipStream_t s, int n, float *w, const float *g, float *m, float *v, float lr, float b1, float b2, float eps,
          float c1, float c2);
struct WeightJob {
    const float *w;      // [27][ci][co]
    int ci, co, up;
    uint16_t *fwd, *bwd;  // [27][co][ci] and [27][ci][co]; up: [8 parities][8 taps][co][ci] and [3][64][ci][co]
};
constexpr int kMaxWeightJobs = 8;
struct WeightJobs {
    int count;
    WeightJob job[kMaxWeightJobs];
};
void weights_bf16(hipStream_t s, const WeightJobs &jobs);

}  // namespace nn
}  // namespace artss
