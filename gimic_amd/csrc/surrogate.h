// Shapes and launchers of the surrogate network's kernels (surrogate.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace gimic {

// Fourier frequencies, input features, hidden width, hidden layers, output
// rows (nine tensor elements, the log amplitude, padding)
constexpr int kMlpF = 64, kMlpK0 = 160, kMlpH = 128, kMlpD = 4, kMlpNO = 16;
constexpr int kMlpParams =
    (kMlpK0 + 1) * kMlpH + (kMlpD - 1) * (kMlpH + 1) * kMlpH + (kMlpH + 1) * kMlpNO;
// transposed BF16 weights of layers 1 .. D
constexpr int kMlpTransposed = (kMlpD - 1) * kMlpH * kMlpH + kMlpH * kMlpNO;
constexpr int kMlpMaxRanges = 64;                       // point ranges of the weight gradients
constexpr int kMlpBiasPart = kMlpD * kMlpH + kMlpNO + 1;  // per tile workgroup

struct MlpTileArgs {
    const double *r, *target;
    long long npts;
    const float *freq, *cs, *oscale;
    float eps2;
    const float *prm;        // FP32 master parameters (biases)
    const __bf16 *W, *WT;    // BF16 copies: flat, and transposed
    // written for training, rows of whole 64-point tiles: inputs of every
    // layer, dZ of the hidden layers, dY; bias gradients and loss per workgroup
    __bf16 *X[kMlpD + 1], *dZ[kMlpD], *dY;
    float *bpart;
    double *J;               // written by the forward-only form
};
struct MlpAdamArgs {
    const float *part, *bpart;
    int ranges, groups;      // of part and bpart
    int adam;                // 0: only the gradient, into grad
    float *grad, *loss;
    float *prm, *m, *v;
    __bf16 *W, *WT;
    float lr, b1, b2, eps, bc1, bc2;
};
int mlp_tile_groups(long long npts);
int mlp_ranges(long long npts);
hipError_t mlp_tiles(const MlpTileArgs &a, bool train, hipStream_t s);
hipError_t mlp_dw(const MlpTileArgs &a, float *part, hipStream_t s);
hipError_t mlp_adam(const MlpAdamArgs &a, hipStream_t s);
hipError_t mlp_cast(const float *p, __bf16 *W, __bf16 *WT, hipStream_t s);
hipError_t mlp_infer(const double *r, long long npts, const float *freq, const float *cs,
                     const __bf16 *W, const float *prm, const float *oscale, double *J, hipStream_t s);

}  // namespace gimic
