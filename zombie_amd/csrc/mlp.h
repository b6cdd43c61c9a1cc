// mlp.h -- device state of the Fourier-feature MLP control variate (see mlp_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace zg {

constexpr int kMaxHidden = 8;

struct MlpShape {
    int inDim;     // 2 or 3
    int nFreq;     // F: Fourier features = 2F
    int hidden;    // units per hidden layer
    int nHidden;   // hidden layers (SiLU)
};

// Parameters live in one fp32 vector theta: for l = 0..nHidden (the last is the output layer)
// W_l (out x in, row-major) at wOffset[l], then b_l at bOffset[l].  wBf mirrors theta in bf16
// (only the hidden weight matrices are read from it); bfIndex[i] = i for those entries, -1 else (fused
// layers: the place in wBf, see there).
struct MlpDevice {
    MlpShape shape;
    int64_t nParams;
    int64_t wOffset[kMaxHidden + 1], bOffset[kMaxHidden + 1];
    float* theta;
    float* grad;
    float* adamM;
    float* adamV;
    uint16_t* wBf;
    int64_t* bfIndex;
    // Fused layers (mlp_fused.hip): wBf, and wBfT for the transposed matrices, hold the hidden weights in the
    // order of the MFMA operand of a wave, so that a wave's load is one contiguous KB: a matrix B[k][n] (K rows)
    // at wOffset[l] + ((n / 16 * (K / 32) + k / 32) * 64 + k / 8 % 4 * 16 + n % 16) * 8 + k % 8.
    uint16_t* wBfT;
    int64_t* bfIndexT;
    float* freq;          // F x inDim
    int64_t maxRows;
    uint16_t* phi;        // maxRows x 2F
    float* dphi;          // maxRows x 2F
    float* pre[kMaxHidden];       // maxRows x hidden, pre-activations
    uint16_t* act[kMaxHidden];    // maxRows x hidden, activations (bf16)
    uint16_t* dz[2];              // maxRows x hidden, ping-pong gradients (bf16)
    float* loss;                  // 1
    // fused layers (mlp_fused.hip): partial gradients
    float* part;                  // [kMlpSplits * max(1, 128 / hidden)][nParams]
    float* partSmall;             // [2 kMlpFusedBlocks][(nHidden + 1) hidden + 2]
    int64_t* weightAt;            // parameter index of the i-th hidden weight
    int64_t nHiddenWeights;
    int64_t step;
};

// fused layers: shapes that they take, and the grid limits that size the partial gradients
constexpr int kMlpFusedBlocks = 256, kMlpSplits = 64;
bool mlpFusable(const MlpShape& s);
hipError_t mlpFusedEvaluate(MlpDevice& m, const float* x, int n, float* value, float* gradient, hipStream_t s);
hipError_t mlpFusedTrain(MlpDevice& m, const float* x, const float* y, int n, const float* lr, hipStream_t s);
hipError_t mlpZero(float* p, int64_t n, hipStream_t s);
hipError_t mlpCast(MlpDevice& m, hipStream_t s);
hipError_t mlpForward(MlpDevice& m, const float* x, int n, float* out, hipStream_t s);
hipError_t mlpBackward(MlpDevice& m, const float* y, int n, int mode, float* loss, float* out, hipStream_t s);
hipError_t mlpInputGrad(MlpDevice& m, const float* x, int n, float* grad, hipStream_t s);
hipError_t mlpAdam(MlpDevice& m, float lr, hipStream_t s);

}  // namespace zg
