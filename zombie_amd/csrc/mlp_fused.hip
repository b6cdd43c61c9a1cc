// mlp_fused.hip -- the Fourier-feature MLP with its layers fused, for the shapes a block can hold: 64 or
// 128 hidden units, 32 or 64 features, up to 4 hidden layers (mlpFusable).  Other shapes keep the GEMM per
// layer of mlp_kernels.hip.
//
// A layer of 128 units moves 48-64 MB at a batch of 65,536 when it goes through memory (bf16 activations
// and 32-bit pre-activations, each way) against 2 GFLOP, so the GEMM-per-layer form was bound by memory and
// launches: 350 us per training step, 250 us per 65,536 evaluations with gradients.  Here a block carries
// 64 rows through all layers, forward and back: activations stay in LDS as bf16, the derivatives of the
// activations in registers in 32 bits.  Training writes only what the weight gradients need (bf16
// activations and their gradients), which one more kernel contracts, and a third adds up the partial
// gradients and takes the Adam step.
//
// Measured at 128 units, 4 layers, 64 features: a training step of 65,536 rows 350 -> 96 us of kernels (fused
// layers 63, weight gradients 24, reduction and Adam 9), 262,144 values and gradients 1,010 -> 205 us.  Bound: the
// chain of barriers and dependent products within a tile (VALU issue, mostly the activations, is a third of
// the time).  What it took: weights stored in the order of the MFMA operand (a row-major load touches 32
// cache lines), 16 waves of 16 x 32 results instead of 8 of 32 x 32 (95 -> 71 us once nothing spilled), and no
// 64-bit address or old pre-activation held per lane (spills: 121 -> 71 -> 61 us, before the divisions below).
//
// Precision is that of the GEMM per layer: bf16 operands, 32-bit products, sums, pre-activations and
// derivatives, divisions as an IEEE division rounds them; the sums are taken in another order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "mlp.h"

namespace zg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = 64;          // rows per block and pass
constexpr int kFusedLayers = 4;

struct FusedArgs {
    int n, d, F;
    const float* x;
    const float* freq;
    const float* theta;
    // bf16 weights in the order in which waves load them (mlp.h): of W_l, and of W_l transposed
    const uint16_t* w;
    const uint16_t* wT;
    int64_t wOff[kFusedLayers + 1], bOff[kFusedLayers + 1];
    const float* y;                // training targets
    float invN;
    float* out;                    // c(x) (nullable)
    float* grad;                   // grad_x c [n x d]
    // training: operands of the weight gradients in blocks of 32 rows, [row / 32][unit][32], the rows of a
    // block in the order of the accumulators (position 8 g + 4 s + j holds row 16 s + 4 g + j; any order does
    // that is the same for both operands)
    uint16_t* phiBlk;
    uint16_t* actBlk[kFusedLayers];
    uint16_t* dzBlk[kFusedLayers];
    float* small;                  // [2 gridDim.x][(L + 1) H + 2]: bias gradients, output layer, loss
};

__device__ __forceinline__ uint16_t bf16Bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf16Value(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

// 1 / d and z / d of a finite d >= 1 as the division rounds them: the hardware's reciprocal (1 ulp) and a Newton
// step, then the quotient corrected by its remainder (Markstein, "Computation of elementary functions on the
// IBM RISC System/6000 processor", 1990).  A reciprocal below the normal range is 0, and so are both results.
// Against the reciprocal alone, two IEEE divisions, with their scaling for operands that do not occur here, make
// a training step 15% and values with gradients 34% slower; this, 3% and 7%.
__device__ __forceinline__ float reciprocal(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}
__device__ __forceinline__ float quotient(float z, float d, float r) {
    const float q = z * r;
    return fmaf(fmaf(-d, q, z), r, q);
}

// MFMA v_mfma_f32_16x16x32_bf16 operand layout, lane l of 64 (g = l / 16), element j of 8 / of 4:
//   A[row = l % 16][k = 8 g + j],  B[k = 8 g + j][col = l % 16],  D[row = 4 g + j][col = l % 16]
// A wave holds 16 columns (units) of 32 rows: two accumulators, v[s][j] = row 16 s + 4 g + j.
struct Tile {
    f32x4 v[2];
};
// 16 columns of a weight matrix of K rows, from the operand-ordered copy: one contiguous KB per load
template <int H>
struct Columns {
    bf16x8 v[H / 32];
};
template <int H>
__device__ __forceinline__ void loadColumns(Columns<H>& c, const uint16_t* b, int cg, int K, int lane) {
    b += cg * (K / 32) * 512;   // uniform: the lane's part of the address is a 32-bit offset
    const uint32_t at = (uint32_t)lane * 8u;
#pragma unroll
    for (int k = 0; k < H / 32; k++)
        if (32 * k < K) c.v[k] = load8(b + 512 * k + at);
}
// A (32 rows of an LDS tile of row stride LD, k contiguous; a: the lane's first element) x the columns
template <int H>
__device__ __forceinline__ Tile tileProduct(const uint16_t* a, const Columns<H>& c, int K) {
    constexpr int LD = H + 8;
    Tile t;
    t.v[0] = t.v[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < H / 32; k++)
        if (32 * k < K) {
            t.v[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load8(a + 32 * k), c.v[k], t.v[0], 0, 0, 0);
            t.v[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load8(a + 16 * LD + 32 * k), c.v[k], t.v[1], 0, 0, 0);
        }
    return t;
}

// stores a lane's 8 values (one unit, 8 rows) to LDS [row][unit] (p: the lane's first row) and, blocked, to
// global memory (8 contiguous elements); returns them rounded to bf16
template <int LD>
__device__ __forceinline__ void storeTile(const float (&v)[8], uint16_t (&b)[8], uint16_t* p, uint16_t* blk) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        b[e] = bf16Bits(v[e]);
        p[(16 * (e >> 2) + (e & 3)) * LD] = b[e];
    }
    if (blk)
        *reinterpret_cast<uint4*>(blk) = make_uint4((uint32_t)b[0] | ((uint32_t)b[1] << 16), (uint32_t)b[2] | ((uint32_t)b[3] << 16),
                                                    (uint32_t)b[4] | ((uint32_t)b[5] << 16), (uint32_t)b[6] | ((uint32_t)b[7] << 16));
}

enum FusedMode { kValue = 0, kTrain = 1, kGradient = 2 };

// H / 8 waves, four per SIMD at 128 units: wave (cg, rg) holds units 16 cg.. of rows 32 rg..
template <int H, int L, int MODE>
__global__ void __launch_bounds__(8 * H) fusedKernel(FusedArgs g) {
    constexpr int T = 8 * H, CG = H / 16, LD = H + 8;   // the row stride of 272 (144) B keeps 16-byte reads apart
    constexpr int kPer = T / kRows;                      // threads per row of the output layer, 8 units each
    constexpr int kPasses = 1024 / T;                    // 32 frequencies x 32 pairs of rows
    __shared__ __attribute__((aligned(16))) uint16_t buf[2][kRows * LD];
    __shared__ float dc[kRows];
    __shared__ float wLds[H], bLds[L * H];
    __shared__ float red[2][T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = lane >> 4;
    const int cg = wave % CG, rg = wave / CG, unit = 16 * cg + (lane & 15), row0 = 32 * rg;
    const int F = g.F, feat = 2 * F;
    const float wOut = g.theta[g.wOff[L] + unit], bOut = g.theta[g.bOff[L]];
    if (tid < H) {   // read after barriers below
        wLds[tid] = g.theta[g.wOff[L] + tid];
#pragma unroll
        for (int l = 0; l < L; l++) bLds[l * H + tid] = g.theta[g.bOff[l] + tid];
    }
    float db[L];
#pragma unroll
    for (int l = 0; l < L; l++) db[l] = 0.0f;
    float dwOut = 0.0f, dbOut = 0.0f, loss = 0.0f;
    const int aOff = (row0 + (lane & 15)) * LD + 8 * grp;   // a lane's operand row in an LDS tile
    const int dOff = (row0 + 4 * grp) * LD + unit;          // its first result there

    const int tiles = (g.n + kRows - 1) / kRows;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t base = (int64_t)tile * kRows;
        // where this lane's 8 rows of a unit go in the blocked layout
        auto blocked = [&](uint16_t* p) -> uint16_t* {
            if (MODE != kTrain) return nullptr;
            p += (base + row0) / 32 * (H * 32);
            asm("" : "+s"(p));   // uniform, with a 32-bit offset per lane: not a 64-bit address per lane and array
            return p + (uint32_t)(unit * 32 + 8 * grp);
        };
        // the weights of a product are loaded ahead of the work that comes before it
        Columns<H> wc;
        loadColumns<H>(wc, g.w + g.wOff[0], cg, feat, lane);
        __syncthreads();   // the previous tile is read, the output weights are there
        // features of 2 rows and one frequency per thread and pass
        float sn[kPasses][2], cs[kPasses][2];
#pragma unroll
        for (int u = 0; u < kPasses; u++) {
            const int i = tid + u * T, f = i % F, q = i / F;
            if (i >= F * 32) continue;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int64_t row = base + 2 * q + r;
                float a = 0.0f;
                if (row < g.n)
                    for (int k = 0; k < g.d; k++) a += g.freq[f * g.d + k] * g.x[row * g.d + k];
                sincosf(a, &sn[u][r], &cs[u][r]);
                buf[0][(2 * q + r) * LD + f] = bf16Bits(sn[u][r]);
                buf[0][(2 * q + r) * LD + F + f] = bf16Bits(cs[u][r]);
            }
            if (MODE == kTrain) {
                const int rr = 2 * q & 31;
                uint16_t* p = g.phiBlk + base * feat;
                asm("" : "+s"(p));
                p += (uint32_t)((q / 16 * feat + f) * 32 + 8 * (rr >> 2 & 3) + 4 * (rr >> 4) + (rr & 3));
                *reinterpret_cast<uint32_t*>(p) = (uint32_t)bf16Bits(sn[u][0]) | ((uint32_t)bf16Bits(sn[u][1]) << 16);
                *reinterpret_cast<uint32_t*>(p + F * 32) = (uint32_t)bf16Bits(cs[u][0]) | ((uint32_t)bf16Bits(cs[u][1]) << 16);
            }
        }
        __syncthreads();
        // forward: h = silu(z), and the derivative of it for the way back
        float slope[L][8];
#pragma unroll
        for (int l = 0; l < L; l++) {
            const Tile t = tileProduct<H>(buf[l & 1] + aOff, wc, l == 0 ? feat : H);
            if (l + 1 < L) loadColumns<H>(wc, g.w + g.wOff[l + 1], cg, H, lane);
            else if (MODE != kValue && 16 * cg < (L == 1 ? feat : H)) loadColumns<H>(wc, g.wT + g.wOff[l], cg, H, lane);
            float h[8];
            const float bias = bLds[l * H + unit];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float z = t.v[e >> 2][e & 3] + bias;
                const float d = fminf(1.0f + __expf(-z), FLT_MAX), s = reciprocal(d);
                h[e] = quotient(z, d, s);
                if (MODE != kValue) {
                    slope[l][e] = s * (1.0f + z * (1.0f - s));
                    asm("" : "+v"(slope[l][e]));   // computed here: z and s are not kept for later (25 registers a layer)
                }
            }
            uint16_t hb[8];
            storeTile<LD>(h, hb, buf[(l + 1) & 1] + dOff, l < L - 1 ? blocked(g.actBlk[l]) : nullptr);
            __syncthreads();
        }
        // output layer
        {
            const int row = tid / kPer, part = tid % kPer;
            const uint4 hv = *reinterpret_cast<const uint4*>(buf[L & 1] + row * LD + 8 * part);
            const uint32_t hw[4] = {hv.x, hv.y, hv.z, hv.w};
            float c = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                c += bf16Value((uint16_t)(hw[j] & 0xffffu)) * wLds[8 * part + 2 * j];
                c += bf16Value((uint16_t)(hw[j] >> 16)) * wLds[8 * part + 2 * j + 1];
            }
#pragma unroll
            for (int off = kPer / 2; off > 0; off >>= 1) c += __shfl_xor(c, off);
            c += bOut;
            const bool mine = part == 0 && base + row < g.n;
            if (mine && g.out) g.out[base + row] = c;
            if (MODE == kTrain) {
                float dcv = 0.0f;
                if (mine) {
                    const float e = c - g.y[base + row];
                    dcv = e * g.invN;
                    loss += 0.5f * e * e * g.invN;
                    dbOut += dcv;
                }
                if (part == 0) dc[row] = dcv;
            }
        }
        if (MODE == kValue) continue;
        if (MODE == kTrain) __syncthreads();
        // backward
        Tile t;
#pragma unroll
        for (int l = L - 1; l >= 0; l--) {
            float v[8];
            if (l == L - 1) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float dcv = MODE == kTrain ? dc[row0 + 16 * (e >> 2) + 4 * grp + (e & 3)] : 1.0f;
                    v[e] = dcv * wOut * slope[l][e];
                    if (MODE == kTrain) dwOut += dcv * bf16Value(buf[L & 1][dOff + (16 * (e >> 2) + (e & 3)) * LD]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = t.v[e >> 2][e & 3] * slope[l][e];
            }
            // the tiles alternate, starting with the one that the output layer did not read
            uint16_t* lds = buf[(L + 1 + (L - 1 - l)) & 1];
            uint16_t zb[8];
            storeTile<LD>(v, zb, lds + dOff, blocked(g.dzBlk[l]));
            if (MODE == kTrain) {
#pragma unroll
                for (int e = 0; e < 8; e++) db[l] += bf16Value(zb[e]);
            }
            if (l > 0) {
                __syncthreads();
                t = tileProduct<H>(lds + aOff, wc, H);
                if (l > 1 || (MODE == kGradient && 16 * cg < feat)) loadColumns<H>(wc, g.wT + g.wOff[l - 1], cg, H, lane);
            } else if (MODE == kGradient) {
                __syncthreads();
                if (16 * cg < feat) t = tileProduct<H>(lds + aOff, wc, H);
            }
        }
        if (MODE == kGradient) {
            // grad_x c = sum_f (dPhi_sin[f] cos(B_f x) - dPhi_cos[f] sin(B_f x)) B_f
            __syncthreads();
            float* dphi = reinterpret_cast<float*>(&buf[0][0]);
            const int ldp = feat + 1;
            if (16 * cg < feat) {
#pragma unroll
                for (int e = 0; e < 8; e++) dphi[(row0 + 16 * (e >> 2) + 4 * grp + (e & 3)) * ldp + unit] = t.v[e >> 2][e & 3];
            }
            __syncthreads();
            // the frequency and rows whose features this thread made; the F lanes of a pair of rows are neighbours
#pragma unroll
            for (int u = 0; u < kPasses; u++) {
                const int i = tid + u * T, f = i % F, q = i / F;
                if (i >= F * 32) continue;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const float* dr = dphi + (2 * q + r) * ldp;
                    const float coef = dr[f] * cs[u][r] - dr[F + f] * sn[u][r];
                    for (int k = 0; k < g.d; k++) {
                        float x = coef * g.freq[f * g.d + k];
                        for (int off = F / 2; off > 0; off >>= 1) x += __shfl_xor(x, off);
                        if (f == k && base + 2 * q + r < g.n) g.grad[(base + 2 * q + r) * g.d + k] = x;
                    }
                }
            }
        }
    }
    if (MODE != kTrain) return;
    // this block's sums of the small gradients, one row of them per row group
    float* sm = g.small + (size_t)(2 * blockIdx.x + rg) * ((L + 1) * H + 2);
#pragma unroll
    for (int l = 0; l < L; l++) {
        db[l] += __shfl_xor(db[l], 16);
        db[l] += __shfl_xor(db[l], 32);
        if (grp == 0) sm[l * H + unit] = db[l];
    }
    dwOut += __shfl_xor(dwOut, 16);
    dwOut += __shfl_xor(dwOut, 32);
    if (grp == 0) sm[L * H + unit] = dwOut;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        loss += __shfl_xor(loss, off);
        dbOut += __shfl_xor(dbOut, off);
    }
    if (lane == 0) { red[0][wave] = dbOut; red[1][wave] = loss; }
    __syncthreads();
    if (tid < 2) {   // both row groups' rows are read: the second one holds zero
        float t = 0.0f;
        for (int w = 0; w < T / 64; w++) t += red[tid][w];
        float* s0 = g.small + (size_t)(2 * blockIdx.x) * ((L + 1) * H + 2) + (L + 1) * H + tid;
        s0[0] = t;
        s0[(L + 1) * H + 2] = 0.0f;
    }
}

// Weight gradients dW_l[m][k] = sum over rows of dZ_l[row][m] H_{l-1}[row][k] from the blocked operands,
// for one layer (blockIdx.y) and one range of row blocks (blockIdx.x): wave w holds the 32 units
// m = 32 (w % (H / 32)).. and all k; with 64 units, waves 2 and 3 take every other block of rows and write
// sums of their own.  MFMA v_mfma_f32_32x32x16_bf16, lane l of 64 (half = l / 32), element j of 8 / e of 16:
//   A[row = l % 32][k = 8 half + j],  B[k = 8 half + j][col = l % 32],
//   D[row = 8 (e / 4) + 4 half + e % 4][col = l % 32]
// Reads both operands once past L2 (126 MB at a batch of 65,536 with 4 layers: 4 gradients and 3 activations of
// 16.8 MB, 8.4 MB of features).
struct WeightArgs {
    int rowBlocks, F, L, splits;
    const uint16_t* phiBlk;
    const uint16_t* actBlk[kFusedLayers];
    const uint16_t* dzBlk[kFusedLayers];
    int64_t wOff[kFusedLayers];
    float* part;       // [splits * 4 / (H / 32)][nParams]
    int64_t nParams;
};

template <int H, int NT>
__device__ __forceinline__ void weightTile(const uint16_t* dz, const uint16_t* in, int rb, int rbEnd, int step, int m0,
                                           int lane, float* dst) {
    constexpr int N = 32 * NT;
    f32x16 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = 0.0f;
    const int ln = lane & 31, half = lane >> 5;
    for (; rb < rbEnd; rb += step) {
        const uint16_t* a = dz + ((int64_t)rb * H + m0 + ln) * 32 + 8 * half;
        const uint16_t* b = in + ((int64_t)rb * N + ln) * 32 + 8 * half;
        const bf16x8 a0 = load8(a), a1 = load8(a + 16);
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const bf16x8 b0 = load8(b + j * 1024), b1 = load8(b + j * 1024 + 16);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, acc[j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) dst[(m0 + 8 * (e / 4) + 4 * half + e % 4) * N + 32 * j + ln] = acc[j][e];
}

template <int H>
__global__ void __launch_bounds__(256) weightKernel(WeightArgs g) {
    constexpr int TM = H / 32, kWays = 4 / TM;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, way = wave / TM, m0 = 32 * (wave % TM);
    const int l = blockIdx.y, per = (g.rowBlocks + g.splits - 1) / g.splits;
    const int rb = blockIdx.x * per, rbEnd = min(g.rowBlocks, rb + per);
    float* dst = g.part + (size_t)(blockIdx.x * kWays + way) * g.nParams + g.wOff[l];
    if (l > 0) weightTile<H, TM>(g.dzBlk[l], g.actBlk[l - 1], rb + way, rbEnd, kWays, m0, lane, dst);
    else if (g.F == 32) weightTile<H, 2>(g.dzBlk[0], g.phiBlk, rb + way, rbEnd, kWays, m0, lane, dst);
    else weightTile<H, 1>(g.dzBlk[0], g.phiBlk, rb + way, rbEnd, kWays, m0, lane, dst);
}

// Adds the partial gradients up (weights: a thread per parameter over the splits; the rest: a wave per
// parameter over the blocks), and takes the Adam step (Kingma & Ba) on the fp32 master weights if asked to.
struct ReduceArgs {
    int64_t nParams, nWeights;      // the first blocks take the weights of the hidden layers
    int H, L, parts, smalls;
    int64_t wOff[kFusedLayers + 1], bOff[kFusedLayers + 1];
    const float* part;
    const float* small;
    const int64_t* weightAt;        // parameter index of the i-th hidden weight
    float* grad;
    float* lossOut;
    int adam;
    float *theta, *m, *v;
    float lr, b1, b2, eps, c1, c2;
    uint16_t *w, *wT;
    const int64_t *at, *atT;        // where a hidden weight lies in them (-1: no hidden weight)
};

__device__ __forceinline__ void adamStep(const ReduceArgs& g, int64_t i, float gr) {
    g.grad[i] = gr;
    if (!g.adam) return;
    const float mi = g.b1 * g.m[i] + (1.0f - g.b1) * gr;
    const float vi = g.b2 * g.v[i] + (1.0f - g.b2) * gr * gr;
    g.m[i] = mi;
    g.v[i] = vi;
    const float t = g.theta[i] - g.lr * (mi / g.c1) / (sqrtf(vi / g.c2) + g.eps);
    g.theta[i] = t;
    if (g.at[i] >= 0) {
        const uint16_t b = bf16Bits(t);
        g.w[g.at[i]] = b;
        g.wT[g.atT[i]] = b;
    }
}

__global__ void __launch_bounds__(256) reduceKernel(ReduceArgs g, int weightBlocks) {
    if ((int)blockIdx.x < weightBlocks) {
        const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (k >= g.nWeights) return;
        const int64_t i = g.weightAt[k];
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        int p = 0;
        for (; p + 4 <= g.parts; p += 4)
#pragma unroll
            for (int u = 0; u < 4; u++) s[u] += g.part[(size_t)(p + u) * g.nParams + i];
        for (; p < g.parts; p++) s[0] += g.part[(size_t)p * g.nParams + i];
        adamStep(g, i, (s[0] + s[1]) + (s[2] + s[3]));
        return;
    }
    const int lane = threadIdx.x & 63, P = (g.L + 1) * g.H + 2;
    const int j = ((int)blockIdx.x - weightBlocks) * 4 + (threadIdx.x >> 6);
    if (j >= P) return;
    float s = 0.0f;
    for (int p = lane; p < g.smalls; p += 64) s += g.small[(size_t)p * P + j];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane) return;
    if (j < g.L * g.H) adamStep(g, g.bOff[j / g.H] + j % g.H, s);
    else if (j < (g.L + 1) * g.H) adamStep(g, g.wOff[g.L] + j - g.L * g.H, s);
    else if (j == (g.L + 1) * g.H) adamStep(g, g.bOff[g.L], s);
    else *g.lossOut = s;
}

// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
// More units, features or layers do not fit a block's registers and LDS.  The smaller shapes between (32 or 96
// units, 8 or 24 frequencies) would, but are not among the kernel's instances: they take a GEMM per layer, 230
// to 330 us per training step of 65,536 rows with 4 layers where the fused shapes around them take 59 to 100.
bool mlpFusable(const MlpShape& s) {
    return (s.hidden == 64 || s.hidden == 128) && (s.nFreq == 16 || s.nFreq == 32) && s.nHidden <= kFusedLayers;
}

static FusedArgs fusedArgs(const MlpDevice& m, const float* x, int n) {
    FusedArgs g{};
    g.n = n; g.d = m.shape.inDim; g.F = m.shape.nFreq;
    g.x = x; g.freq = m.freq; g.theta = m.theta; g.w = m.wBf; g.wT = m.wBfT;
    for (int l = 0; l <= m.shape.nHidden; l++) { g.wOff[l] = m.wOffset[l]; g.bOff[l] = m.bOffset[l]; }
    return g;
}

template <int L, int MODE>
static void launchFusedLayers(const FusedArgs& g, int hidden, int blocks, hipStream_t s) {
    if (hidden == 128) hipLaunchKernelGGL((fusedKernel<128, L, MODE>), dim3(blocks), dim3(1024), 0, s, g);
    else hipLaunchKernelGGL((fusedKernel<64, L, MODE>), dim3(blocks), dim3(512), 0, s, g);
}
template <int MODE>
static hipError_t launchFused(const FusedArgs& g, int layers, int hidden, int blocks, hipStream_t s) {
    switch (layers) {
    case 1: launchFusedLayers<1, MODE>(g, hidden, blocks, s); break;
    case 2: launchFusedLayers<2, MODE>(g, hidden, blocks, s); break;
    case 3: launchFusedLayers<3, MODE>(g, hidden, blocks, s); break;
    case 4: launchFusedLayers<4, MODE>(g, hidden, blocks, s); break;
    default: return hipErrorInvalidValue;   // mlpFusable
    }
    return hipGetLastError();
}

hipError_t mlpFusedEvaluate(MlpDevice& m, const float* x, int n, float* value, float* gradient, hipStream_t s) {
    FusedArgs g = fusedArgs(m, x, n);
    g.out = value;
    g.grad = gradient;
    const int blocks = std::min((n + kRows - 1) / kRows, 2 * kMlpFusedBlocks);
    return gradient ? launchFused<kGradient>(g, m.shape.nHidden, m.shape.hidden, blocks, s)
                    : launchFused<kValue>(g, m.shape.nHidden, m.shape.hidden, blocks, s);
}

// gradients of 0.5 mean (c(x) - y)^2 into m.grad, the loss into m.loss, and the Adam step if lr is given
hipError_t mlpFusedTrain(MlpDevice& m, const float* x, const float* y, int n, const float* lr, hipStream_t s) {
    const int H = m.shape.hidden, L = m.shape.nHidden;
    FusedArgs g = fusedArgs(m, x, n);
    g.y = y;
    g.invN = 1.0f / (float)n;
    WeightArgs w{};
    g.phiBlk = m.phi;
    w.phiBlk = m.phi;
    for (int l = 0; l < L; l++) {
        g.actBlk[l] = m.act[l];
        g.dzBlk[l] = reinterpret_cast<uint16_t*>(m.pre[l]);   // the GEMM path's pre-activations: twice the room
        w.actBlk[l] = g.actBlk[l];
        w.dzBlk[l] = g.dzBlk[l];
        w.wOff[l] = m.wOffset[l];
    }
    g.small = m.partSmall;
    const int tiles = (n + kRows - 1) / kRows, blocks = std::min(tiles, kMlpFusedBlocks);
    hipError_t e = launchFused<kTrain>(g, L, H, blocks, s);
    if (e != hipSuccess) return e;
    w.rowBlocks = 2 * tiles;
    w.F = m.shape.nFreq; w.L = L;
    w.splits = std::min(w.rowBlocks, kMlpSplits);
    w.part = m.part;
    w.nParams = m.nParams;
    if (H == 128) hipLaunchKernelGGL(weightKernel<128>, dim3(w.splits, L), dim3(256), 0, s, w);
    else hipLaunchKernelGGL(weightKernel<64>, dim3(w.splits, L), dim3(256), 0, s, w);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    ReduceArgs r{};
    r.nParams = m.nParams;
    r.nWeights = m.nHiddenWeights;
    r.H = H; r.L = L; r.parts = w.splits * (H == 128 ? 1 : 2); r.smalls = 2 * blocks;
    for (int l = 0; l <= L; l++) { r.wOff[l] = m.wOffset[l]; r.bOff[l] = m.bOffset[l]; }
    r.part = m.part; r.small = m.partSmall; r.weightAt = m.weightAt; r.grad = m.grad; r.lossOut = m.loss;
    r.theta = m.theta; r.m = m.adamM; r.v = m.adamV; r.w = m.wBf; r.wT = m.wBfT; r.at = m.bfIndex; r.atT = m.bfIndexT;
    r.adam = lr != nullptr;
    if (lr) {
        m.step++;
        r.lr = *lr; r.b1 = 0.9f; r.b2 = 0.999f; r.eps = 1e-8f;
        r.c1 = 1.0f - powf(r.b1, (float)m.step);
        r.c2 = 1.0f - powf(r.b2, (float)m.step);
    }
    const int weightBlocks = (int)((r.nWeights + 255) / 256), smallBlocks = ((L + 1) * H + 2 + 3) / 4;
    hipLaunchKernelGGL(reduceKernel, dim3(weightBlocks + smallBlocks), dim3(256), 0, s, r, weightBlocks);
    return hipGetLastError();
}

}  // namespace zg
