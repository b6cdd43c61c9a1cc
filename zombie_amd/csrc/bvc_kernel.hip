// bvc_kernel.hip -- boundary value caching splat for gfx950
// (variance_reduction/boundary_value_caching.h:370-402 splat, :683-810 splatBoundaryData /
// splatSourceData, core/distributions.h:12-55 kernel regularization, :84-177 free-space harmonic
// and :271-321 3D Yukawa Green's functions and Poisson kernels with their gradients).
//
// Every evaluation point x receives one estimate per cached sample y: the boundary term of
// Green's representation formula (Dirichlet, Neumann or Robin form) or the source term, each
// divided by the sample's density.  The work is an all-pairs gather.  One wave owns 64 evaluation
// points and a chunk of the samples; it stages 256 samples at a time in LDS, sorted by category, as
// records (y, A, n, B) with which every form of the estimate is alpha (G A - P B) and its gradient
// alphaG (grad G A - grad P B), so that the divisions by density and Robin coefficient are made once per
// sample and not per pair.  Sums and sums of squares are FP64.
//
// Bound: VALU issue (about 50 FP32 and 12 FP64 instructions per pair in 3D).  Splitting the samples
// over blockIdx.y keeps the chip full when the evaluation points alone are too few waves; the chunks'
// sums then go through a workspace that a second kernel adds up in order.  10,000 points x (40,000
// boundary + 10,000 source samples) in 3D, both splats: 38.5 ms with one 256-thread block per 256 points and
// the divisions in the loop, 1.0 ms now among other calls and 1.4 alone (2D: 32.8, 0.9 and 1.0).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "../../include/zombie_amd.h"
#include "device.h"
#include "kernels.h"

namespace zg {

constexpr int kBvcTile = 256;
constexpr int kBvcCats = 5;   // absorbing, absorbing aligned, reflecting, reflecting aligned, source

struct BvcParams {
    zg_bvc_samples S;
    zg_bvc_eval_points E;
    zg_bvc_statistics out;
    float radiusClamp, kreg, robinCutoff, cutoffA, cutoffR;
    float mu;   // sqrt(absorption): 3D Yukawa kernels when > 0
    int64_t chunk;        // samples per blockIdx.y, a multiple of kBvcTile
    double* sums;         // with several chunks: [chunk][category][2 + 2 D][E.n]
    int32_t* counts;      //                      [chunk][category][E.n]
    uint32_t* present;    //                      [chunk] categories that the chunk holds (bit mask)
};

template <int D>
struct BvcSums {
    int n;
    double s, q, gs[D], gq[D];
};

// The loops multiply every estimate by 1 / (4 pi), in 2D 1 / (2 pi), rounded to 32 bits: an error of 4e-8 that all
// pairs share, where their other roundings average out.  kUnround takes it out of the 64-bit sums.
constexpr float kInv4Pi = 0.25f / kPi, kLn2 = 0.69314718055994530942f;
constexpr double kUnround = 0.25 / 3.14159265358979323846 / (double)kInv4Pi;

// Chan merge of a batch into the caller's statistics of point i, category c (common.h:268-310)
template <int D>
ZG_DEV void bvcMerge(const zg_bvc_statistics& out, int64_t i, int c, BvcSums<D> b) {
    if (b.n == 0) return;
    b.s *= kUnround;
    b.q *= kUnround * kUnround;
#pragma unroll
    for (int a = 0; a < D; a++) { b.gs[a] *= kUnround; b.gq[a] *= kUnround * kUnround; }
    const size_t k = (size_t)i * kBvcCats + c;
    const int64_t N1 = out.n[k], nb = b.n, N = N1 + nb;
    const double f2 = (double)nb / (double)N, f12 = (double)N1 * (double)nb / (double)N;
    const double mB = b.s / (double)nb, m2B = fmax(0.0, b.q - b.s * mB);
    if (N1 == 0) { out.solution_mean[k] = mB; out.solution_m2[k] = m2B; }
    else {
        const double d = mB - out.solution_mean[k];
        out.solution_mean[k] += d * f2;
        out.solution_m2[k] += m2B + d * d * f12;
    }
#pragma unroll
    for (int a = 0; a < D; a++) {
        const size_t kg = k * D + a;
        const double gm = b.gs[a] / (double)nb, g2 = fmax(0.0, b.gq[a] - b.gs[a] * gm);
        if (N1 == 0) { out.gradient_mean[kg] = gm; out.gradient_m2[kg] = g2; }
        else {
            const double d = gm - out.gradient_mean[kg];
            out.gradient_mean[kg] += d * f2;
            out.gradient_m2[kg] += g2 + d * d * f12;
        }
    }
    out.n[k] = N;
}

// points whose statistics a splat leaves alone: those within a cutoff of the boundary
ZG_DEV bool bvcActive(const BvcParams& B, int64_t i) {
    if (i >= B.E.n) return false;
    const float dA = B.E.dist_to_absorbing_boundary[i];
    const float dR = B.E.dist_to_reflecting_boundary ? B.E.dist_to_reflecting_boundary[i] : FLT_MAX;
    return !(dA < B.cutoffA || dR < B.cutoffR);
}

template <int D, bool YUKAWA, bool KREG>
__global__ void __launch_bounds__(64) bvcSplatKernel(BvcParams B) {
    __shared__ float4 sY[kBvcTile], sN[kBvcTile];   // (y, A) and (n, B) of the tile's samples, by category

    const int lane = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * 64 + lane;
    const bool active = bvcActive(B, i);
    Vec<D> x = vzero<D>();
    float alpha = 1.0f, alphaG = 1.0f;
    if (active) {
        uint8_t ty = B.E.type ? B.E.type[i] : (uint8_t)ZG_SAMPLE_IN_DOMAIN;
        if (ty == ZG_SAMPLE_ON_ABSORBING_BOUNDARY || ty == ZG_SAMPLE_ON_REFLECTING_BOUNDARY) { alpha = 2.0f; alphaG = 0.0f; }
        x = vload<D>(B.E.pt + (size_t)i * D);
    }
    BvcSums<D> acc[kBvcCats];
#pragma unroll
    for (int c = 0; c < kBvcCats; c++) acc[c] = BvcSums<D>{};
    uint32_t present = 0;

    const int64_t begin = (int64_t)blockIdx.y * B.chunk, end = min(B.S.n, begin + B.chunk);
    for (int64_t base = begin; base < end; base += kBvcTile) {
        __syncthreads();
        // four samples per lane, placed by category (a stable counting sort with ballots)
        int cat[4], count[kBvcCats] = {0, 0, 0, 0, 0};
        float4 ry[4], rn[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int64_t j = base + 64 * g + lane;
            cat[g] = -1;
            if (j < end) {
                const uint8_t ty = B.S.type[j];
                const bool src = ty == ZG_SAMPLE_IN_DOMAIN;
                const bool al = B.S.normal_aligned && B.S.normal_aligned[j];
                const float sgn = al ? -1.0f : 1.0f;
                float y[3] = {0.0f, 0.0f, 0.0f}, n[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int a = 0; a < D; a++) {
                    y[a] = B.S.pt[(size_t)j * D + a];
                    n[a] = src ? 0.0f : sgn * B.S.normal[(size_t)j * D + a];
                }
                const float pdf = B.S.pdf[j], u = B.S.solution[j], dn = B.S.normal_derivative[j];
                const float h = B.S.contribution ? B.S.contribution[j] : 0.0f;
                const float kappa = B.S.robin_coeff ? B.S.robin_coeff[j] : 0.0f;
                // source: G h / pdf.  Boundary: (G dn - P u) / pdf; with a Robin coefficient beyond the
                // cutoff ((G + P / kappa) dn - P h / kappa) / pdf, up to it (G h - (P + kappa G) u) / pdf
                float A = dn / pdf, Bc = u / pdf;
                if (src) { A = h / pdf; Bc = 0.0f; }
                else if (fabsf(kappa) > B.robinCutoff) Bc = (h - dn) / (kappa * pdf);
                else if (fabsf(kappa) > 0.0f) A = (h - kappa * u) / pdf;
                ry[g] = make_float4(y[0], y[1], y[2], A);
                rn[g] = make_float4(n[0], n[1], n[2], Bc);
                cat[g] = src ? 4 : (ty == ZG_SAMPLE_ON_ABSORBING_BOUNDARY ? 0 : 2) + (al ? 1 : 0);
            }
#pragma unroll
            for (int c = 0; c < kBvcCats; c++) count[c] += (int)__popcll(__ballot(cat[g] == c));
        }
        int first = 0;
#pragma unroll
        for (int c = 0; c < kBvcCats; c++) {
            int at = first;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint64_t mine = __ballot(cat[g] == c);
                if (cat[g] == c) {
                    const int k = at + (int)mbcnt64(mine);
                    sY[k] = ry[g];
                    sN[k] = rn[g];
                }
                at += (int)__popcll(mine);
            }
            first += count[c];
            present |= count[c] ? 1u << c : 0u;
        }
        __syncthreads();
        if (!active) continue;
        int t = 0;
#pragma unroll
        for (int c = 0; c < kBvcCats; c++) {
            BvcSums<D>& s = acc[c];
            const int stop = t + count[c];
            for (; t < stop; t++) {
                const float4 fy = sY[t], fn = sN[t];
                const float yv[3] = {fy.x, fy.y, fy.z}, nv[3] = {fn.x, fn.y, fn.z};
                Vec<D> n, xy;
#pragma unroll
                for (int a = 0; a < D; a++) { n[a] = nv[a]; xy[a] = x[a] - yv[a]; }
                // r = max(clamp, |x - y|) and 1 / r by a reciprocal square root and a Newton step (below an ulp)
                const float r2 = fmaxf(B.radiusClamp * B.radiusClamp, norm2(xy));
                float inv = __builtin_amdgcn_rsqf(r2);
                inv = fmaf(0.5f * inv, fmaf(-(r2 * inv), inv, 1.0f), inv);
                const float inv2 = inv * inv, nx = dot(n, xy);
                // free-space kernels, gradients in the pole x: harmonic (distributions.h:84-177), or in
                // 3D with absorption the Yukawa ones (:271-321) with q1 = e^{-mu r} (mu r + 1):
                // G = e^{-mu r} / (4 pi r), grad G = -(x - y) q1 / (4 pi r^3), P = n.(x - y) q1 / (4 pi r^3),
                // grad P = [n q1 - (x - y) (n.(x - y) / r^2) e^{-mu r} (mu^2 r^2 + 3 mu r + 3)] / (4 pi r^3)
                // (the derivative of P; mu = 0 gives the harmonic kernels); in 2D G = -log(r) / (2 pi),
                // grad G = -(x - y) / (2 pi r^2), P = n.(x - y) / (2 pi r^2),
                // grad P = [n - (x - y) 2 n.(x - y) / r^2] / (2 pi r^2)
                float G, K, Q;   // grad G = -(x - y) K, P = n.(x - y) K, grad P = n K - (x - y) Q
                if constexpr (D == 2) {
                    // v_log_f32 rounds down, which over many pairs is a common error of half an ulp (4e-8), in logf
                    // too; that of -log(1 / r2) is the opposite
                    const float l2 = __builtin_amdgcn_logf(inv2) - __builtin_amdgcn_logf(r2);
                    G = l2 * (0.5f * kLn2) * kInv4Pi;
                    K = inv2 * (2.0f * kInv4Pi);
                    Q = 2.0f * (nx * inv2) * K;
                } else {
                    const float g0 = inv * kInv4Pi, g2 = inv2 * g0;
                    if constexpr (YUKAWA) {
                        const float mr = B.mu * (r2 * inv), e = expf(-mr);
                        G = e * g0;
                        K = e * (mr + 1.0f) * g2;
                        Q = (nx * inv2) * (e * ((mr + 3.0f) * mr + 3.0f)) * g2;
                    } else {
                        G = g0;
                        K = g2;
                        Q = 3.0f * (nx * inv2) * K;
                    }
                }
                float P = nx * K;
                Vec<D> dG, dP;
#pragma unroll
                for (int a = 0; a < D; a++) { dG[a] = -(xy[a] * K); dP[a] = n[a] * K - xy[a] * Q; }
                // samples whose kernels or gradients overflow are left out (source samples: n = 0, P = 0)
                if (!isfinite(fabsf(G) + fabsf(P) + norm2(dG) + norm2(dP))) continue;
                if constexpr (KREG) {
                    const float rr = (r2 * inv) / B.kreg;
                    if constexpr (D == 2) {
                        P *= 1.0f - expf(-rr * rr);
                    } else {
                        const float e = erff(rr);
                        G *= e;
                        P *= e - 2.0f * rr * expf(-rr * rr) / sqrtf(kPi);
                    }
                }
                const double e = (double)(alpha * (G * fy.w - P * fn.w));
                s.n++; s.s += e; s.q += e * e;
#pragma unroll
                for (int a = 0; a < D; a++) {
                    const double g = (double)(alphaG * (dG[a] * fy.w - dP[a] * fn.w));
                    s.gs[a] += g; s.gq[a] += g * g;
                }
            }
        }
    }
    if (gridDim.y == 1) {
        if (!active) return;
#pragma unroll
        for (int c = 0; c < kBvcCats; c++) bvcMerge<D>(B.out, i, c, acc[c]);
        return;
    }
    if (blockIdx.x == 0 && lane == 0) B.present[blockIdx.y] = present;
    if (!active) return;
#pragma unroll
    for (int c = 0; c < kBvcCats; c++) {
        if (!(present >> c & 1u)) continue;
        const size_t row = (size_t)blockIdx.y * kBvcCats + c;
        double* o = B.sums + row * (2 + 2 * D) * (size_t)B.E.n + i;
        B.counts[row * (size_t)B.E.n + i] = acc[c].n;
        o[0] = acc[c].s;
        o[B.E.n] = acc[c].q;
#pragma unroll
        for (int a = 0; a < D; a++) {
            o[(size_t)(2 + a) * B.E.n] = acc[c].gs[a];
            o[(size_t)(2 + D + a) * B.E.n] = acc[c].gq[a];
        }
    }
}

// adds the chunks' sums of a point and category in order and merges them
template <int D>
__global__ void __launch_bounds__(256) bvcMergeKernel(BvcParams B, int chunks) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = blockIdx.y;
    if (!bvcActive(B, i)) return;
    BvcSums<D> t{};
    for (int k = 0; k < chunks; k++) {
        if (!(B.present[k] >> c & 1u)) continue;
        const size_t row = (size_t)k * kBvcCats + c;
        const double* o = B.sums + row * (2 + 2 * D) * (size_t)B.E.n + i;
        t.n += B.counts[row * (size_t)B.E.n + i];
        t.s += o[0];
        t.q += o[B.E.n];
#pragma unroll
        for (int a = 0; a < D; a++) {
            t.gs[a] += o[(size_t)(2 + a) * B.E.n];
            t.gq[a] += o[(size_t)(2 + D + a) * B.E.n];
        }
    }
    bvcMerge<D>(B.out, i, c, t);
}

template <int D>
static void launchSplat(const BvcParams& B, dim3 g, hipStream_t s) {
    if (D == 3 && B.mu > 0.0f) {
        if (B.kreg > 0.0f) hipLaunchKernelGGL((bvcSplatKernel<3, true, true>), g, dim3(64), 0, s, B);
        else hipLaunchKernelGGL((bvcSplatKernel<3, true, false>), g, dim3(64), 0, s, B);
    } else {
        if (B.kreg > 0.0f) hipLaunchKernelGGL((bvcSplatKernel<D, false, true>), g, dim3(64), 0, s, B);
        else hipLaunchKernelGGL((bvcSplatKernel<D, false, false>), g, dim3(64), 0, s, B);
    }
}

hipError_t launchBvcSplat(int dim, float absorption, const zg_bvc_samples& S, const zg_bvc_eval_points& E,
                          const zg_bvc_statistics& out, float radiusClamp, float kreg, float robinCutoff, float cutoffA,
                          float cutoffR, int targetWaves, hipStream_t s) {
    if (E.n <= 0 || S.n <= 0) return hipSuccess;
    BvcParams B{S, E, out, radiusClamp, kreg, robinCutoff, cutoffA, cutoffR, sqrtf(fmaxf(absorption, 0.0f)), 0, nullptr, nullptr, nullptr};
    // as many chunks of whole tiles as fill the chip
    const int64_t waves = (E.n + 63) / 64, tiles = (S.n + kBvcTile - 1) / kBvcTile;
    int64_t chunks = std::min({tiles, (targetWaves + waves - 1) / waves, (int64_t)65535});
    const int64_t perChunk = (tiles + chunks - 1) / chunks;
    chunks = (tiles + perChunk - 1) / perChunk;
    // the workspace is stream-ordered; a call that is being captured, or that finds no memory, runs in one
    // chunk, which needs none
    void* ws = nullptr;
    if (chunks > 1) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) chunks = 1;
    }
    if (chunks > 1) {
        const size_t rows = (size_t)chunks * kBvcCats * (size_t)E.n;
        const size_t sumBytes = rows * (2 + 2 * dim) * sizeof(double), countBytes = rows * sizeof(int32_t);
        if (hipMallocAsync(&ws, sumBytes + countBytes + (size_t)chunks * sizeof(uint32_t), s) == hipSuccess) {
            B.sums = static_cast<double*>(ws);
            B.counts = reinterpret_cast<int32_t*>(static_cast<char*>(ws) + sumBytes);
            B.present = reinterpret_cast<uint32_t*>(static_cast<char*>(ws) + sumBytes + countBytes);
        } else {
            (void)hipGetLastError();
            ws = nullptr;
            chunks = 1;
        }
    }
    B.chunk = chunks > 1 ? perChunk * kBvcTile : tiles * kBvcTile;
    dim3 g((unsigned)waves, (unsigned)chunks);
    if (dim == 2) launchSplat<2>(B, g, s);
    else launchSplat<3>(B, g, s);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && chunks > 1) {
        dim3 m((unsigned)((E.n + 255) / 256), kBvcCats);
        if (dim == 2) hipLaunchKernelGGL(bvcMergeKernel<2>, m, dim3(256), 0, s, B, (int)chunks);
        else hipLaunchKernelGGL(bvcMergeKernel<3>, m, dim3(256), 0, s, B, (int)chunks);
        e = hipGetLastError();
    }
    if (ws) {
        const hipError_t ef = hipFreeAsync(ws, s);
        if (e == hipSuccess) e = ef;
    }
    return e;
}

}  // namespace zg
