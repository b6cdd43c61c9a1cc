// obb_kernel.hip -- oriented child boxes of a boundary's BVH (layout.h), built once per scene.
//
// One wave at a time reads a child slot's primitives (a contiguous range) three times: mean normal and
// mean vertex, in-plane covariance, extents.  The frame is the mean normal with the principal in-plane
// axes; a child whose normals cancel, or whose axis-aligned box is the smaller one, keeps that.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "device.h"
#include "kernels.h"

namespace zg {

ZG_DEV float waveSum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}
ZG_DEV float waveMax(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

template <int D> ZG_DEV Vec<D> primVertex(const float* prims, int i, int v) {
    return vload<D>(prims + (size_t)i * PrimLayout<D>::kFloats + v * D);
}

// Extents of the primitives [r.x, r.x + r.y) in the frame ax: centre (world) and half extents, widened so
// that a distance computed from them in float never exceeds the distance computed to any primitive: the
// projections round at a few ulps of the box's size, the primitives' closest points at a few ulps of
// their coordinates.
template <int D>
ZG_DEV void frameExtents(const float* prims, int2 r, const Vec<D> (&ax)[D], const Vec<D>& origin, int lane, Vec<D>& c,
                         float (&half)[D]) {
    float lo[D], hi[D];
    for (int a = 0; a < D; a++) { lo[a] = FLT_MAX; hi[a] = -FLT_MAX; }
    for (int i = r.x + lane; i < r.x + r.y; i += 64)
        for (int v = 0; v < D; v++) {
            const Vec<D> p = primVertex<D>(prims, i, v) - origin;
            for (int a = 0; a < D; a++) { const float t = dot(ax[a], p); lo[a] = fminf(lo[a], t); hi[a] = fmaxf(hi[a], t); }
        }
    c = origin;
    for (int a = 0; a < D; a++) {
        hi[a] = waveMax(hi[a]); lo[a] = -waveMax(-lo[a]);
        c = c + ax[a] * (0.5f * (lo[a] + hi[a]));
        half[a] = 0.0f;
    }
    // against the rounded centre
    float mag = 0.0f;
    for (int i = r.x + lane; i < r.x + r.y; i += 64)
        for (int v = 0; v < D; v++) {
            const Vec<D> w = primVertex<D>(prims, i, v), p = w - c;
            for (int a = 0; a < D; a++) { half[a] = fmaxf(half[a], fabsf(dot(ax[a], p))); mag = fmaxf(mag, fabsf(w[a])); }
        }
    float size = 0.0f;
    mag = waveMax(mag);
    for (int a = 0; a < D; a++) { half[a] = waveMax(half[a]); size += half[a]; }
    for (int a = 0; a < D; a++) half[a] += 2e-6f * size + 5e-7f * mag;
}
template <int D> ZG_DEV float boxMeasure(const float (&h)[D]) {
    return D == 3 ? h[0] * h[1] + h[1] * h[D - 1] + h[D - 1] * h[0] : h[0] + h[1];
}

// box of child slot s, whose primitives are [r.x, r.x + r.y), by one wave
template <int D, int W>
ZG_DEV void buildBox(const float* nodes, const float* prims, int64_t s, int2 r, int lane, float4* obb) {
    const int code = __float_as_int(nodes[(size_t)(s / W) * NodeLayout<D, W>::kFloats + NodeLayout<D, W>::kChildOffset + s % W]);
    Vec<D> ax[D], c = vzero<D>();
    float half[D];
    for (int a = 0; a < D; a++) { ax[a] = vzero<D>(); ax[a][a] = 1.0f; half[a] = -kEmptyBox; }
    if (r.y > 0) {
        Vec<D> mean = vzero<D>(), nrm = vzero<D>();
        float total = 0.0f;
        for (int i = r.x + lane; i < r.x + r.y; i += 64) {
            for (int v = 0; v < D; v++) mean = mean + primVertex<D>(prims, i, v);
            if constexpr (D == 3) {
                const Vec<3> a = primVertex<3>(prims, i, 0);
                const Vec<3> n = cross3(primVertex<3>(prims, i, 1) - a, primVertex<3>(prims, i, 2) - a);
                nrm = nrm + n;
                total += __builtin_sqrtf(norm2(n));
            }
        }
        for (int a = 0; a < D; a++) { mean[a] = waveSum(mean[a]) / (float)(D * r.y); nrm[a] = waveSum(nrm[a]); }
        total = waveSum(total);
        // plane of the in-plane axes: e0, e1
        Vec<D> e0 = ax[0], e1 = ax[1];
        bool oriented = true;
        if constexpr (D == 3) {
            const float l = __builtin_sqrtf(norm2(nrm));
            oriented = l > 0.3f * total;
            if (oriented) {
                nrm = nrm * (1.0f / l);
                Vec<3> d0 = vzero<3>(), d1 = vzero<3>();
                d0[0] = 1.0f; d1[1] = 1.0f;
                e0 = fromFrame(nrm, d0);
                e1 = fromFrame(nrm, d1);
            }
        }
        frameExtents<D>(prims, r, ax, mean, lane, c, half);   // axis-aligned
        if (oriented) {
            float cxx = 0.0f, cxy = 0.0f, cyy = 0.0f;
            for (int i = r.x + lane; i < r.x + r.y; i += 64)
                for (int v = 0; v < D; v++) {
                    const Vec<D> p = primVertex<D>(prims, i, v) - mean;
                    const float a = dot(p, e0), b = dot(p, e1);
                    cxx += a * a; cxy += a * b; cyy += b * b;
                }
            cxx = waveSum(cxx); cxy = waveSum(cxy); cyy = waveSum(cyy);
            const float ang = 0.5f * atan2f(2.0f * cxy, cxx - cyy);
            Vec<D> f[D], fc;
            float fh[D];
            f[0] = e0 * cosf(ang) + e1 * sinf(ang);
            f[1] = e1 * cosf(ang) - e0 * sinf(ang);
            if constexpr (D == 3) f[D - 1] = nrm;
            frameExtents<D>(prims, r, f, mean, lane, fc, fh);
            if (boxMeasure<D>(fh) < boxMeasure<D>(half)) {
                c = fc;
                for (int a = 0; a < D; a++) { ax[a] = f[a]; half[a] = fh[a]; }
            }
        }
    }
    if (lane) return;
    float4* o = obb + s * ObbLayout<D>::kVec;
    if constexpr (D == 3) {
        o[0] = make_float4(c[0], c[1], c[D - 1], __int_as_float(code));
        for (int a = 0; a < 3; a++) o[1 + a] = make_float4(ax[a][0], ax[a][1], ax[a][D - 1], half[a]);
    } else {
        // the second axis is the first turned by 90 degrees; its sign does not matter
        o[0] = make_float4(c[0], c[1], ax[0][0], ax[0][1]);
        o[1] = make_float4(half[0], half[1], __int_as_float(code), 0.0f);
    }
}

// A wave takes every (4 gridDim.x)-th slot: with a wave per slot, 2^26 slots (some 60 million triangles in a
// 4-wide tree) would need more than the 2^32 threads of a launch.
constexpr int64_t kObbBlocks = 8192;

template <int D, int W>
__global__ void __launch_bounds__(256) buildObbKernel(const float* __restrict__ nodes, const float* __restrict__ prims,
                                                      int nNodes, const int2* __restrict__ ranges,
                                                      float4* __restrict__ obb) {
    for (int64_t s = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); s < (int64_t)nNodes * W; s += (int64_t)gridDim.x * 4)
        buildBox<D, W>(nodes, prims, s, ranges[s], threadIdx.x & 63, obb);
}

hipError_t launchBuildObb(const float* nodes, const float* prims, int dim, int width, int nNodes, const int2* ranges,
                          float4* obb, hipStream_t s) {
    if (nNodes <= 0) return hipSuccess;
    dim3 g((unsigned)std::min(kObbBlocks, ((int64_t)nNodes * width + 3) / 4)), bl(256);
    if (dim == 2 && width == 4) hipLaunchKernelGGL((buildObbKernel<2, 4>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else if (dim == 2) hipLaunchKernelGGL((buildObbKernel<2, 8>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else if (width == 4) hipLaunchKernelGGL((buildObbKernel<3, 4>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else hipLaunchKernelGGL((buildObbKernel<3, 8>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    return hipGetLastError();
}

// One thread builds one entry node: the cover starts as the root's children within reach, and its largest
// inner item is replaced by that item's children within reach for as long as the result fits in W slots, so
// that an entry sits as deep in the tree as W items allow.
template <int D, int W>
__global__ void __launch_bounds__(256) buildEntriesKernel(const float* __restrict__ nodes, int nNodes,
                                                          const int32_t* __restrict__ leafSlots, int nLeaves,
                                                          float4* __restrict__ obb, float2* __restrict__ primEntry) {
    using L = NodeLayout<D, W>;
    constexpr int V = ObbLayout<D>::kVec;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)nLeaves * kEntryLevels) return;
    const int leaf = (int)(t / kEntryLevels), level = (int)(t % kEntryLevels);
    const float* ln = nodes + (size_t)(leafSlots[leaf] / W) * L::kFloats;
    const int slot = leafSlots[leaf] % W;
    float lo[D], hi[D], diag2 = 0.0f, mag = 0.0f;
    for (int a = 0; a < D; a++) {
        lo[a] = ln[a * W + slot];
        hi[a] = ln[(D + a) * W + slot];
        diag2 += (hi[a] - lo[a]) * (hi[a] - lo[a]);
        mag = fmaxf(mag, fmaxf(fabsf(lo[a]), fabsf(hi[a])));
    }
    float reach = kEntryReach * __builtin_sqrtf(diag2);
    if (level == 0) {
        const int code = __float_as_int(ln[L::kChildOffset + slot]);
        const int first = leafFirstD(code), cnt = leafCountD(code);
        for (int i = first; i < first + cnt; i++)
            primEntry[i] = make_float2(0.25f * reach * reach, __int_as_float(nNodes + leaf * kEntryLevels));
    }
    // the cover's radius: the reach plus what rounding can add to the distances that are compared with it
    // (coordinates of magnitude mag leave a few ulps of mag in a computed distance)
    for (int j = 0; j < level; j++) reach *= kEntryRatio;
    reach = reach * 1.001f + 8e-6f * mag;
    const float reach2 = reach * reach;

    int src[W], code[W];   // child slot (node * W + k) an item comes from, and its code
    float size[W];
    bool open[W];          // an inner item that may still be replaced by its children
    int n = 1;
    src[0] = 0; code[0] = 0; open[0] = true; size[0] = FLT_MAX;   // the root: replaced at once
    for (;;) {
        int pick = -1;
        for (int i = 0; i < n; i++)
            if (open[i] && (pick < 0 || size[i] > size[pick])) pick = i;
        if (pick < 0) break;
        const int node = code[pick];
        const float* nd = nodes + (size_t)node * L::kFloats;
        int keep[W], m = 0;
        for (int k = 0; k < W; k++) {
            if (L::emptySlot(nd, k)) continue;
            float d2 = 0.0f;
            for (int a = 0; a < D; a++) {
                const float g = fmaxf(fmaxf(nd[a * W + k] - hi[a], lo[a] - nd[(D + a) * W + k]), 0.0f);
                d2 += g * g;
            }
            if (!(d2 > reach2)) keep[m++] = k;
        }
        if (n - 1 + m > W) { open[pick] = false; continue; }
        n--;   // the picked item leaves, its children within reach enter
        src[pick] = src[n]; code[pick] = code[n]; open[pick] = open[n]; size[pick] = size[n];
        for (int q = 0; q < m; q++, n++) {
            const int k = keep[q];
            src[n] = node * W + k;
            code[n] = __float_as_int(nd[L::kChildOffset + k]);
            open[n] = !isLeaf(code[n]);
            size[n] = 0.0f;
            for (int a = 0; a < D; a++) size[n] += nd[(D + a) * W + k] - nd[a * W + k];
        }
    }
    float4* out = obb + (size_t)(nNodes + (int64_t)leaf * kEntryLevels + level) * W * V;
    for (int k = 0; k < W; k++)
        for (int v = 0; v < V; v++) {
            // an empty slot
            const float none = __int_as_float(kEmptyChild);
            float4 e = D == 3 ? make_float4(0.0f, 0.0f, 0.0f, v ? -kEmptyBox : none)
                              : (v ? make_float4(-kEmptyBox, -kEmptyBox, none, 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
            if (k < n) e = obb[(size_t)src[k] * V + v];
            out[k * V + v] = e;
        }
}

hipError_t launchBuildEntries(const float* nodes, int dim, int width, int nNodes, const int32_t* leafSlots, int nLeaves,
                              float4* obb, float2* primEntry, hipStream_t s) {
    if (nLeaves <= 0) return hipSuccess;
    dim3 g((unsigned)(((int64_t)nLeaves * kEntryLevels + 255) / 256)), bl(256);
    if (dim == 2 && width == 4) hipLaunchKernelGGL((buildEntriesKernel<2, 4>), g, bl, 0, s, nodes, nNodes, leafSlots, nLeaves, obb, primEntry);
    else if (dim == 2) hipLaunchKernelGGL((buildEntriesKernel<2, 8>), g, bl, 0, s, nodes, nNodes, leafSlots, nLeaves, obb, primEntry);
    else if (width == 4) hipLaunchKernelGGL((buildEntriesKernel<3, 4>), g, bl, 0, s, nodes, nNodes, leafSlots, nLeaves, obb, primEntry);
    else hipLaunchKernelGGL((buildEntriesKernel<3, 8>), g, bl, 0, s, nodes, nNodes, leafSlots, nLeaves, obb, primEntry);
    return hipGetLastError();
}

}  // namespace zg
