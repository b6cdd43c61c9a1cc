// obb_kernel.hip -- oriented child boxes of a boundary's BVH (layout.h), built once per scene.
//
// One wave per child slot reads the child's primitives (a contiguous range) three times: mean normal and
// mean vertex, in-plane covariance, extents.  The frame is the mean normal with the principal in-plane
// axes; a child whose normals cancel, or whose axis-aligned box is the smaller one, keeps that.
#include <hip/hip_runtime.h>

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

template <int D, int W>
__global__ void __launch_bounds__(256) buildObbKernel(const float* __restrict__ nodes, const float* __restrict__ prims,
                                                      int nNodes, const int2* __restrict__ ranges,
                                                      float4* __restrict__ obb) {
    const int64_t s = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (s >= (int64_t)nNodes * W) return;
    const int2 r = ranges[s];
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

hipError_t launchBuildObb(const float* nodes, const float* prims, int dim, int width, int nNodes, const int2* ranges,
                          float4* obb, hipStream_t s) {
    if (nNodes <= 0) return hipSuccess;
    dim3 g((unsigned)(((int64_t)nNodes * width + 3) / 4)), bl(256);
    if (dim == 2 && width == 4) hipLaunchKernelGGL((buildObbKernel<2, 4>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else if (dim == 2) hipLaunchKernelGGL((buildObbKernel<2, 8>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else if (width == 4) hipLaunchKernelGGL((buildObbKernel<3, 4>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    else hipLaunchKernelGGL((buildObbKernel<3, 8>), g, bl, 0, s, nodes, prims, nNodes, ranges, obb);
    return hipGetLastError();
}

}  // namespace zg
