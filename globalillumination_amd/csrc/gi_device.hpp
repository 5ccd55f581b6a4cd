// gi_device.hpp — device-side arithmetic shared by the gfx950 kernels.
//
// Numerics contract: every kernel is compiled with -ffp-contract=off, so each
// a*b+c below is a rounded multiply then a rounded add, in the order written;
// FP32 division and sqrt are IEEE correctly rounded (the HIP default).  GLSL
// built-ins are implemented with their GLSL-spec definitions so results are
// reproducible on any IEEE machine:
//   mix(x,y,a) = x*(1-a) + y*a     max(x,y) = x < y ? y : x
//   min(x,y)   = y < x ? y : x     clamp(x,a,b) = min(max(x,a),b)
//   fract(x)   = x - floor(x)      normalize(v) = v * (1/sqrt(dot(v,v)))
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gi {

__device__ __forceinline__ float gmax(float x, float y) { return x < y ? y : x; }
__device__ __forceinline__ float gmin(float x, float y) { return y < x ? y : x; }
__device__ __forceinline__ float gclamp(float x, float a, float b) { return gmin(gmax(x, a), b); }
__device__ __forceinline__ float gmix(float x, float y, float a) { return x * (1.0f - a) + y * a; }
__device__ __forceinline__ float gfract(float x) { return x - floorf(x); }
__device__ __forceinline__ float le01(float z, float d) { return (z <= d) ? 1.0f : 0.0f; }

// Shadow-map texel at (s, t): GL_NEAREST, CLAMP_TO_BORDER with border depth 0
// (ShadowMapping/src/Viewers/MyGLTextureViewer.cpp:3-28).  Out-of-range
// coordinates (and NaN) read the border, i.e. count as shadowed.
struct DepthMap {
    const float* __restrict__ texels;
    int w, h;
    float fw, fh;  // (float)w, (float)h

    __device__ __forceinline__ bool inside(float u, float v) const {
        return u >= 0.0f && u < fw && v >= 0.0f && v < fh;
    }
    // Texel (u, v) inside the map; row and width are below 2^24 and the texel
    // index below 2^28 (GI_MAX_EDGE).
    __device__ __forceinline__ float texel(float u, float v, bool in) const {
        const uint32_t k = in ? __umul24((uint32_t)(int)v, (uint32_t)w) + (uint32_t)(int)u : 0u;
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(texels) + k * 4u);
    }
    __device__ __forceinline__ float fetch(float s, float t) const {
        const float u = s * fw, v = t * fh;
        if (!inside(u, v)) return 0.0f;
        return texel(u, v, true);
    }
    // The same without a branch (texel 0 is loaded where the coordinates are
    // outside): the fetches of a tap loop are then in flight together, where
    // behind a branch each waits for the one before it.  For tap loops; in the
    // edge walks, whose fetches depend on one another and whose lanes end at
    // different steps, it costs more than it hides (RPCF's taps on a
    // 200k-triangle soup at 1080p: 131 us with it, 101 us without; 115 us with
    // a floor and a 64-bit offset per fetch).
    __device__ __forceinline__ float fetch_all(float s, float t) const {
        const float u = s * fw, v = t * fh;
        const bool in = inside(u, v);
        const float d = texel(u, v, in);
        return in ? d : 0.0f;
    }
};

// M * (x, y, z, w) with GLSL column-major order, summed left to right.
__device__ __forceinline__ void mat4_vec4(const float* m, float x, float y, float z, float w,
                                          float o[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float acc = m[0 * 4 + i] * x;
        acc = acc + m[1 * 4 + i] * y;
        acc = acc + m[2 * 4 + i] * z;
        acc = acc + m[3 * 4 + i] * w;
        o[i] = acc;
    }
}

__device__ __forceinline__ void normalize3(const float v[3], float o[3]) {
    float sqr = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    float inv = 1.0f / sqrtf(sqr);
    o[0] = v[0] * inv;
    o[1] = v[1] * inv;
    o[2] = v[2] * inv;
}

// Kernel-argument copies of small matrices (passed by value).
struct Mat4 { float m[16]; };
struct Mat3 { float m[9]; };

}  // namespace gi
