// raster_kernels.hpp — device side of the binned raster (see raster.hip for
// the design and the raster rules).  Included by raster.hip (single-instance
// passes) and batch.hip (batched passes); everything here has internal
// linkage, so each translation unit holds its own instantiations.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/gi.h"
#include "gi_device.hpp"

namespace gi {
namespace {


// Tile edge of the binned raster: a template parameter of every tile-shaped
// kernel.  The single-instance passes use kTile; the batched path picks 32 or
// 64 per batch.
constexpr int kTile = 64;
constexpr int kRasterThreads = 256;
constexpr float kGuard = 4.0f;
constexpr int kMaxPoly = 9;
// 28 setup records (64 B each) beside the 18 KiB tile and the record count
// keep a workgroup's LDS at 20,228 bytes, so 8 workgroups fit in a CU's
// 160 KiB (7 of 20,484 bytes ran 3% slower).
constexpr int kRecQueue = 28;  // at most 31; LDS setup records that a workgroup puts aside
constexpr int kShareList = 128;   // entries up to which a tile's list counts as short
constexpr int kShareBlocks = 4;       // blocks over which a record of a short list is put aside
constexpr int kShareBlocksLong = 44;  // and of a long one
constexpr int kScanThreads = 1024;

struct MeshView {
    const float* __restrict__ pos;  // nverts x 3
    const float* __restrict__ nrm;  // nverts x 3 or null
    const int* __restrict__ idx;    // ntris x 3
    int nt;
};

// Per-map transform: a device array of 16-float matrices, or one by value.
struct MvpSource {
    const float* __restrict__ dev;
    Mat4 single;
    __device__ __forceinline__ void load(int map, float m[16]) const {
        if (dev) {
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = dev[16 * map + i];
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = single.m[i];
        }
    }
};

struct RasterCfg {
    int w, h;
    int tiles_x, tiles_y;
    float off_factor, off_units;
};

template <int NA>
struct CV {
    float c[4];
    float a[NA > 0 ? NA : 1];
};

template <int NA>
struct Tri {
    // 24.8 fixed-point window coordinates: within the guard band (|x_ndc| <=
    // kGuard) and a view of at most GI_MAX_EDGE pixels they stay below 2^24
    // in magnitude, so they, their differences and pixel-centre offsets fit
    // in int32; edge functions and areas are formed as 32 x 32 -> 64-bit
    // products.
    int X[3], Y[3];
    float w[3];
    float a[3][NA > 0 ? NA : 1];
    int front;
    int px0, px1, py0, py1;
    int tl[3];
    float z0, A, B, zoff;  // depth plane about vertex 0, per 1/256 pixel
};


__device__ __forceinline__ float plane_dist(const float c[4], int p) {
    switch (p) {
    case 0: return c[2] + c[3];
    case 1: return c[3] - c[2];
    case 2: return c[0] + kGuard * c[3];
    case 3: return kGuard * c[3] - c[0];
    case 4: return c[1] + kGuard * c[3];
    default: return kGuard * c[3] - c[1];
    }
}

template <int NA>
__device__ __forceinline__ void load_vertex(const MeshView& m, const float mvp[16], int vi, CV<NA>& v) {
    const float x = m.pos[3 * vi + 0], y = m.pos[3 * vi + 1], z = m.pos[3 * vi + 2];
    mat4_vec4(mvp, x, y, z, 1.0f, v.c);
    if constexpr (NA == 6) {
        v.a[0] = x;
        v.a[1] = y;
        v.a[2] = z;
        v.a[3] = m.nrm[3 * vi + 0];
        v.a[4] = m.nrm[3 * vi + 1];
        v.a[5] = m.nrm[3 * vi + 2];
    }
}

template <int NA>
__device__ void load_tri(const MeshView& m, const float mvp[16], int tri, CV<NA> v[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) load_vertex<NA>(m, mvp, m.idx[3 * tri + k], v[k]);
}

template <int NA>
__device__ __forceinline__ void lerp_cv(const CV<NA>& in, const CV<NA>& out, float din, float dout,
                                        CV<NA>& r) {
    float t = din / (din - dout);
#pragma unroll
    for (int k = 0; k < 4; ++k) r.c[k] = in.c[k] + t * (out.c[k] - in.c[k]);
#pragma unroll
    for (int k = 0; k < NA; ++k) r.a[k] = in.a[k] + t * (out.a[k] - in.a[k]);
}

// Fills `t` from three clip-space vertices.  Returns false for an empty piece.
template <int NA>
__device__ bool setup_piece(const CV<NA>& v0, const CV<NA>& v1, const CV<NA>& v2, const RasterCfg& cfg,
                            Tri<NA>& t) {
    const CV<NA>* vs[3] = {&v0, &v1, &v2};
    float hw = (float)cfg.w * 0.5f, hh = (float)cfg.h * 0.5f;
    float z[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float* c = vs[i]->c;
        if (!(c[3] > 0.0f)) return false;
        float xn = c[0] / c[3], yn = c[1] / c[3], zn = c[2] / c[3];
        float xw = xn * hw + hw;
        float yw = yn * hh + hh;
        z[i] = zn * 0.5f + 0.5f;
        t.X[i] = (int)rintf(xw * 256.0f);
        t.Y[i] = (int)rintf(yw * 256.0f);
        t.w[i] = c[3];
#pragma unroll
        for (int q = 0; q < NA; ++q) t.a[i][q] = vs[i]->a[q];
    }
    long long area = (long long)(t.X[1] - t.X[0]) * (t.Y[2] - t.Y[0]) - (long long)(t.Y[1] - t.Y[0]) * (t.X[2] - t.X[0]);
    if (area == 0) return false;
    t.front = area > 0;
    if (area < 0) {
        int sx = t.X[1]; t.X[1] = t.X[2]; t.X[2] = sx;
        int sy = t.Y[1]; t.Y[1] = t.Y[2]; t.Y[2] = sy;
        float sz = z[1]; z[1] = z[2]; z[2] = sz;
        float sw = t.w[1]; t.w[1] = t.w[2]; t.w[2] = sw;
#pragma unroll
        for (int q = 0; q < NA; ++q) { float sa = t.a[1][q]; t.a[1][q] = t.a[2][q]; t.a[2][q] = sa; }
        area = -area;
    }
    int minX = min(t.X[0], min(t.X[1], t.X[2])), maxX = max(t.X[0], max(t.X[1], t.X[2]));
    int minY = min(t.Y[0], min(t.Y[1], t.Y[2])), maxY = max(t.Y[0], max(t.Y[1], t.Y[2]));
    int px0 = (minX - 128 + 255) >> 8, px1 = (maxX - 128) >> 8;
    int py0 = (minY - 128 + 255) >> 8, py1 = (maxY - 128) >> 8;
    if (px0 < 0) px0 = 0;
    if (py0 < 0) py0 = 0;
    if (px1 > cfg.w - 1) px1 = cfg.w - 1;
    if (py1 > cfg.h - 1) py1 = cfg.h - 1;
    if (px0 > px1 || py0 > py1) return false;
    t.px0 = (int)px0; t.px1 = (int)px1; t.py0 = (int)py0; t.py1 = (int)py1;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        int a = (i + 1) % 3, b = (i + 2) % 3;
        int dy = t.Y[b] - t.Y[a], dx = t.X[b] - t.X[a];
        t.tl[i] = (dy < 0 || (dy == 0 && dx < 0)) ? 1 : 0;
    }
    const double dz1 = (double)z[1] - (double)z[0];
    const double dz2 = (double)z[2] - (double)z[0];
    const double inv_area = 1.0 / (double)area;
    const double a = ((double)(t.Y[2] - t.Y[0]) * dz1 + (double)(t.Y[0] - t.Y[1]) * dz2) * inv_area;
    const double b = ((double)(t.X[0] - t.X[2]) * dz1 + (double)(t.X[1] - t.X[0]) * dz2) * inv_area;
    t.z0 = z[0];
    t.A = (float)a;
    t.B = (float)b;
    t.zoff = 0.0f;
    if (cfg.off_factor != 0.0f || cfg.off_units != 0.0f) {
        double m = fmax(fabs(a), fabs(b)) * 256.0;
        float zmax = fmaxf(fmaxf(fabsf(z[0]), fabsf(z[1])), fabsf(z[2]));
        double r = 0.0;
        if (zmax > 0.0f) {
            int e;
            frexpf(zmax, &e);
            r = ldexp(1.0, (e - 1) - 23);
        }
        t.zoff = (float)((double)cfg.off_factor * m + (double)cfg.off_units * r);
    }
    return true;
}

// Sutherland-Hodgman over the six clip planes, from the triangle in
// poly[0..2]; `poly` and `tmp` hold kMaxPoly vertices each and swap roles
// after every plane.  Sets up fan piece `piece` of the result and returns the
// number of fan pieces; `ok` tells whether `piece` is non-empty.
template <int NA>
__device__ __forceinline__ int clip_fan(CV<NA>* poly, CV<NA>* tmp, int piece, const RasterCfg& cfg, Tri<NA>& t,
                                        bool& ok) {
    int n = 3;
    ok = false;
    for (int p = 0; p < 6; ++p) {
        int m = 0;
        for (int k = 0; k < n; ++k) {
            const CV<NA>& prev = poly[k == 0 ? n - 1 : k - 1];
            const CV<NA>& cur = poly[k];
            float dp = plane_dist(prev.c, p), dc = plane_dist(cur.c, p);
            if (dc >= 0.0f) {
                if (dp < 0.0f) lerp_cv<NA>(cur, prev, dc, dp, tmp[m++]);
                tmp[m++] = cur;
            } else if (dp >= 0.0f) {
                lerp_cv<NA>(prev, cur, dp, dc, tmp[m++]);
            }
        }
        n = m;
        if (n < 3) return 0;
        CV<NA>* x = poly;
        poly = tmp;
        tmp = x;
    }
    if (piece + 2 < n) ok = setup_piece<NA>(poly[0], poly[piece + 1], poly[piece + 2], cfg, t);
    return n - 2;
}

// clip_fan with the polygons in private memory.
template <int NA>
__device__ __noinline__ int clip_and_setup(const CV<NA> v[3], int piece, const RasterCfg& cfg,
                                           Tri<NA>& t, bool& ok) {
    CV<NA> poly[kMaxPoly], tmp[kMaxPoly];
    poly[0] = v[0];
    poly[1] = v[1];
    poly[2] = v[2];
    return clip_fan<NA>(poly, tmp, piece, cfg, t, ok);
}

// Number of fan pieces of `tri` (0 when trivially rejected) and the setup of
// piece `piece`; `ok` is false when that piece covers no pixel centre.
template <int NA>
__device__ int get_piece(const MeshView& m, const float mvp[16], int tri, int piece, const RasterCfg& cfg,
                         Tri<NA>& t, bool& ok) {
    CV<NA> v[3];
    load_tri<NA>(m, mvp, tri, v);
    bool inside_all = true;
    for (int p = 0; p < 6; ++p) {
        float d0 = plane_dist(v[0].c, p), d1 = plane_dist(v[1].c, p), d2 = plane_dist(v[2].c, p);
        int nin = (d0 >= 0.0f) + (d1 >= 0.0f) + (d2 >= 0.0f);
        if (nin == 0) { ok = false; return 0; }
        if (nin != 3) inside_all = false;
    }
    if (inside_all) {
        ok = (piece == 0) && setup_piece<NA>(v[0], v[1], v[2], cfg, t);
        return 1;
    }
    return clip_and_setup<NA>(v, piece, cfg, t, ok);
}

// Clip-free classification used by the hot kernels: kReject (outside a clip
// plane), kClip (crosses a plane: handled by k_clip through setup records) or
// kInside, in which case `t` is set up and `ok` tells whether it covers a
// pixel centre.
enum { kReject = 0, kClip = 1, kInside = 2 };

template <int NA>
__device__ __forceinline__ int classify(const MeshView& m, const float mvp[16], int tri, const RasterCfg& cfg,
                                        Tri<NA>& t, bool& ok) {
    CV<NA> v[3];
    load_tri<NA>(m, mvp, tri, v);
    bool inside_all = true;
    ok = false;
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        float d0 = plane_dist(v[0].c, p), d1 = plane_dist(v[1].c, p), d2 = plane_dist(v[2].c, p);
        int nin = (d0 >= 0.0f) + (d1 >= 0.0f) + (d2 >= 0.0f);
        if (nin == 0) return kReject;
        if (nin != 3) inside_all = false;
    }
    if (!inside_all) return kClip;
    ok = setup_piece<NA>(v[0], v[1], v[2], cfg, t);
    return kInside;
}

// Conservative test: can any pixel centre of [x0,x1]x[y0,y1] be inside?
template <int NA>
__device__ __forceinline__ bool rect_overlap(const Tri<NA>& t, int x0, int x1, int y0, int y1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int a = (k + 1) % 3, b = (k + 2) % 3;
        const int ex = t.X[b] - t.X[a], ey = t.Y[b] - t.Y[a];
        const int Px = ((ey < 0) ? x1 : x0) * 256 + 128;
        const int Py = ((ex > 0) ? y1 : y0) * 256 + 128;
        const long long e = (long long)ex * (Py - t.Y[a]) - (long long)ey * (Px - t.X[a]);
        if (e + t.tl[k] <= 0) return false;
    }
    return true;
}

__device__ __forceinline__ uint32_t fbits(float f) { return __float_as_uint(f); }

// ---------------------------------------------------------------------------
// Compact setup record of one screen-space piece.  Wide pieces get one record
// per map in HBM (written once by the binning pass); pieces a whole workgroup
// rasterizes are shared through LDS.
// ---------------------------------------------------------------------------
// An edge of 2^23 units (32,768 pixels) or more in x or y, past the 24-bit
// factors of tile_edges: such a record takes the 64-bit edge functions.  The
// vertices themselves decide: the guard band keeps an unclipped triangle's
// edges below four views, but a clipped vertex's x and w are rounded one by one
// and can lie outside it by any factor (a ground of 10^8 units seen from 1:
// 1.7%, so past the limit from views of 8,060 pixels on).
constexpr int kLongEdge = 8;
__device__ __forceinline__ int long_edge(const int X[3], const int Y[3]) {
    const int dx = max(max(abs(X[1] - X[0]), abs(X[2] - X[1])), abs(X[0] - X[2]));
    const int dy = max(max(abs(Y[1] - Y[0]), abs(Y[2] - Y[1])), abs(Y[0] - Y[2]));
    return max(dx, dy) < (1 << 23) ? 0 : kLongEdge;
}

struct Setup {
    int X[3], Y[3];            // 24.8 fixed-point window coordinates
    int px0, px1, py0, py1;    // pixel-centre bounding box (clamped)
    int tl;                    // bit k: top-left tie bit of the edge opposite vertex k; kLongEdge
    uint32_t id;               // tri * 8 + fan piece
    float z0, A, B, zoff;      // depth plane about vertex 0
};

template <int NA>
__device__ __forceinline__ Setup to_setup(const Tri<NA>& t, uint32_t id) {
    Setup s;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        s.X[i] = t.X[i];
        s.Y[i] = t.Y[i];
    }
    s.px0 = t.px0; s.px1 = t.px1; s.py0 = t.py0; s.py1 = t.py1;
    s.tl = t.tl[0] | (t.tl[1] << 1) | (t.tl[2] << 2) | long_edge(t.X, t.Y);
    s.id = id;
    s.z0 = t.z0; s.A = t.A; s.B = t.B; s.zoff = t.zoff;
    return s;
}

// The count pass's record of a directly binned triangle, 32 bytes: the list
// entry supplies the id, the tie bits and the pixel box follow from the
// vertices, and vertices 1 and 2 are kept as 16-bit offsets from vertex 0.  A
// triangle with a vertex 128 pixels or more from vertex 0 (a thin one, or one
// that leaves the view) keeps them in a FarRec beside the record.  The
// records are the raster's and the count pass's largest traffic after the
// maps themselves; with 48 bytes (32-bit coordinates, packed box) 289 maps of
// a 50,002-triangle mesh took 206 us in the count pass and 450 us in the
// raster, with 32 bytes 187 and 401 us (64 maps of 2048^2 and 100,822
// triangles, whose count pass is bound by its arithmetic: raster 326 and 306).
struct alignas(16) SetupRec {
    int X0, Y0;
    uint32_t d1, d2;  // (X - X0) | (Y - Y0) << 16 of vertices 1 and 2
    float z0, A, B, zoff;
};
static_assert(sizeof(SetupRec) == 32, "two 16-byte loads");
struct alignas(16) FarRec {
    int X1, Y1, X2, Y2;
};
constexpr uint32_t kFar = 0x80008000u;  // SetupRec::d1 of a record with a FarRec: no 16-bit offsets are these

// Every vertex within 127 pixels of vertex 0.
__device__ __forceinline__ bool rec_fits(const Tri<0>& t) {
    const int dx1 = t.X[1] - t.X[0], dx2 = t.X[2] - t.X[0], dy1 = t.Y[1] - t.Y[0], dy2 = t.Y[2] - t.Y[0];
    return max(max(abs(dx1), abs(dx2)), max(abs(dy1), abs(dy2))) < 32768;
}

__device__ __forceinline__ void store_rec(SetupRec* recs, FarRec* fars, size_t at, const Tri<0>& t) {
    SetupRec r;
    r.X0 = t.X[0];
    r.Y0 = t.Y[0];
    r.d1 = ((uint32_t)(t.X[1] - t.X[0]) & 0xFFFFu) | ((uint32_t)(t.Y[1] - t.Y[0]) << 16);
    r.d2 = ((uint32_t)(t.X[2] - t.X[0]) & 0xFFFFu) | ((uint32_t)(t.Y[2] - t.Y[0]) << 16);
    r.z0 = t.z0; r.A = t.A; r.B = t.B; r.zoff = t.zoff;
    if (!rec_fits(t)) {
        r.d1 = kFar;
        fars[at] = FarRec{t.X[1], t.Y[1], t.X[2], t.Y[2]};
    }
    recs[at] = r;
}

// A record's vertices, from its first 16 bytes.
__device__ __forceinline__ void rec_vertices(int X0, int Y0, uint32_t d1, uint32_t d2, const FarRec& far, int X[3],
                                             int Y[3]) {
    X[0] = X0;
    Y[0] = Y0;
    X[1] = X0 + (int)(int16_t)(d1 & 0xFFFFu);
    Y[1] = Y0 + ((int)d1 >> 16);
    X[2] = X0 + (int)(int16_t)(d2 & 0xFFFFu);
    Y[2] = Y0 + ((int)d2 >> 16);
    if (d1 == kFar) {
        const FarRec f = far;
        X[1] = f.X1;
        Y[1] = f.Y1;
        X[2] = f.X2;
        Y[2] = f.Y2;
    }
}

// Pixel-centre box of a record's vertices, not yet clamped to the view.
__device__ __forceinline__ void rec_box(const int X[3], const int Y[3], int& px0, int& px1, int& py0, int& py1) {
    px0 = (min(X[0], min(X[1], X[2])) + 127) >> 8;
    px1 = (max(X[0], max(X[1], X[2])) - 128) >> 8;
    py0 = (min(Y[0], min(Y[1], Y[2])) + 127) >> 8;
    py1 = (max(Y[0], max(Y[1], Y[2])) - 128) >> 8;
}

// Same box and tie rules as setup_piece, on the same 24.8 coordinates.  Never a
// long edge: the triangle was not clipped, so it reaches at most 1.5 views past
// the view (24,576 pixels), and at most four tiles into it.
__device__ __forceinline__ Setup from_rec(const SetupRec& r, const FarRec& far, uint32_t id, const RasterCfg& cfg) {
    Setup s;
    rec_vertices(r.X0, r.Y0, r.d1, r.d2, far, s.X, s.Y);
    rec_box(s.X, s.Y, s.px0, s.px1, s.py0, s.py1);
    s.px0 = max(s.px0, 0);
    s.px1 = min(s.px1, cfg.w - 1);
    s.py0 = max(s.py0, 0);
    s.py1 = min(s.py1, cfg.h - 1);
    s.tl = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        int a = (i + 1) % 3, b = (i + 2) % 3;
        const int dy = s.Y[b] - s.Y[a], dx = s.X[b] - s.X[a];
        s.tl |= (dy < 0 || (dy == 0 && dx < 0)) ? (1 << i) : 0;
    }
    s.id = id;
    s.z0 = r.z0; s.A = r.A; s.B = r.B; s.zoff = r.zoff;
    return s;
}

// Edge tests and depth at the centre of pixel (i, j); false when not covered.
__device__ __forceinline__ bool eval_setup(const Setup& s, int i, int j, float& zout) {
    const int Px = i * 256 + 128, Py = j * 256 + 128;
    long long e0 = (long long)(s.X[2] - s.X[1]) * (Py - s.Y[1]) - (long long)(s.Y[2] - s.Y[1]) * (Px - s.X[1]);
    long long e1 = (long long)(s.X[0] - s.X[2]) * (Py - s.Y[2]) - (long long)(s.Y[0] - s.Y[2]) * (Px - s.X[2]);
    long long e2 = (long long)(s.X[1] - s.X[0]) * (Py - s.Y[0]) - (long long)(s.Y[1] - s.Y[0]) * (Px - s.X[0]);
    if (e0 + (s.tl & 1) <= 0 || e1 + ((s.tl >> 1) & 1) <= 0 || e2 + ((s.tl >> 2) & 1) <= 0) return false;
    float dx = (float)(Px - s.X[0]), dy = (float)(Py - s.Y[0]);
    float z = s.z0 + (s.A * dx + s.B * dy);
    z = z + s.zoff;
    if (!(z > 0.0f)) z = 0.0f;
    if (z > 1.0f) z = 1.0f;
    zout = z;
    return true;
}

__device__ __forceinline__ bool rect_overlap_s(const Setup& s, int x0, int x1, int y0, int y1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int a = (k + 1) % 3, b = (k + 2) % 3;
        const int ex = s.X[b] - s.X[a], ey = s.Y[b] - s.Y[a];
        const int Px = ((ey < 0) ? x1 : x0) * 256 + 128;
        const int Py = ((ex > 0) ? y1 : y0) * 256 + 128;
        const long long e = (long long)ex * (Py - s.Y[a]) - (long long)ey * (Px - s.X[a]);
        if (e + ((s.tl >> k) & 1) <= 0) return false;
    }
    return true;
}

// ---------------------------------------------------------------------------
// Binning
// ---------------------------------------------------------------------------
// Pieces overlapping more than wide_span<TS>() tiles are "wide" (binned from
// setup records by k_bin_wide): 4 tiles of 64x64 texels, the same texel area
// for other tile edges, so the set of wide pieces does not grow as tiles
// shrink.
template <int TS>
constexpr int wide_span() {
    return 4 * (64 / TS) * (64 / TS);
}
constexpr uint32_t kWideBit = 0x80000000u;
constexpr int kWideBlocks = 64;         // workgroups per map binning wide pieces
constexpr int kClipBlocks = 16;         // workgroups per map clipping listed triangles
constexpr int kClipThreads = 64;        // threads per clipping workgroup

constexpr int kMaxPieces = kMaxPoly - 2;  // fan pieces of a clipped triangle

// What the G-buffer resolve reads of a clipped triangle's fan piece: its
// window coordinates, clip w, attributes and facing, as setup_piece leaves
// them.
struct alignas(16) ResolveRec {
    int X[3], Y[3];
    float w[3];
    float a[3][6];
    int tl[3];
    int front;
    int pad;
};
static_assert(sizeof(ResolveRec) == 128, "one cache line");

struct BinBufs {
    uint32_t* counts;    // nmaps x ntiles (scatter cursors after k_scan)
    uint32_t* offsets;   // nmaps x (ntiles + 1)
    int* overflow;       // nmaps: lists or wide records exceed the workspace
    int* wide_over;      // nmaps
    uint32_t* nwide;     // nmaps
    Setup* wide;         // nmaps x wcap
    uint32_t* nclip;     // nmaps
    uint32_t* clip;      // nmaps x ccap: triangles crossing a clip plane
    uint32_t* entries;   // nmaps x cap
    uint32_t* tiles;     // nmaps x tstride: the count pass's tiles of each directly binned triangle
    SetupRec* setups;    // nmaps x tstride: its setup record (64-texel tiles only)
    FarRec* fars;        // nmaps x tstride: and its vertices 1 and 2, where the record cannot hold them
    ResolveRec* attrs;   // G-buffer pass only (one map): acap x kMaxPieces, the clipped pieces' attributes
    uint32_t cap, wcap, ccap, tstride, acap;
};

// The tiles a directly binned triangle overlaps, as the count pass found
// them, for the scatter pass: bits 0-15 the first tile of its tile box,
// bits 16-17 the box width in tiles minus 1, bits 18-21 which of the box's
// (at most 4) tiles it overlaps.  Bits 18-21 zero: none (rejected, clipped,
// wide or empty); bit 31 then marks a clipped triangle, whose place in the
// clip list fills the other bits (0-17, then 22-30).  The counter that gives
// the places runs past the list's capacity, up to the mesh's triangles; all
// places past the list are one, the capacity, which fits these 27 bits.
constexpr uint32_t kClipCode = 0x80000000u;
__device__ __forceinline__ uint32_t tiles_code(int base, int ntx, uint32_t mask) {
    return mask ? ((uint32_t)base | ((uint32_t)(ntx - 1) << 16) | (mask << 18)) : 0u;
}
__host__ __device__ constexpr uint32_t clip_code(uint32_t c, uint32_t ccap) {
    c = c < ccap ? c : ccap;
    return kClipCode | (c & 0x3FFFFu) | ((c >> 18) << 22);
}
__host__ __device__ constexpr uint32_t clip_place(uint32_t code) {
    return (code & 0x3FFFFu) | (((code & ~kClipCode) >> 22) << 18);
}

__device__ __forceinline__ void bin_tile(const BinBufs& b, int map, int ntiles, int tile, uint32_t entry,
                                         bool scatter) {
    uint32_t* cnt = b.counts + (size_t)map * ntiles;
    if (!scatter) {
        atomicAdd(&cnt[tile], 1u);
    } else {
        uint32_t pos = b.offsets[(size_t)map * (ntiles + 1) + tile] + atomicAdd(&cnt[tile], 1u);
        if (pos < b.cap) b.entries[(size_t)map * b.cap + pos] = entry;
    }
}

// A workgroup barrier that orders LDS only.  __syncthreads() also waits for
// the workgroup's outstanding global stores and atomics (its release fence
// covers global memory); the binning kernels' barriers guard their LDS
// histograms and prefix sums, and what they write to global memory is read
// only by later kernels (an atomic whose result goes to LDS has returned
// before that LDS write).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Appends a setup record (count pass only); records past the capacity flag
// the map for the fallback raster.
template <int NA>
__device__ __forceinline__ void push_record(const BinBufs& b, int map, const Tri<NA>& t, uint32_t entry) {
    uint32_t w = atomicAdd(&b.nwide[map], 1u);
    if (w < b.wcap) b.wide[(size_t)map * b.wcap + w] = to_setup(t, entry);
    else b.wide_over[map] = 1;
}

// One thread per (triangle, map).  Triangles inside every clip plane whose
// piece spans at most kWideSpan tiles are binned here; wider ones get a setup
// record (binned by k_bin_wide), and triangles crossing a clip plane are
// listed for k_clip.
//
// Tile counts are first aggregated in an LDS histogram, so the workgroup
// issues one device-scope atomic per touched tile instead of one per
// triangle: consecutive triangles of a mesh are neighbours and share tiles,
// and device-scope atomics on the same line serialize outside the XCD's L2.
constexpr int kBinHist = 4096;  // largest tile grid aggregated in LDS (64 x 64 tiles)

template <int TS, bool kScatter>
__device__ __forceinline__ void bin_body(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                         const BinBufs& b, int bx, int map) {
    __shared__ uint32_t hist[kBinHist];
    const int tid = threadIdx.x;
    const int tri = bx * kRasterThreads + tid;
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const bool lds = ntiles <= kBinHist;
    if (kScatter && b.overflow[map]) return;  // uniform per workgroup
    if (lds)
        for (int p = tid; p < ntiles; p += blockDim.x) hist[p] = 0;
    // Up to wide_span<TS>() tiles per thread, kept in registers (static indices).
    constexpr int kWideSpan = wide_span<TS>();
    // 64-texel tiles: the count pass stores each triangle's tiles and the
    // scatter pass reads them back; smaller tiles (a wider span than the code
    // holds) classify again in the scatter pass
    constexpr bool kCache = kWideSpan <= 4;
    int tile_of[kWideSpan];
    uint32_t rank_of[kWideSpan];
#pragma unroll
    for (int k = 0; k < kWideSpan; ++k) tile_of[k] = -1;
    const uint32_t entry = (uint32_t)tri * 8u;
    if (kScatter && kCache) {
        // the count pass classified this (triangle, map) already
        if (tri < mesh.nt) {
            const uint32_t code = b.tiles[(size_t)map * b.tstride + tri];
            const int base = (int)(code & 0xFFFFu), ntx = (int)((code >> 16) & 3u) + 1;
            const uint32_t mask = code >> 18;
#pragma unroll
            for (int k = 0; k < kWideSpan; ++k)
                if (mask & (1u << k)) tile_of[k] = base + (k / ntx) * cfg.tiles_x + (k % ntx);
        }
    } else if (tri < mesh.nt) {
        float mvp[16];
        mvps.load(map, mvp);
        uint32_t code = 0;
        Tri<0> t;
        bool ok;
        int cls = classify<0>(mesh, mvp, tri, cfg, t, ok);
        if (cls == kClip) {
            if (!kScatter) {
                uint32_t c = atomicAdd(&b.nclip[map], 1u);
                if (c < b.ccap) b.clip[(size_t)map * b.ccap + c] = (uint32_t)tri;
                else b.wide_over[map] = 1;
                code = clip_code(c, b.ccap);
            }
        } else if (ok) {
            int tx0 = t.px0 / TS, tx1 = t.px1 / TS, ty0 = t.py0 / TS, ty1 = t.py1 / TS;
            int ntx = tx1 - tx0 + 1;
            int span = ntx * (ty1 - ty0 + 1);
            if (span > kWideSpan) {
                if (!kScatter) push_record(b, map, t, entry);
            } else {
                uint32_t mask = 0;
#pragma unroll
                for (int k = 0; k < kWideSpan; ++k) {
                    if (k >= span) continue;
                    int tx = tx0 + k % ntx, ty = ty0 + k / ntx;
                    if (span > 1) {
                        int x0 = max(tx * TS, t.px0), x1 = min(tx * TS + TS - 1, t.px1);
                        int y0 = max(ty * TS, t.py0), y1 = min(ty * TS + TS - 1, t.py1);
                        if (!rect_overlap<0>(t, x0, x1, y0, y1)) continue;
                    }
                    tile_of[k] = ty * cfg.tiles_x + tx;
                    mask |= 1u << k;
                }
                code = tiles_code(ty0 * cfg.tiles_x + tx0, ntx, mask);
                if (!kScatter && kCache && mask) store_rec(b.setups, b.fars, (size_t)map * b.tstride + tri, t);
            }
        }
        if (!kScatter && kCache) b.tiles[(size_t)map * b.tstride + tri] = code;
    }
    if (!lds) {
#pragma unroll
        for (int k = 0; k < kWideSpan; ++k)
            if (tile_of[k] >= 0) bin_tile(b, map, ntiles, tile_of[k], entry, kScatter);
        return;
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < kWideSpan; ++k)
        if (tile_of[k] >= 0) rank_of[k] = atomicAdd(&hist[tile_of[k]], 1u);
    lds_barrier();
    uint32_t* cnt = b.counts + (size_t)map * ntiles;
    for (int p = tid; p < ntiles; p += blockDim.x) {
        uint32_t c = hist[p];
        if (c == 0) continue;
        if (!kScatter) atomicAdd(&cnt[p], c);
        else hist[p] = atomicAdd(&cnt[p], c);  // this workgroup's base within the tile's list
    }
    if (!kScatter) return;
    lds_barrier();
    const uint32_t* off = b.offsets + (size_t)map * (ntiles + 1);
#pragma unroll
    for (int k = 0; k < kWideSpan; ++k) {
        if (tile_of[k] < 0) continue;
        uint32_t pos = off[tile_of[k]] + hist[tile_of[k]] + rank_of[k];
        if (pos < b.cap) b.entries[(size_t)map * b.cap + pos] = entry;
    }
}

template <int TS, bool kScatter>
__global__ __launch_bounds__(256) void k_bin(MeshView mesh, MvpSource mvps, RasterCfg cfg, BinBufs b) {
    bin_body<TS, kScatter>(mesh, mvps, cfg, b, blockIdx.x, blockIdx.y);
}


// Clips the listed triangles; every non-empty fan piece becomes a setup
// record.  Runs between the count passes, before k_bin_wide.  A wave of 64
// clips four triangles, 16 lanes each: lane j of a group holds polygon vertex
// j, so a clip plane is one step (every vertex's distance and intersection
// at once, the survivors' places from ballots) where one thread per piece
// walked the vertices in turn, once for every piece; a plane that cuts none
// of the wave's polygons moves nothing.  The kernel is one dependent chain,
// so that chain's length is its time: for a view of a ground quad (two
// triangles to clip) 12.3 us before, 4.5 us now; for 289 maps of it 35 and
// 9 us.  The arithmetic of a vertex
// is clip_fan's.  The polygons live in LDS: as private arrays indexed at run
// time they would sit in scratch memory.  Workgroup `part` of `nparts` takes
// every nparts-th run of four triangles of the map.
constexpr int kClipGroup = 16;  // lanes (and polygon slots) per triangle
constexpr int kClipGroups = kClipThreads / kClipGroup;
static_assert(kClipThreads == 64 && kMaxPoly <= kClipGroup, "a workgroup is one wave, a polygon fits its lanes");

// LDS written by other lanes of this wave: orders the compiler's accesses.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// NA = 6 (the G-buffer pass): the attributes are clipped along, and each
// piece of the first acap listed triangles leaves them in b.attrs.
template <int NA>
__device__ __forceinline__ void clip_body(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                          const BinBufs& b, int part, int nparts, int map) {
    __shared__ CV<NA> pool[kClipGroups][2][kClipGroup];
    const uint32_t n = min(b.nclip[map], b.ccap);
    if ((uint32_t)part * kClipGroups >= n) return;  // uniform
    float mvp[16];
    mvps.load(map, mvp);
    const int grp = (int)threadIdx.x / kClipGroup, j = (int)threadIdx.x % kClipGroup;
    const unsigned below = (1u << j) - 1u;
    for (uint32_t base = (uint32_t)part * kClipGroups; base < n; base += (uint32_t)nparts * kClipGroups) {
        const uint32_t c = base + (uint32_t)grp;
        const int tri = c < n ? (int)b.clip[(size_t)map * b.ccap + c] : 0;
        int cnt = c < n ? 3 : 0;
        CV<NA>* poly = pool[grp][0];
        CV<NA>* tmp = pool[grp][1];
        wave_lds_fence();
        if (j < cnt) load_vertex<NA>(mesh, mvp, mesh.idx[3 * tri + j], poly[j]);
        wave_lds_fence();
        for (int p = 0; p < 6; ++p) {
            const bool act = j < cnt;
            CV<NA> cur, prev;
            bool cut = false, keep = false;
            float dc = 0.0f, dp = 0.0f;
            if (act) {
                cur = poly[j];
                prev = poly[j == 0 ? cnt - 1 : j - 1];
                dc = plane_dist(cur.c, p);
                dp = plane_dist(prev.c, p);
                keep = dc >= 0.0f;
                cut = keep ? dp < 0.0f : dp >= 0.0f;
            }
            if (!__any(act && (cut || !keep))) continue;  // uniform: the polygons stay as they are
            const unsigned mk = (unsigned)(__ballot(keep) >> (kClipGroup * grp)) & 0xFFFFu;
            const unsigned mc = (unsigned)(__ballot(cut) >> (kClipGroup * grp)) & 0xFFFFu;
            int at = __popc(mk & below) + __popc(mc & below);
            if (cut) {
                CV<NA> r;
                if (keep) lerp_cv<NA>(cur, prev, dc, dp, r);
                else lerp_cv<NA>(prev, cur, dp, dc, r);
                if (at < kClipGroup) tmp[at] = r;
                ++at;
            }
            if (keep && at < kClipGroup) tmp[at] = cur;
            cnt = min(__popc(mk) + __popc(mc), kClipGroup);
            if (cnt < 3) cnt = 0;
            CV<NA>* x = poly;
            poly = tmp;
            tmp = x;
            wave_lds_fence();
        }
        if (j + 2 < cnt && j < kMaxPieces) {
            Tri<NA> t;
            if (setup_piece<NA>(poly[0], poly[j + 1], poly[j + 2], cfg, t)) {
                push_record(b, map, t, (uint32_t)tri * 8u + (uint32_t)j);
                if constexpr (NA == 6) {
                    if (c < b.acap) {
                        ResolveRec r;
#pragma unroll
                        for (int i = 0; i < 3; ++i) {
                            r.X[i] = t.X[i];
                            r.Y[i] = t.Y[i];
                            r.w[i] = t.w[i];
                            r.tl[i] = t.tl[i];
#pragma unroll
                            for (int q = 0; q < 6; ++q) r.a[i][q] = t.a[i][q];
                        }
                        r.front = t.front;
                        r.pad = 0;
                        b.attrs[(size_t)c * kMaxPieces + j] = r;
                    }
                }
            }
        }
    }
}

template <int NA>
__global__ __launch_bounds__(kClipThreads) void k_clip(MeshView mesh, MvpSource mvps, RasterCfg cfg, BinBufs b) {
    clip_body<NA>(mesh, mvps, cfg, b, blockIdx.x, gridDim.x, blockIdx.y);
}

// Wide pieces (setup records), kWideThreads threads per workgroup, nparts
// workgroups a map.  A round holds kWideThreads records, one per thread; its
// (record, tile) pairs are numbered through a prefix sum of the records' tile
// spans, so that the pairs' appends (whose scatter atomics return the list
// slot) are all in flight at once whether the round holds many records of a
// few tiles or one record over the whole map.  A map of one round (a ground
// plane's clipped pieces) has its pairs dealt to `shares` parts, each of which
// numbers the same round: a piece over the 4,096 tiles of a 4096^2 map was one
// part's 16 appends per thread, one after another (count 11.5 us, scatter 17
// us; dealt out 4.5 and 8.4).  With more records, part p takes records p, p +
// nparts, ... and every kWideThreads-th pair of them.  Launches of many maps
// deal each map's to fewer parts, about 1,024 in all (wide_shares): 289 maps
// of 81 tiles took 24 and 87 us with 64 parts each, 18 and 78 without dealing.
constexpr int kWideThreads = 256;
__device__ __forceinline__ int wide_shares(int nmaps) { return max(8, min(kWideBlocks, 1024 / nmaps)); }

template <int TS, bool kScatter>
__device__ __forceinline__ void wide_tile(const RasterCfg& cfg, const BinBufs& b, int map, int ntiles, const Setup& s,
                                          uint32_t w, int tx0, int ty0, int ntx, int q) {
    const int tx = tx0 + q % ntx, ty = ty0 + q / ntx;
    const int x0 = max(tx * TS, s.px0), x1 = min(tx * TS + TS - 1, s.px1);
    const int y0 = max(ty * TS, s.py0), y1 = min(ty * TS + TS - 1, s.py1);
    if (rect_overlap_s(s, x0, x1, y0, y1)) bin_tile(b, map, ntiles, ty * cfg.tiles_x + tx, kWideBit | w, kScatter);
}

template <int TS, bool kScatter>
__device__ __forceinline__ void bin_wide_body(const RasterCfg& cfg, const BinBufs& b, int part, int nparts, int map,
                                              int shares) {
    __shared__ int incl[kWideThreads];  // inclusive prefix of the round's spans
    __shared__ int wave_sum[kWideThreads / 64];
    if (kScatter && b.overflow[map]) return;  // uniform per workgroup
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const uint32_t n = min(b.nwide[map], b.wcap);
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool share = n <= (uint32_t)kWideThreads;
    const uint32_t first = share ? 0u : (uint32_t)part, stride = share ? 1u : (uint32_t)nparts;
    const int pair0 = share ? part * kWideThreads + tid : tid, pairs = share ? shares * kWideThreads : kWideThreads;
    if (share && part >= shares) return;  // uniform
    const Setup* recs = b.wide + (size_t)map * b.wcap;
    for (uint32_t r0 = 0; first + stride * r0 < n; r0 += kWideThreads) {  // uniform
        const uint32_t w = first + stride * (r0 + (uint32_t)tid);
        int span = 0;
        if (w < n) {
            const Setup& s = recs[w];
            span = (s.px1 / TS - s.px0 / TS + 1) * (s.py1 / TS - s.py0 / TS + 1);
        }
        int v = span;  // inclusive scan in the wave, then across the waves
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(v, d, 64);
            if (lane >= d) v += u;
        }
        if (lane == 63) wave_sum[wave] = v;
        lds_barrier();
        int base = 0, total = 0;
#pragma unroll
        for (int k = 0; k < kWideThreads / 64; ++k) {
            base += k < wave ? wave_sum[k] : 0;
            total += wave_sum[k];
        }
        incl[tid] = base + v;
        lds_barrier();
        for (int p = pair0; p < total; p += pairs) {
            // the round's record holding pair p: the first k with incl[k] > p
            int lo = 0, hi = kWideThreads - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (incl[mid] > p) hi = mid;
                else lo = mid + 1;
            }
            const uint32_t wk = first + stride * (r0 + (uint32_t)lo);
            const Setup s = recs[wk];
            const int tx0 = s.px0 / TS, ty0 = s.py0 / TS;
            const int ntx = s.px1 / TS - tx0 + 1;
            const int q = p - (lo == 0 ? 0 : incl[lo - 1]);
            wide_tile<TS, kScatter>(cfg, b, map, ntiles, s, wk, tx0, ty0, ntx, q);
        }
        lds_barrier();  // incl and wave_sum are rewritten by the next round
    }
}

template <int TS, bool kScatter>
__global__ __launch_bounds__(256) void k_bin_wide(RasterCfg cfg, BinBufs b) {
    bin_wide_body<TS, kScatter>(cfg, b, blockIdx.x, gridDim.x, blockIdx.y, wide_shares((int)gridDim.y));
}

// The scatter pass when the count pass stored each triangle's tile code
// (64-texel tiles): kT triangles per thread.  A workgroup's appends cost two
// dependent global round trips (the atomics that reserve its slice of each
// tile's list, then the list offsets), so covering kT x 256 triangles per
// workgroup divides those rounds by kT.  Entries land in the same lists as
// bin_body's scatter (their order within a list does not matter: the raster
// takes the minimum).  `block` covers triangles [block kT 256, (block + 1) kT 256)
// of map `map`.
template <int TS, int kT>
__device__ __forceinline__ void bin_scatter_body(const MeshView& mesh, const RasterCfg& cfg, const BinBufs& b,
                                                 int block, int map) {
    constexpr int kWideSpan = wide_span<TS>();
    static_assert(kWideSpan <= 4, "tile codes are stored for 64-texel tiles");
    __shared__ uint32_t hist[kBinHist];
    const int tid = (int)threadIdx.x;
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    if (b.overflow[map]) return;  // uniform per workgroup
    const bool lds = ntiles <= kBinHist;
    if (lds)
        for (int p = tid; p < ntiles; p += 256) hist[p] = 0;
    int tile_of[kT][kWideSpan];
    uint32_t rank_of[kT][kWideSpan];
#pragma unroll
    for (int t = 0; t < kT; ++t) {
        const int tri = (block * kT + t) * 256 + tid;
#pragma unroll
        for (int k = 0; k < kWideSpan; ++k) tile_of[t][k] = -1;
        if (tri < mesh.nt) {
            const uint32_t code = b.tiles[(size_t)map * b.tstride + tri];
            const int base = (int)(code & 0xFFFFu), ntx = (int)((code >> 16) & 3u) + 1;
            const uint32_t mask = code >> 18;
#pragma unroll
            for (int k = 0; k < kWideSpan; ++k)
                if (mask & (1u << k)) tile_of[t][k] = base + (k / ntx) * cfg.tiles_x + (k % ntx);
        }
    }
    if (!lds) {
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int k = 0; k < kWideSpan; ++k)
                if (tile_of[t][k] >= 0)
                    bin_tile(b, map, ntiles, tile_of[t][k], (uint32_t)((block * kT + t) * 256 + tid) * 8u,
                             true);
        return;
    }
    lds_barrier();
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int k = 0; k < kWideSpan; ++k)
            if (tile_of[t][k] >= 0) rank_of[t][k] = atomicAdd(&hist[tile_of[t][k]], 1u);
    lds_barrier();
    uint32_t* cnt = b.counts + (size_t)map * ntiles;
    for (int p = tid; p < ntiles; p += 256) {
        const uint32_t c = hist[p];
        if (c != 0) hist[p] = atomicAdd(&cnt[p], c);  // this workgroup's base within the tile's list
    }
    lds_barrier();
    const uint32_t* off = b.offsets + (size_t)map * (ntiles + 1);
#pragma unroll
    for (int t = 0; t < kT; ++t) {
        const uint32_t entry = (uint32_t)((block * kT + t) * 256 + tid) * 8u;
#pragma unroll
        for (int k = 0; k < kWideSpan; ++k) {
            if (tile_of[t][k] < 0) continue;
            const uint32_t pos = off[tile_of[t][k]] + hist[tile_of[t][k]] + rank_of[t][k];
            if (pos < b.cap) b.entries[(size_t)map * b.cap + pos] = entry;
        }
    }
}
// The single-instance scatter: workgroups past `tri_blocks` bin the wide
// pieces' records instead (bin_wide_body's scatter, kWideBlocks of them per
// map), so the two appends share one launch and overlap.
template <int TS, int kT>
__global__ __launch_bounds__(256) void k_bin_scatter(MeshView mesh, RasterCfg cfg, BinBufs b, int tri_blocks) {
    if ((int)blockIdx.x >= tri_blocks) {  // uniform per workgroup
        bin_wide_body<TS, true>(cfg, b, (int)blockIdx.x - tri_blocks, kWideBlocks, (int)blockIdx.y,
                                wide_shares((int)gridDim.y));
        return;
    }
    bin_scatter_body<TS, kT>(mesh, cfg, b, (int)blockIdx.x, (int)blockIdx.y);
}

constexpr int kScatterTris = 4;  // triangles per thread in k_bin_scatter

// Tiles of a map whose lists count as long, kept where the clip list was (dead
// once k_clip has run): word 0 their number, word 1 the length from which a
// list is one, then the tiles.
__device__ __forceinline__ uint32_t* split_tiles(const BinBufs& b, int map) {
    return b.clip + (size_t)map * b.ccap;
}

// Entries from which a tile's list is split, for a launch of `nmaps` maps like
// one with `total` entries: one of `shares` even shares of the launch
// (split_shares), and no less than kSplitMin, below which the 16 passes over the
// list cost more than they spread.
constexpr uint32_t kSplitMin = 48;
__device__ __forceinline__ uint32_t split_bound(unsigned long long total, int nmaps, uint32_t shares) {
    const unsigned long long even = total * (unsigned)nmaps / shares;
    return even > kSplitMin ? (uint32_t)min(even, 0x7FFFFFFFull) : kSplitMin;
}

// Exclusive scan of one map's tile counts; resets counts to 0 (they become
// the scatter cursors), flags maps whose lists exceed the workspace and, for
// launches that split long lists (split_maps > 0), lists those.  A chain of loads
// and sums in one workgroup: 2.9 us for 256 tiles with the sums by lane
// exchanges and 16 wave totals, 3.6 with ten rounds of LDS between barriers.
__device__ __forceinline__ void scan_body(const BinBufs& b, int ntiles, int map, int split_maps, uint32_t shares) {
    __shared__ unsigned long long wave_sum[kScanThreads / 64];
    __shared__ uint32_t nsplit;
    uint32_t* c = b.counts + (size_t)map * ntiles;
    uint32_t* o = b.offsets + (size_t)map * (ntiles + 1);
    int per = (ntiles + kScanThreads - 1) / kScanThreads;
    int lo = threadIdx.x * per, hi = min(lo + per, ntiles);
    unsigned long long s = 0;
    for (int i = lo; i < hi; ++i) s += c[i];
    // inclusive sums in the wave, then across the 16 waves
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    unsigned long long v = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
    }
    if (lane == 63) wave_sum[wave] = v;
    if (threadIdx.x == 0) nsplit = 0;
    __syncthreads();
    unsigned long long run = v - s, total = 0;  // exclusive prefix
#pragma unroll
    for (int k = 0; k < kScanThreads / 64; ++k) {
        run += k < wave ? wave_sum[k] : 0ull;
        total += wave_sum[k];
    }
    const uint32_t bound = split_maps > 0 ? split_bound(total, split_maps, shares) : 0u;
    uint32_t* split = split_tiles(b, map);
    for (int i = lo; i < hi; ++i) {
        o[i] = (uint32_t)run;
        const uint32_t n = c[i];
        run += n;
        c[i] = 0;
        if (split_maps > 0 && n > bound) {
            const uint32_t at = atomicAdd(&nsplit, 1u);
            if (at + 2 < b.ccap) split[at + 2] = (uint32_t)i;
        }
    }
    if (split_maps > 0) {
        __syncthreads();
        if (threadIdx.x == 0) {
            const bool fits = nsplit + 2 <= b.ccap;  // else no list of this map is split
            split[0] = fits ? nsplit : 0u;
            split[1] = fits ? bound : ~0u;
        }
    }
    if (threadIdx.x == kScanThreads - 1) {
        bool over = total > b.cap || b.wide_over[map] != 0;
        o[ntiles] = (uint32_t)(total > b.cap ? b.cap : total);
        b.overflow[map] = over ? 1 : 0;
    }
}

__global__ __launch_bounds__(kScanThreads) void k_scan(BinBufs b, int ntiles, int split_maps, uint32_t shares) {
    scan_body(b, ntiles, blockIdx.x, split_maps, shares);
}

// ---------------------------------------------------------------------------
// Tile raster
// ---------------------------------------------------------------------------
template <bool kVis>
struct KeyOf;
template <>
struct KeyOf<false> {
    using T = uint32_t;
    static constexpr uint32_t clear = 0x3F800000u;  // 1.0f
};
template <>
struct KeyOf<true> {
    using T = unsigned long long;
    static constexpr unsigned long long clear = ~0ull;
};

// Depth of a covered pixel centre at fixed-point offset (dx, dy) from vertex 0.
__device__ __forceinline__ uint32_t window_bits(float z, float zoff) {
    z = z + zoff;
    if (!(z > 0.0f)) z = 0.0f;  // NaN and -0 become +0
    // z is +0 or positive here (never NaN), where min(z, 1) is `z > 1 ? 1 : z`
    return fbits(__builtin_fminf(z, 1.0f));
}
__device__ __forceinline__ uint32_t plane_bits(const Setup& s, int dx, int dy) {
    return window_bits(s.z0 + (s.A * (float)dx + s.B * (float)dy), s.zoff);
}

template <bool kVis>
__device__ __forceinline__ void store_min(uint32_t id, uint32_t zb, int slot, typename KeyOf<kVis>::T* tile) {
    if constexpr (kVis) {
        atomicMin(&tile[slot], ((unsigned long long)zb << 32) | id);
    } else {
        atomicMin(&tile[slot], zb);
    }
}

// LDS row pitch of a tile: 8 words more than the tile's edge, so that the 64
// pixels of an aligned 8x8 block lie in 64 different banks.
template <int TS>
constexpr int tile_pitch() {
    return TS + 8;
}

// True when every pixel centre of [rx0, rx1] x [ry0, ry1] passes the three
// edge tests.  Each edge value is affine in the pixel indices, so its
// minimum over the rectangle is at a corner, and the test `e + tl > 0` holds
// everywhere once it holds at the four corners.
__device__ __forceinline__ bool rect_inside(const Setup& s, int rx0, int rx1, int ry0, int ry1) {
    const int cx[2] = {rx0 * 256 + 128, rx1 * 256 + 128};
    const int cy[2] = {ry0 * 256 + 128, ry1 * 256 + 128};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = (k + 1) % 3, b = (k + 2) % 3;
        const int ex = s.X[b] - s.X[a], ey = s.Y[b] - s.Y[a];
        const long long tl = (s.tl >> k) & 1;
        // the corner minimising ex * Py - ey * Px
        const int px = ey > 0 ? cx[1] : cx[0];
        const int py = ex > 0 ? cy[0] : cy[1];
        if ((long long)ex * (py - s.Y[a]) - (long long)ey * (px - s.X[a]) + tl <= 0) return false;
    }
    return true;
}

// The edge tests of one record over one tile in 32 bits.  Edge k's value at
// pixel (i, j) of the tile is E + 256 (j ex - i ey) with E its value at the
// tile's first pixel centre, so
//   E + 256 (..) + tl > 0   <=>   ((E + tl - 1) >> 8) + j ex - i ey >= 0
// exactly (`>>` rounds down).  Within a tile of at most 64 pixels the second
// part stays below 2^30 in magnitude when |ex| and |ey| are below 2^23, and a
// first part of 2^30 or more then decides the test in the whole tile, so it is
// clamped there and every sum fits in int32; the factors fit the 24-bit
// multipliers.  Not for records with kLongEdge, which go to raster_long.
struct TileEdges {
    int e[3];
    int ex[3], ey[3];
};
__device__ __forceinline__ TileEdges tile_edges(const Setup& s, int x0, int y0) {
    TileEdges t;
    const int Px = x0 * 256 + 128, Py = y0 * 256 + 128;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = (k + 1) % 3, b = (k + 2) % 3;
        const int ex = s.X[b] - s.X[a], ey = s.Y[b] - s.Y[a];
        const long long E = (long long)ex * (Py - s.Y[a]) - (long long)ey * (Px - s.X[a]) + ((s.tl >> k) & 1) - 1;
        const long long r = E >> 8;
        t.e[k] = (int)(r > (1ll << 30) ? (1ll << 30) - 1 : r < -(1ll << 30) ? -(1ll << 30) : r);
        t.ex[k] = ex;
        t.ey[k] = ey;
    }
    return t;
}

// Pixels n0, n0 + n, ... of the rectangle with the 64-bit edge functions.
template <int TS, bool kVis>
__device__ __forceinline__ void raster_rect_slow(const Setup& s, int x0, int y0, int rx0, int rx1, int ry0, int ry1,
                                                 int n0, int n, typename KeyOf<kVis>::T* tile) {
    const int rw = rx1 - rx0 + 1, area = rw * (ry1 - ry0 + 1);
    for (int q = n0; q < area; q += n) {
        const int i = rx0 + q % rw, j = ry0 + q / rw;
        float z;
        if (eval_setup(s, i, j, z)) store_min<kVis>(s.id, fbits(z), (j - y0) * tile_pitch<TS>() + (i - x0), tile);
    }
}

// One thread covers the whole (small) rectangle, row by row.
template <int TS, bool kVis>
__device__ __forceinline__ void raster_rect_self(const Setup& s, const TileEdges& t, int x0, int y0, int rx0, int rx1,
                                                 int ry0, int ry1, typename KeyOf<kVis>::T* tile) {
    int row[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) row[k] = t.e[k] + __mul24(ry0 - y0, t.ex[k]) - __mul24(rx0 - x0, t.ey[k]);
    const int width = rx1 - rx0;
    const float dx0 = (float)(rx0 * 256 + 128 - s.X[0]);
    int slot0 = (ry0 - y0) * tile_pitch<TS>() + (rx0 - x0);
    for (int j = ry0; j <= ry1; ++j) {
        int e0 = row[0], e1 = row[1], e2 = row[2];
        const float bdy = s.B * (float)(j * 256 + 128 - s.Y[0]);
        float dx = dx0;  // pixel-centre offsets are at most 2^24: exact in FP32, steps too
        const int end = slot0 + width;
        for (int slot = slot0; slot <= end; ++slot) {
            if ((e0 | e1 | e2) >= 0)
                store_min<kVis>(s.id, window_bits(s.z0 + (s.A * dx + bdy), s.zoff), slot, tile);
            e0 -= t.ey[0];
            e1 -= t.ey[1];
            e2 -= t.ey[2];
            dx += 256.0f;
        }
        slot0 += tile_pitch<TS>();
#pragma unroll
        for (int k = 0; k < 3; ++k) row[k] += t.ex[k];
    }
}

// 8x8-pixel blocks of the tile that a rectangle (tile-local pixels) touches,
// bit (TS / 8) * by + bx of block (bx, by).
template <int TS>
__device__ __forceinline__ unsigned long long block_mask(int rx0, int rx1, int ry0, int ry1) {
    constexpr int NB = TS / 8;
    const int bx0 = rx0 >> 3, bx1 = rx1 >> 3, by0 = ry0 >> 3, by1 = ry1 >> 3;
    const unsigned row = (2u << bx1) - (1u << bx0);
    unsigned long long m;
    if constexpr (NB == 8) {
        const unsigned r4 = row * 0x01010101u;
        m = ((unsigned long long)r4 << 32) | r4;
    } else {
        m = row * (NB == 4 ? 0x1111u : 0x5u);
    }
    return m & (~0ull << (NB * by0)) & (~0ull >> (63 - (NB * by1 + NB - 1)));
}

// Keeps a value in a vector register (the compiler otherwise forms sums of
// wave-uniform values with scalar multiplications).
__device__ __forceinline__ int in_vector(int v) {
    asm("" : "+v"(v));
    return v;
}

// The same for a scalar register.
__device__ __forceinline__ int in_scalar(int v) {
    asm("" : "+s"(v));
    return v;
}
// a * b + c of factors of 24 bits (tile_edges), b wave-uniform.
__device__ __forceinline__ int mad24(int a, int b, int c) {
    int r;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// Lane b: the largest depth (as bits) that block b of the tile holds now.
// Depths only fall, so a value that other waves have lowered since is still an
// upper bound.  The lanes start at different rows and halves of their blocks,
// which spreads each read over the banks.
template <int TS, bool kVis>
__device__ __forceinline__ uint32_t block_zmax(int lane, const typename KeyOf<kVis>::T* tile) {
    constexpr int NB = TS / 8;
    const int bx = lane % NB, by = lane / NB;
    uint32_t z = 0u;
    if (lane < NB * NB) {
#pragma unroll 2
        for (int r = 0; r < 8; ++r) {
            const int row = (by * 8 + ((r + by) & 7)) * tile_pitch<TS>() + bx * 8;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int at = row + ((h + by) & 1) * 4;
                if constexpr (kVis) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) z = max(z, (uint32_t)(tile[at + q] >> 32));
                } else {
                    const uint4 v = *reinterpret_cast<const uint4*>(&tile[at]);
                    z = max(max(z, max(v.x, v.y)), max(v.z, v.w));
                }
            }
        }
    }
    return z;
}

// The wave covers one record (all arguments but `lane` and `zmax` are
// wave-uniform): lane b first tests block b of the tile against the three
// edges (the block's pixel nearest to each edge's inside) and against the
// depth the block already has (zmax, block_zmax's), then the blocks left are
// taken row by row, a lane per pixel, 13 vector instructions each.  The
// record's smallest depth in a block is that of the corner pixel its plane
// falls to: every rounded step of the depth expression is monotonic in dx and
// in dy, so no pixel of the block comes out below it.
// kWhole: blocks that lie inside all three edges (most of a ground plane's)
// are taken in a loop of their own, with no edge tests and no lane masking (8
// vector and 6 scalar instructions each).
template <int TS, bool kVis, bool kWhole>
__device__ __forceinline__ void raster_blocks(const int er[3], const int ex[3], const int ey[3], float z0, float A,
                                              float B, float zoff, int dx0, int dy0, uint32_t id,
                                              unsigned long long blocks, int lane, uint32_t zmax,
                                              typename KeyOf<kVis>::T* tile) {
    constexpr int NB = TS / 8;
    const int blx = (lane % NB) * 8, bly = (lane / NB) * 8;
    const int lx = lane & 7, ly = lane >> 3;
    int near[3], off[3], step[3], inner[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        step[k] = in_vector(-ey[k]);
        const int ny = -ey[k];
        const int far = er[k] + max(0, 7 * ex[k]) + max(0, -7 * ey[k]);
        near[k] = mad24(blx, ny, mad24(bly, ex[k], in_vector(far)));
        if constexpr (kWhole) inner[k] = near[k] - in_scalar(7 * (abs(ex[k]) + abs(ey[k])));
        off[k] = mad24(lx, ny, mad24(ly, ex[k], in_vector(er[k])));
    }
    const uint32_t zmin =
        window_bits(z0 + (A * (float)(dx0 + (blx + (A < 0.0f ? 7 : 0)) * 256) +
                          B * (float)(dy0 + (bly + (B < 0.0f ? 7 : 0)) * 256)), zoff);
    const bool open = kVis ? zmin <= zmax : zmin < zmax;
    unsigned long long live = __ballot((near[0] | near[1] | near[2]) >= 0 && open) & blocks;
    unsigned long long whole = 0ull;
    if constexpr (kWhole) whole = __ballot((inner[0] | inner[1] | inner[2]) >= 0);
    const int dxl = in_vector(dx0 + lx * 256), dyl = in_vector(dy0 + ly * 256);
    const int slot = ly * tile_pitch<TS>() + lx;
    constexpr unsigned kRow = (1u << NB) - 1u;
    while (live) {
        const int row = (__ffsll((long long)live) - 1) / NB;
        unsigned cols = (unsigned)(live >> (row * NB)) & kRow;
        live &= ~((unsigned long long)kRow << (row * NB));
        const float bdy = B * (float)(dyl + row * 2048);
        const int srow = in_vector(slot + row * 8 * tile_pitch<TS>());
        if constexpr (kWhole) {
            unsigned inside = cols & (unsigned)(whole >> (row * NB));
            cols &= ~inside;
            while (inside) {
                const int bx = __ffs((int)inside) - 1;
                inside &= inside - 1;
                store_min<kVis>(id, window_bits(z0 + (A * (float)(dxl + (bx << 11)) + bdy), zoff), srow + 8 * bx, tile);
            }
            if (!cols) continue;
        }
        const int e0 = in_vector(off[0] + 8 * row * ex[0]), e1 = in_vector(off[1] + 8 * row * ex[1]),
                  e2 = in_vector(off[2] + 8 * row * ex[2]);
        while (cols) {
            const int bx = __ffs((int)cols) - 1, i = 8 * bx;
            cols &= cols - 1;
            if ((mad24(step[0], i, e0) | mad24(step[1], i, e1) | mad24(step[2], i, e2)) >= 0)
                store_min<kVis>(id, window_bits(z0 + (A * (float)(dxl + (bx << 11)) + bdy), zoff), srow + i, tile);
        }
    }
}

__device__ __forceinline__ int lane_int(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_float(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// raster_blocks for the records of the lanes with `want`, one after another;
// the wave looks at the tile's depths again after every kZmaxAge of them.
constexpr int kZmaxAge = 8;
template <int TS, bool kVis, bool kWhole>
__device__ __forceinline__ void raster_lanes(const Setup& s, const TileEdges& t, unsigned long long blocks, bool want,
                                             int x0, int y0, int lane, uint32_t& zmax, int& age,
                                             typename KeyOf<kVis>::T* tile) {
    const int dx0 = x0 * 256 + 128 - s.X[0], dy0 = y0 * 256 + 128 - s.Y[0];
    unsigned long long todo = __ballot(want);
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        if (++age == kZmaxAge) {
            age = 0;
            zmax = block_zmax<TS, kVis>(lane, tile);
        }
        const int er[3] = {lane_int(t.e[0], l), lane_int(t.e[1], l), lane_int(t.e[2], l)};
        const int a0 = lane_int(t.ex[0], l), a1 = lane_int(t.ex[1], l);
        const int b0 = lane_int(t.ey[0], l), b1 = lane_int(t.ey[1], l);
        const int ex[3] = {a0, a1, -(a0 + a1)}, ey[3] = {b0, b1, -(b0 + b1)};  // the edges close
        const unsigned long long m = ((unsigned long long)(unsigned)lane_int((int)(blocks >> 32), l) << 32) |
                                     (unsigned)lane_int((int)(unsigned)blocks, l);
        raster_blocks<TS, kVis, kWhole>(er, ex, ey, lane_float(s.z0, l), lane_float(s.A, l), lane_float(s.B, l),
                                lane_float(s.zoff, l), lane_int(dx0, l), lane_int(dy0, l),
                                kVis ? (uint32_t)lane_int((int)s.id, l) : 0u, m, lane, zmax, tile);
    }
}

// Why both: on a 200k-triangle soup in one 2048^2 map the raster took 213 us
// with records over 256 pixels covered by the whole workgroup, one after
// another between barriers (each wave repeating the record's setup for a
// quarter of its pixels), and 130 us with a wave per record; a batch of twelve
// frames (soups on 512^2-4096^2 maps) 4.82 and 2.94 ms.  In that batch a
// short list is one wave's, so its records of more than kShareBlocks blocks
// are put aside for all four: 2.12 ms with a bound of 16, 2.01 of 8, 1.96 of
// 4, 1.97 of 2 (a workgroup per tile; 2.74 ms with 8 from a queue of tiles).
//
// Records a lane rasterizes alone: those with at most self_bound() pixels of
// bounding box in the tile.  The wave then runs as long as the largest such
// box (about 14 vector instructions a pixel), while a larger record takes the
// whole wave for the instructions in `cost` (its blocks by box size).  The
// bound that is cheapest for these 64 records, out of 8, 16, .. 1024 pixels.
__device__ __forceinline__ int self_bound(int area, bool has) {
    constexpr int cost[8] = {75, 80, 90, 105, 135, 190, 285, 500};  // boxes over 8, 16, .. 1024 pixels
    unsigned long long over = __ballot(has && area > 1024);
    int sum = cost[7] * __popcll(over);
    int best = 1024, least = sum + 14 * 1024;
#pragma unroll
    for (int q = 6; q >= 0; --q) {
        const int b = 8 << q;
        const unsigned long long o = __ballot(has && area > b);
        sum += cost[q] * __popcll(o & ~over);
        over = o;
        if (sum + 14 * b < least) {
            least = sum + 14 * b;
            best = b;
        }
    }
    return best;
}

// A square region of a map (a tile, or a part of a long list's tile) that a
// workgroup rasterizes into LDS: its edge RS, its first and last pixels.
struct Region {
    int x0, y0, x1, y1;
};
template <int RS>
__device__ __forceinline__ Region region_at(const RasterCfg& cfg, int x0, int y0) {
    return Region{x0, y0, min(x0 + RS - 1, cfg.w - 1), min(y0 + RS - 1, cfg.h - 1)};
}

template <int RS, bool kVis>
__device__ __forceinline__ void clear_region(typename KeyOf<kVis>::T* tile, int& nrec) {
    constexpr int kWords = RS * tile_pitch<RS>();
    if constexpr (!kVis) {  // 16-byte LDS writes
        constexpr uint32_t c = KeyOf<kVis>::clear;
        for (int q = (int)threadIdx.x; q < kWords / 4; q += kRasterThreads)
            reinterpret_cast<uint4*>(tile)[q] = make_uint4(c, c, c, c);
    } else {
        for (int p = (int)threadIdx.x; p < kWords; p += kRasterThreads) tile[p] = KeyOf<kVis>::clear;
    }
    if (threadIdx.x == 0) nrec = 0;
}

// What a wave knows of the region's depths: lane b the bound of block b's, as
// read `age` wave records ago.
struct ZBound {
    uint32_t zmax;
    int age;
};

// Walk of the fallback, which has no list: the first pieces of 256 triangles,
// then their second ones, and so on, so that a round's lanes have work together
// (a piece per lane of triangles in turn leaves seven lanes of eight idle).
__device__ __forceinline__ uint32_t fallback_length(const MeshView& mesh) {
    return (uint32_t)(mesh.nt + 255) / 256u * 2048u;
}
__device__ __forceinline__ uint32_t fallback_entry(uint32_t k) {
    return ((k / 2048u * 256u + k % 256u) << 3) | (k / 256u % 8u);
}

// Entry k of a tile's list; `has` is false past its end.
template <bool kFallback>
__device__ __forceinline__ uint32_t list_entry(const MeshView& mesh, const BinBufs& b, int map, uint32_t k,
                                               uint32_t end, bool& has) {
    has = k < end;
    if constexpr (kFallback) {
        const uint32_t e = fallback_entry(k);
        has = has && (e >> 3) < (uint32_t)mesh.nt;
        return e;
    } else {
        return has ? b.entries[(size_t)map * b.cap + k] : 0u;
    }
}

// The setup record of a list entry; `has` becomes false for an empty piece.
template <int TS, bool kFallback>
__device__ __forceinline__ void load_setup(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                           const BinBufs& b, int map, uint32_t entry, bool& has, Setup& s) {
    if (!has) return;
    if (!kFallback && (entry & kWideBit)) {
        s = b.wide[(size_t)map * b.wcap + (entry & ~kWideBit)];
    } else if constexpr (!kFallback && wide_span<TS>() <= 4) {
        // a directly binned triangle: the count pass stored its setup
        const size_t at = (size_t)map * b.tstride + (entry >> 3);
        s = from_rec(b.setups[at], b.fars[at], entry, cfg);
    } else {
        float mvp[16];
        mvps.load(map, mvp);
        Tri<0> t;
        if constexpr (kFallback)
            get_piece<0>(mesh, mvp, (int)(entry >> 3), (int)(entry & 7u), cfg, t, has);
        else
            classify<0>(mesh, mvp, (int)(entry >> 3), cfg, t, has);
        if (has) s = to_setup(t, entry);
    }
}

// One round of list entries, one per lane (`has`: the lane has one).  Small
// records are rasterized by their lane, larger ones by the wave in 8x8
// blocks, those of more than `aside` blocks and those with a long edge are put
// aside in `rec`; a long one that finds it full leaves a flag in nrec
// (raster_long).
constexpr int kMoreLong = (int)0x80000000u;
template <int TS, int RS, bool kVis, bool kFallback>
__device__ __forceinline__ void raster_round(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                             const BinBufs& b, int map, const Region& g, uint32_t entry, bool has,
                                             int aside, typename KeyOf<kVis>::T* tile, Setup* rec, int& nrec,
                                             ZBound& z) {
    const int lane = (int)threadIdx.x & 63;
    Setup s;
    load_setup<TS, kFallback>(mesh, mvps, cfg, b, map, entry, has, s);
    int rx0 = 0, rx1 = -1, ry0 = 0, ry1 = -1;
    if (has) {
        rx0 = max(g.x0, s.px0);
        rx1 = min(g.x1, s.px1);
        ry0 = max(g.y0, s.py0);
        ry1 = min(g.y1, s.py1);
        has = rx0 <= rx1 && ry0 <= ry1;
    }
    TileEdges t = {};
    unsigned long long blocks = 0;
    int area = 0;
    if (has) {
        t = tile_edges(s, g.x0, g.y0);
        blocks = block_mask<RS>(rx0 - g.x0, rx1 - g.x0, ry0 - g.y0, ry1 - g.y0);
        area = (rx1 - rx0 + 1) * (ry1 - ry0 + 1);
        if ((s.tl & kLongEdge) || __popcll(blocks) > aside) {
            const int slot = atomicAdd(&nrec, 1) & ~kMoreLong;
            if (slot < kRecQueue) {
                rec[slot] = s;
                has = false;
            } else if (s.tl & kLongEdge) {
                atomicOr(&nrec, kMoreLong);
                has = false;
            }
        }
    }
    const int bound = self_bound(area, has);
    const bool self = has && area <= bound;
    raster_lanes<RS, kVis, false>(s, t, blocks, has && !self, g.x0, g.y0, lane, z.zmax, z.age, tile);
    if (self) raster_rect_self<RS, kVis>(s, t, g.x0, g.y0, rx0, rx1, ry0, ry1, tile);
}

// The records of the queue whose bit is set in `which` (wave-uniform, the same
// in all waves), each by the whole workgroup with the 64-bit edge functions.
template <int RS, bool kVis>
__device__ __forceinline__ void raster_queued_long(const Region& g, const Setup* rec, unsigned which,
                                                   typename KeyOf<kVis>::T* tile) {
    while (which) {
        const Setup r = rec[__ffs((int)which) - 1];
        which &= which - 1;
        raster_rect_slow<RS, kVis>(r, g.x0, g.y0, max(g.x0, r.px0), min(g.x1, r.px1), max(g.y0, r.py0),
                                   min(g.y1, r.py1), (int)threadIdx.x, kRasterThreads, tile);
    }
}

// All records with a long edge among entries [begin, end), where the queue
// could not hold them.  Walking the list again keeps the 64-bit edge functions'
// registers out of raster_round.
template <int TS, int RS, bool kVis, bool kFallback>
__device__ __forceinline__ void raster_long(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                            const BinBufs& b, int map, const Region& g, uint32_t begin, uint32_t end,
                                            typename KeyOf<kVis>::T* tile, Setup* rec, int& nrec) {
    const int tid = (int)threadIdx.x;
    for (uint32_t base = begin; base < end; base += kRasterThreads) {
        bool mine;
        Setup s;
        const uint32_t entry = list_entry<kFallback>(mesh, b, map, base + (uint32_t)tid, end, mine);
        load_setup<TS, kFallback>(mesh, mvps, cfg, b, map, entry, mine, s);
        mine = mine && (s.tl & kLongEdge) && s.px0 <= g.x1 && s.px1 >= g.x0 && s.py0 <= g.y1 && s.py1 >= g.y0;
        for (int n = kRecQueue + 1; n > kRecQueue;) {  // until the queue held all that were left
            __syncthreads();
            if (tid == 0) nrec = 0;
            __syncthreads();
            if (mine) {
                const int slot = atomicAdd(&nrec, 1);
                if (slot < kRecQueue) {
                    rec[slot] = s;
                    mine = false;
                }
            }
            __syncthreads();
            n = nrec;
            raster_queued_long<RS, kVis>(g, rec, (1u << min(n, kRecQueue)) - 1u, tile);
        }
    }
    __syncthreads();
}

// The records put aside; then the region is complete.  A record goes to one
// wave, which sets it up once (about 80 vector instructions, as many as six
// blocks take), and only the remainder of four is shared by block rows; with
// `by_rows`, for launches that leave the GPU room, all are, which ends sooner.  Depth maps go out with non-temporal stores: a frame writes far
// more map bytes than the caches hold (64 x 16 MiB), and with ordinary stores
// the last-written lines stay dirty in the MALL and are written back while
// the screen pass reads the maps.  On the 64-sample 1080p frame this took the
// raster from 0.363 to 0.346 ms, the soft pass that follows from 0.374 to
// 0.341 ms and the frame from 0.991 to 0.940 ms.
template <int TS, int RS, bool kVis, bool kFallback>
__device__ __forceinline__ void finish_region(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                              const BinBufs& b, const Region& g, void* out, int map, uint32_t begin,
                                              uint32_t end, typename KeyOf<kVis>::T* tile, Setup* rec, int& nrec,
                                              ZBound& z, bool by_rows) {
    constexpr int kWaves = kRasterThreads / 64;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __syncthreads();
    const bool more_long = (nrec & kMoreLong) != 0;
    const int nq = min(nrec & ~kMoreLong, kRecQueue);
    if (nq > 0) {  // uniform
        Setup s;
        TileEdges t = {};
        unsigned long long blocks = 0;
        const bool has = lane < nq;
        if (has) {
            s = rec[lane];
            t = tile_edges(s, g.x0, g.y0);
            unsigned long long rows = 0;
            if (!by_rows && lane < (nq & ~(kWaves - 1))) {
                if (lane % kWaves == wave) rows = ~0ull;
            } else {
#pragma unroll
                for (int r = 0; r < RS / 8; r += kWaves) rows |= ((1ull << (RS / 8)) - 1ull) << ((RS / 8) * (r + wave));
            }
            blocks = rows & block_mask<RS>(max(g.x0, s.px0) - g.x0, min(g.x1, s.px1) - g.x0,
                                           max(g.y0, s.py0) - g.y0, min(g.y1, s.py1) - g.y0);
        }
        raster_lanes<RS, kVis, true>(s, t, blocks, has && blocks && !(s.tl & kLongEdge), g.x0, g.y0, lane, z.zmax, z.age, tile);
        raster_queued_long<RS, kVis>(g, rec, (unsigned)__ballot(has && (s.tl & kLongEdge)), tile);
        __syncthreads();
    }
    if (more_long) raster_long<TS, RS, kVis, kFallback>(mesh, mvps, cfg, b, map, g, begin, end, tile, rec, nrec);  // uniform
    constexpr int kPx = RS * RS;
    const size_t plane = (size_t)cfg.w * cfg.h;
    if constexpr (!kVis) {
        float* dst = reinterpret_cast<float*>(out) + (size_t)map * plane;
        const bool full = (g.x1 - g.x0 + 1 == RS) && ((cfg.w & 3) == 0);
        if (full) {
            typedef float f4 __attribute__((ext_vector_type(4)));
            for (int q = tid; q < kPx / 4; q += kRasterThreads) {
                const int r = q / (RS / 4), cidx = (q % (RS / 4)) * 4;
                const int j = g.y0 + r;
                if (j > g.y1) continue;
                const f4 v = *reinterpret_cast<const f4*>(&tile[r * tile_pitch<RS>() + cidx]);
                __builtin_nontemporal_store(v, reinterpret_cast<f4*>(dst + (size_t)j * cfg.w + g.x0 + cidx));
            }
        } else {
            for (int p = tid; p < kPx; p += kRasterThreads) {
                const int i = g.x0 + p % RS, j = g.y0 + p / RS;
                if (i > g.x1 || j > g.y1) continue;
                __builtin_nontemporal_store(__uint_as_float(tile[(p / RS) * tile_pitch<RS>() + p % RS]),
                                            dst + (size_t)j * cfg.w + i);
            }
        }
    } else {
        unsigned long long* dst = reinterpret_cast<unsigned long long*>(out) + (size_t)map * plane;
        if (g.x1 - g.x0 + 1 == RS && (cfg.w & 1) == 0) {  // 16-byte stores
            for (int q = tid; q < kPx / 2; q += kRasterThreads) {
                const int r = q / (RS / 2), cidx = (q % (RS / 2)) * 2;
                const int j = g.y0 + r;
                if (j > g.y1) continue;
                const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(&tile[r * tile_pitch<RS>() + cidx]);
                *reinterpret_cast<ulonglong2*>(dst + (size_t)j * cfg.w + g.x0 + cidx) = v;
            }
            return;
        }
        for (int p = tid; p < kPx; p += kRasterThreads) {
            const int i = g.x0 + p % RS, j = g.y0 + p / RS;
            if (i > g.x1 || j > g.y1) continue;
            dst[(size_t)j * cfg.w + i] = tile[(p / RS) * tile_pitch<RS>() + p % RS];
        }
    }
}

// One (tile, map) of the raster.  kFallback: the map's lists overflowed the
// workspace, so every (triangle, piece) pair is visited with full clipping.
//
// Each wave takes 64 records of every 256 (a record per lane: load, box, edge
// values); no barrier stands between the rounds.  `spread` interleaves them,
// so that a short list reaches all four waves: for launches that leave the GPU
// room (kSpreadTiles).
template <int TS, bool kVis, bool kFallback>
__device__ __forceinline__ void raster_tile(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                            const BinBufs& b, void* out, int map, int tile_id,
                                            typename KeyOf<kVis>::T* tile, Setup* rec, int& nrec, bool spread) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int kWaves = kRasterThreads / 64;
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const Region g = region_at<TS>(cfg, tile_id % cfg.tiles_x * TS, tile_id / cfg.tiles_x * TS);
    uint32_t begin = 0, end;
    if constexpr (!kFallback) {
        begin = b.offsets[(size_t)map * (ntiles + 1) + tile_id];
        end = b.offsets[(size_t)map * (ntiles + 1) + tile_id + 1];
    } else {
        end = fallback_length(mesh);
    }
    if constexpr (!kFallback && !kVis) {
        // A whole tile whose list is one wide record covering every pixel
        // centre (most tiles of a large ground plane): each depth is that
        // plane's, written straight from registers.  The LDS path would store
        // the same bits: min(clear, z) is z for every clamped depth.
        if (end - begin == 1 && g.x1 - g.x0 + 1 == TS && g.y1 - g.y0 + 1 == TS && (cfg.w & 3) == 0) {
            const uint32_t entry = b.entries[(size_t)map * b.cap + begin];
            if (entry & kWideBit) {
                const Setup& w = b.wide[(size_t)map * b.wcap + (entry & ~kWideBit)];
                const Setup s = w;
                if (s.px0 <= g.x0 && s.px1 >= g.x1 && s.py0 <= g.y0 && s.py1 >= g.y1 &&
                    rect_inside(s, g.x0, g.x1, g.y0, g.y1)) {
                    typedef float f4 __attribute__((ext_vector_type(4)));
                    float* dst = reinterpret_cast<float*>(out) + (size_t)map * ((size_t)cfg.w * cfg.h);
                    for (int q = tid; q < TS * TS / 4; q += kRasterThreads) {
                        const int r = q / (TS / 4), cidx = (q % (TS / 4)) * 4;
                        const int i = g.x0 + cidx, j = g.y0 + r;
                        const int dy = j * 256 + 128 - s.Y[0];
                        const f4 v = {__uint_as_float(plane_bits(s, i * 256 + 128 - s.X[0], dy)),
                                      __uint_as_float(plane_bits(s, (i + 1) * 256 + 128 - s.X[0], dy)),
                                      __uint_as_float(plane_bits(s, (i + 2) * 256 + 128 - s.X[0], dy)),
                                      __uint_as_float(plane_bits(s, (i + 3) * 256 + 128 - s.X[0], dy))};
                        __builtin_nontemporal_store(v, reinterpret_cast<f4*>(dst + (size_t)j * cfg.w + i));
                    }
                    return;
                }
            }
        }
    }
    clear_region<TS, kVis>(tile, nrec);
    __syncthreads();
    const int aside = end - begin <= (uint32_t)kShareList ? kShareBlocks : kShareBlocksLong;
    ZBound z{0xFFFFFFFFu, 0};
    for (uint32_t base = begin; base < end; base += kRasterThreads) {
        bool has;
        const uint32_t entry =
            list_entry<kFallback>(mesh, b, map, base + (uint32_t)(spread ? lane * kWaves + wave : tid), end, has);
        raster_round<TS, TS, kVis, kFallback>(mesh, mvps, cfg, b, map, g, entry, has, aside, tile, rec, nrec, z);
    }
    finish_region<TS, TS, kVis, kFallback>(mesh, mvps, cfg, b, g, out, map, begin, end, tile, rec, nrec, z, spread);
}

// ---------------------------------------------------------------------------
// Long lists.  Where a launch has few tiles, one tile's list can be the whole
// launch's time (a mesh far away, a soup in the middle of a large map: 64
// tiles of 1,024 hold 200,000 triangles).  k_scan lists the tiles whose lists
// are long beside the launch's average (split_bound); each is rasterized in 16
// regions of 16x16 pixels by workgroups of their own.  A region's workgroup
// goes through the tile's whole list, but reads only each record's box (its
// first 16 bytes, kBoxes in flight per thread), and rasterizes the entries that
// touch the region from a list in LDS.  Raster of one map, tiles only and with
// split lists: 200k soup, 2048^2: 130 and 46 us (its G-buffer at 1920x1080: 232
// and 67 us); 100,822 triangles seen from 315 units, 2048^2: 98 and 34 us (42
// with a box at a time); a 3,970-triangle scene, 1024^2: 43 and 17 us, 256^2: 26
// and 13 us.
// ---------------------------------------------------------------------------
constexpr int kSplitEdge = 16;
constexpr int kSplitRegions = (kTile / kSplitEdge) * (kTile / kSplitEdge);
constexpr int kSplitLoads = 8;                              // entries per thread and pass over the list
constexpr int kBoxes = 4;                                   // of them whose boxes are read together
static_assert(kSplitLoads % kBoxes == 0, "a pass is whole groups of boxes");
constexpr int kSplitPass = kSplitLoads * kRasterThreads;    // entries a pass looks at, and its LDS list's size

// The region list in LDS, behind the region's pixels in the tile's memory.
template <int TS, bool kVis>
__device__ __forceinline__ uint32_t* split_list(typename KeyOf<kVis>::T* tile) {
    static_assert((size_t)(TS * tile_pitch<TS>() - kSplitEdge * tile_pitch<kSplitEdge>()) *
                          sizeof(typename KeyOf<kVis>::T) >= (size_t)kSplitPass * 4, "the list fits behind the region");
    return reinterpret_cast<uint32_t*>(tile + kSplitEdge * tile_pitch<kSplitEdge>());
}

template <int TS, bool kVis>
__device__ __forceinline__ void raster_region(const MeshView& mesh, const MvpSource& mvps, const RasterCfg& cfg,
                                              const BinBufs& b, void* out, int map, int tile_id, int part,
                                              typename KeyOf<kVis>::T* tile, Setup* rec, int& nrec, int& nlist) {
    constexpr int kParts = TS / kSplitEdge, RS = kSplitEdge, kWaves = kRasterThreads / 64;
    const int tid = (int)threadIdx.x;
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const Region g = region_at<RS>(cfg, tile_id % cfg.tiles_x * TS + part % kParts * RS,
                                   tile_id / cfg.tiles_x * TS + part / kParts * RS);
    if (g.x0 >= cfg.w || g.y0 >= cfg.h) return;  // uniform
    const uint32_t begin = b.offsets[(size_t)map * (ntiles + 1) + tile_id];
    const uint32_t end = b.offsets[(size_t)map * (ntiles + 1) + tile_id + 1];
    const uint32_t* entries = b.entries + (size_t)map * b.cap;
    const char* boxes = reinterpret_cast<const char*>(b.wide + (size_t)map * b.wcap) + offsetof(Setup, px0);
    const char* recs = reinterpret_cast<const char*>(b.setups + (size_t)map * b.tstride);
    uint32_t* list = split_list<TS, kVis>(tile);
    clear_region<RS, kVis>(tile, nrec);
    ZBound z{0xFFFFFFFFu, 0};
    for (uint32_t base = begin; base < end; base += kSplitPass) {
        if (tid == 0) nlist = 0;
        __syncthreads();  // also: the region is cleared, the last pass's list is done with
        // a wide record's box, or the first 16 bytes of a direct one: one load
        // from either address (behind a branch each would wait for the one
        // before it), kBoxes in flight together.  Holding all of a pass takes 95
        // registers, so 5 workgroups per CU instead of 6: the far map above 32
        // us, but a soup over the whole of a 2048^2 map 121 us instead of 116.
        typedef int quad __attribute__((ext_vector_type(4), aligned(8)));
        for (uint32_t b0 = base; b0 < min(base + kSplitPass, end); b0 += kBoxes * kRasterThreads) {  // uniform
            uint32_t e[kBoxes];
            quad v[kBoxes];
#pragma unroll
            for (int q = 0; q < kBoxes; ++q) {
                const uint32_t k = b0 + (uint32_t)(q * kRasterThreads + tid);
                e[q] = k < end ? entries[k] : ~0u;
            }
#pragma unroll
            for (int q = 0; q < kBoxes; ++q) {
                const bool wide = (e[q] & kWideBit) != 0;
                const uint32_t idx = e[q] == ~0u ? 0u : wide ? e[q] & ~kWideBit : e[q] >> 3;
                const uint32_t size = wide ? (uint32_t)sizeof(Setup) : (uint32_t)sizeof(SetupRec);
                v[q] = *reinterpret_cast<const quad*>((wide ? boxes : recs) + (size_t)idx * size);
            }
#pragma unroll
            for (int q = 0; q < kBoxes; ++q) {
                int px0 = v[q].x, px1 = v[q].y, py0 = v[q].z, py1 = v[q].w;
                if (!(e[q] & kWideBit)) {
                    int X[3], Y[3];
                    rec_vertices(v[q].x, v[q].y, (uint32_t)v[q].z, (uint32_t)v[q].w,
                                 b.fars[(size_t)map * b.tstride + (e[q] >> 3)], X, Y);
                    rec_box(X, Y, px0, px1, py0, py1);
                }
                if (e[q] != ~0u && px0 <= g.x1 && px1 >= g.x0 && py0 <= g.y1 && py1 >= g.y0)
                    list[atomicAdd(&nlist, 1)] = e[q];
            }
        }
        __syncthreads();
        const int n = nlist;
        for (int k0 = 0; k0 < n; k0 += kRasterThreads) {
            const int k = k0 + (tid & 63) * kWaves + (tid >> 6);
            const bool has = k < n;
            raster_round<TS, RS, kVis, false>(mesh, mvps, cfg, b, map, g, has ? list[k] : 0u, has,
                                                    (RS / 8) * (RS / 8), tile, rec, nrec, z);
        }
        __syncthreads();  // nlist and the list are rewritten by the next pass
    }
    finish_region<TS, RS, kVis, false>(mesh, mvps, cfg, b, g, out, map, begin, end, tile, rec, nrec, z, true);
}

// Binned raster: one workgroup per (tile, map); overflowed maps are left to
// k_raster_fallback.  Workgroups go out tile-major (the map_count maps of
// tile 0, then of tile 1, ...).  The hardware deals workgroups to CUs in
// turn, about equally many to each, whatever their cost; in map-major order
// the costly tiles (those under the occluder, about 7x the time of a tile
// holding only the ground) arrive in runs that pile onto a few CUs while the
// rest idle.  Tile-major order spreads each costly tile's maps over the XCDs
// and CUs.
template <int TS, bool kVis>
__global__ __launch_bounds__(kRasterThreads, kVis ? 1 : 8) void k_raster(MeshView mesh, MvpSource mvps, RasterCfg cfg,
                                                                         BinBufs b, void* out, int map_base,
                                                                         int map_count, bool spread) {
    __shared__ __align__(16) typename KeyOf<kVis>::T tile[TS * tile_pitch<TS>()];
    __shared__ Setup rec[kRecQueue];
    __shared__ int nrec;
    const int map = map_base + (int)(blockIdx.x % (unsigned)map_count);
    const int tile_id = (int)(blockIdx.x / (unsigned)map_count);
    if (b.overflow[map]) return;
    raster_tile<TS, kVis, false>(mesh, mvps, cfg, b, out, map, tile_id, tile, rec, nrec, spread);
}

// k_raster for launches that split long lists: the first workgroups take a
// (tile, map) each, and of a split tile its first region; kSplitWorkers more
// take the other regions in turn.
constexpr int kSplitWorkers = 1024;
template <int TS, bool kVis>
__global__ __launch_bounds__(kRasterThreads, kVis ? 1 : 6) void k_raster_split(MeshView mesh, MvpSource mvps,
                                                                               RasterCfg cfg, BinBufs b, void* out,
                                                                               int map_base, int map_count) {
    __shared__ __align__(16) typename KeyOf<kVis>::T tile[TS * tile_pitch<TS>()];
    __shared__ Setup rec[kRecQueue];
    __shared__ int nrec, nlist;
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const int bid = (int)blockIdx.x - kSplitWorkers;  // the regions first: they are the long ones
    int map = 0, tile_id = 0, part = 0;
    // the workers' walk: lane m holds the tasks of map m (at most 64 maps)
    int tasks = 0, m = 0, first = 0, t = (int)blockIdx.x;
    if (bid >= 0) {
        map = map_base + bid % map_count;
        tile_id = bid / map_count;
        if (b.overflow[map]) return;
        const uint32_t* o = b.offsets + (size_t)map * (ntiles + 1) + tile_id;
        if (o[1] - o[0] <= split_tiles(b, map)[1]) {
            raster_tile<TS, kVis, false>(mesh, mvps, cfg, b, out, map, tile_id, tile, rec, nrec, true);
            return;
        }
    } else {
        const int lane = (int)threadIdx.x & 63;
        if (lane < map_count && !b.overflow[map_base + lane])
            tasks = (int)split_tiles(b, map_base + lane)[0] * (kSplitRegions - 1);
    }
    for (;;) {
        if (bid < 0) {
            int n = __builtin_amdgcn_readlane(tasks, m);
            while (t >= n) {  // uniform: on to the next map with a task for this worker
                first = (first + n) % kSplitWorkers;
                if (++m == map_count) return;
                t = ((int)blockIdx.x + kSplitWorkers - first) % kSplitWorkers;
                n = __builtin_amdgcn_readlane(tasks, m);
            }
            map = map_base + m;
            tile_id = (int)split_tiles(b, map)[2 + t / (kSplitRegions - 1)];
            part = 1 + t % (kSplitRegions - 1);
            t += kSplitWorkers;
        }
        raster_region<TS, kVis>(mesh, mvps, cfg, b, out, map, tile_id, part, tile, rec, nrec, nlist);
        if (bid >= 0) return;
        __syncthreads();  // the region's LDS is used again
    }
}

// One workgroup per tile, looping over the maps whose lists overflowed.
template <int TS, bool kVis>
__global__ __launch_bounds__(kRasterThreads) void k_raster_fallback(MeshView mesh, MvpSource mvps, RasterCfg cfg,
                                                                    BinBufs b, void* out, int nmaps) {
    __shared__ __align__(16) typename KeyOf<kVis>::T tile[TS * tile_pitch<TS>()];
    __shared__ Setup rec[kRecQueue];
    __shared__ int nrec;
    // The usual case is no overflowed map: the threads read the flags
    // together and the workgroup returns after one barrier.
    bool any = false;
    for (int m = (int)threadIdx.x; m < nmaps; m += (int)blockDim.x) any |= b.overflow[m] != 0;
    if (!__syncthreads_or(any)) return;
    for (int map = 0; map < nmaps; ++map) {
        if (!b.overflow[map]) continue;
        raster_tile<TS, kVis, true>(mesh, mvps, cfg, b, out, map, blockIdx.x, tile, rec, nrec, true);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// G-buffer resolve: GBuffer.frag:35-37 (position, normal, gl_FrontFacing)
// ---------------------------------------------------------------------------
// Perspective-correct attributes of the visible piece at pixel (i, j); false
// when the piece does not cover the pixel centre.  T: Tri<6> or ResolveRec.
template <typename T>
__device__ __forceinline__ bool resolve_attrs(const T& t, int i, int j, float out[6]) {
    const int Px = i * 256 + 128, Py = j * 256 + 128;
    long long e[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = (k + 1) % 3, b = (k + 2) % 3;
        e[k] = (long long)(t.X[b] - t.X[a]) * (Py - t.Y[a]) - (long long)(t.Y[b] - t.Y[a]) * (Px - t.X[a]);
    }
    if (e[0] + t.tl[0] <= 0 || e[1] + t.tl[1] <= 0 || e[2] + t.tl[2] <= 0) return false;
    double b0 = (double)e[0] / (double)t.w[0];
    double b1 = (double)e[1] / (double)t.w[1];
    double b2 = (double)e[2] / (double)t.w[2];
    double den = (b0 + b1) + b2;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        double num = (b0 * (double)t.a[0][q] + b1 * (double)t.a[1][q]) + b2 * (double)t.a[2][q];
        out[q] = (float)(num / den);
    }
    return true;
}

__device__ __forceinline__ void write_gbuffer(size_t npx, size_t k, bool hit, int front, const float a[6],
                                              float* pos_out, float* nrm_out, float* facing_out) {
    float out[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) out[q] = !hit ? 0.0f : (q >= 3 && !front) ? -a[q] : a[q];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        pos_out[q * npx + k] = out[q];
        nrm_out[q * npx + k] = out[3 + q];
    }
    if (facing_out) facing_out[k] = hit && front ? 1.0f : 0.0f;
}

// A thread per pixel, rows of 64 pixels per wave.  The count pass left each
// triangle's class in b.tiles: a clipped one's pieces are read from the
// table that k_clip filled, any other visible triangle lies inside the clip
// planes and is set up from its vertices.  Bound by HBM: 63 us at 3840x2160
// (a 100,822-triangle mesh on a ground quad; 36 B a pixel, 4.7 TB/s).  A
// ground quad that crosses a clip plane covers most of a view; clipping it
// again in every one of its pixels, the kernel took 2.72 ms there, and 200 us
// against 9.6 us now at 800x600 (3,970 triangles).  With the table but the
// pieces past it clipped in this kernel it took 0.33 ms (the call holds 82
// VGPRs and 1.2 KB of scratch per lane), so those have a kernel of their own;
// reading a record once for a wave whose pixels show one piece took the whole
// pass from 154 to 145 us.
// facing_out (optional): gl_FrontFacing as 1 / 0 (GBuffer.frag:36), 0 for
// background.  The normal is stored negated on back faces.
__global__ __launch_bounds__(256) void k_gbuffer_resolve(MeshView mesh, Mat4 mvp_arg, RasterCfg cfg, BinBufs b,
                                                         const unsigned long long* vis, float* pos_out,
                                                         float* nrm_out, float* facing_out) {
    const int i = (int)(blockIdx.x * 64 + (threadIdx.x & 63)), j = (int)(blockIdx.y * 4 + (threadIdx.x >> 6));
    if (i >= cfg.w || j >= cfg.h) return;
    const size_t npx = (size_t)cfg.w * cfg.h;
    const size_t k = (size_t)j * cfg.w + i;
    const unsigned long long key = vis[k];
    float out[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    bool hit = false;
    int front = 0;
    if (key != ~0ull) {
        const uint32_t id = (uint32_t)(key & 0xffffffffull);
        const int tri = (int)(id >> 3), piece = (int)(id & 7u);
        const uint32_t code = b.tiles[tri];
        if (!(code & kClipCode)) {
            CV<6> v[3];
            Tri<6> t;
            load_tri<6>(mesh, mvp_arg.m, tri, v);
            hit = piece == 0 && setup_piece<6>(v[0], v[1], v[2], cfg, t) && resolve_attrs(t, i, j, out);
            front = hit ? t.front : 0;
        } else if (clip_place(code) < b.acap && piece < kMaxPieces) {
            const uint32_t at = clip_place(code) * kMaxPieces + (uint32_t)piece;
            const uint32_t at0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
            if (__ballot(at != at0) == 0ull) {  // one piece in all these lanes
                const ResolveRec t = b.attrs[at0];
                hit = resolve_attrs(t, i, j, out);
                front = t.front;
            } else {
                const ResolveRec t = b.attrs[at];
                hit = resolve_attrs(t, i, j, out);
                front = t.front;
            }
        }
    }
    write_gbuffer(npx, k, hit, front, out, pos_out, nrm_out, facing_out);
}

// The pixels of clipped triangles past the attribute table, clipped again
// here.  Launched where a mesh has more triangles than the table (the host
// does not know how many were listed) and over at once where it sufficed.
__global__ __launch_bounds__(256) void k_gbuffer_resolve_rest(MeshView mesh, Mat4 mvp_arg, RasterCfg cfg, BinBufs b,
                                                              const unsigned long long* vis, float* pos_out,
                                                              float* nrm_out, float* facing_out) {
    if (b.nclip[0] <= b.acap) return;  // uniform
    const size_t npx = (size_t)cfg.w * cfg.h;
    for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < npx; k += (size_t)gridDim.x * 256) {
        const unsigned long long key = vis[k];
        if (key == ~0ull) continue;
        const uint32_t id = (uint32_t)(key & 0xffffffffull);
        const uint32_t code = b.tiles[id >> 3];
        if (!(code & kClipCode) || clip_place(code) < b.acap) continue;
        Tri<6> t;
        bool ok;
        float out[6];
        get_piece<6>(mesh, mvp_arg.m, (int)(id >> 3), (int)(id & 7u), cfg, t, ok);
        const bool hit = ok && resolve_attrs(t, (int)(k % (size_t)cfg.w), (int)(k / (size_t)cfg.w), out);
        write_gbuffer(npx, k, hit, hit ? t.front : 0, out, pos_out, nrm_out, facing_out);
    }
}

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// ---------------------------------------------------------------------------
// Host side: workspace layout of the binned raster (shared by the single
// passes and the batched frames)
// ---------------------------------------------------------------------------
struct Workspace {
    BinBufs bins;
    void* vis;  // gbuffer only
};

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Tile-list entries per map: up to wide_span tiles per directly binned piece
// (pieces are rarely that wide, so 4 tiles per triangle at the 64-texel edge,
// scaled with the tile count for smaller edges) plus the wide pieces' tiles.
inline uint32_t entry_cap(int ntris, int ntiles, int ts = kTile) {
    const unsigned long long per = 4ull * (unsigned long long)(64 / ts) * (unsigned long long)(64 / ts);
    unsigned long long cap = per * (unsigned long long)ntris + 4ull * (unsigned long long)ntiles + 1024ull;
    if (cap > 0x7FFFFFFFull) cap = 0x7FFFFFFFull;
    return (uint32_t)cap;
}

// Clipped triangles whose pieces keep their attributes for the G-buffer
// resolve (14 MiB); the resolve clips those past it again.
constexpr uint32_t kAttrTriangles = 16384u;

constexpr uint32_t wide_cap(int ntris) { return 1024u + (uint32_t)ntris / 16u; }

inline size_t layout(int ntris, int nmaps, int w, int h, bool vis, Workspace* ws, char* base, int ts = kTile) {
    int tx = (w + ts - 1) / ts, ty = (h + ts - 1) / ts;
    size_t ntiles = (size_t)tx * ty;
    uint32_t cap = entry_cap(ntris, (int)ntiles, ts);
    uint32_t wcap = wide_cap(ntris);
    // the G-buffer pass lists every triangle of a mesh that its attribute table holds
    const uint32_t ccap = vis ? std::max(wcap, std::min((uint32_t)std::max(ntris, 0), kAttrTriangles)) : wcap;
    size_t off = 0;
    size_t o_counts = off; off = align256(off + sizeof(uint32_t) * ntiles * nmaps);
    size_t o_nwide = off; off = align256(off + sizeof(uint32_t) * nmaps);
    size_t o_wover = off; off = align256(off + sizeof(int) * nmaps);
    size_t o_nclip = off; off = align256(off + sizeof(uint32_t) * nmaps);
    size_t zero_end = off;  // [0, zero_end) is cleared before binning
    size_t o_offsets = off; off = align256(off + sizeof(uint32_t) * (ntiles + 1) * nmaps);
    size_t o_over = off; off = align256(off + sizeof(int) * nmaps);
    size_t o_wide = off; off = align256(off + sizeof(Setup) * (size_t)wcap * nmaps);
    size_t o_clip = off; off = align256(off + sizeof(uint32_t) * (size_t)ccap * nmaps);
    size_t o_entries = off; off = align256(off + sizeof(uint32_t) * (size_t)cap * nmaps);
    size_t o_tiles = off; off = align256(off + sizeof(uint32_t) * (size_t)(ntris > 0 ? ntris : 0) * nmaps);
    const bool records = 4 * (64 / ts) * (64 / ts) <= 4;  // the tile code's span (wide_span<ts>() <= 4)
    const size_t nrecs = records ? (size_t)(ntris > 0 ? ntris : 0) * nmaps : 0;
    size_t o_setups = off;
    size_t o_fars = off + sizeof(SetupRec) * nrecs;
    off = align256(o_fars + sizeof(FarRec) * nrecs);
    // the G-buffer pass (one map): visibility keys and the clipped pieces' attributes
    const uint32_t acap = vis ? std::min(ccap, kAttrTriangles) : 0u;
    size_t o_vis = off;
    if (vis) off = align256(off + sizeof(unsigned long long) * (size_t)w * h);
    size_t o_attrs = off;
    off = align256(off + sizeof(ResolveRec) * kMaxPieces * (size_t)acap);
    if (ws) {
        BinBufs& b = ws->bins;
        b.counts = reinterpret_cast<uint32_t*>(base + o_counts);
        b.nwide = reinterpret_cast<uint32_t*>(base + o_nwide);
        b.wide_over = reinterpret_cast<int*>(base + o_wover);
        b.offsets = reinterpret_cast<uint32_t*>(base + o_offsets);
        b.overflow = reinterpret_cast<int*>(base + o_over);
        b.wide = reinterpret_cast<Setup*>(base + o_wide);
        b.nclip = reinterpret_cast<uint32_t*>(base + o_nclip);
        b.clip = reinterpret_cast<uint32_t*>(base + o_clip);
        b.entries = reinterpret_cast<uint32_t*>(base + o_entries);
        b.tiles = reinterpret_cast<uint32_t*>(base + o_tiles);
        b.setups = records ? reinterpret_cast<SetupRec*>(base + o_setups) : nullptr;
        b.fars = records ? reinterpret_cast<FarRec*>(base + o_fars) : nullptr;
        b.tstride = (uint32_t)(ntris > 0 ? ntris : 0);
        b.cap = cap;
        b.wcap = wcap;
        b.ccap = ccap;
        b.attrs = vis ? reinterpret_cast<ResolveRec*>(base + o_attrs) : nullptr;
        b.acap = acap;
        ws->vis = vis ? reinterpret_cast<void*>(base + o_vis) : nullptr;
    }
    (void)zero_end;
    return off;
}

// Words to clear before binning: counts, nwide and wide_over are laid out
// contiguously at the start of the workspace.
inline size_t zero_words(int nmaps, const RasterCfg& cfg) {
    size_t ntiles = (size_t)cfg.tiles_x * cfg.tiles_y;
    size_t off = align256(sizeof(uint32_t) * ntiles * nmaps);
    off = align256(off + sizeof(uint32_t) * nmaps);
    off = align256(off + sizeof(int) * nmaps);
    off = align256(off + sizeof(uint32_t) * nmaps);
    return off / sizeof(uint32_t);
}

inline bool size_ok(int w, int h) { return w > 0 && h > 0 && w <= GI_MAX_EDGE && h <= GI_MAX_EDGE; }

}  // namespace
}  // namespace gi
