// raster.hip — light-view depth pass and camera visibility/G-buffer pass for gfx950.
//
// Replaces the reference's fixed-function OpenGL rasterization of the light
// view (ShadowMapping/src/main.cpp:221-274 with Scene.vert:11-20, depth into a
// GL_DEPTH_COMPONENT32F texture cleared to 1.0, depth test LESS, no culling)
// and of the camera G-buffer (GBuffer.vert:15-21, GBuffer.frag:35-37).
//
// Design (binned raster, one launch sequence for a whole batch of maps; the
// kernels live in raster_kernels.hpp):
//   1. k_bin      one thread per (triangle, map): transform, classify against
//                 the clip planes, snap, and count the screen tiles each
//                 triangle overlaps (LDS-aggregated); wide and clipped pieces
//                 become setup records (k_clip, k_bin_wide);
//   2. k_scan     one workgroup per map: exclusive scan of the tile counts;
//   3. k_bin      scatter pass: append the triangle id to every overlapped
//                 tile's list;
//   4. k_raster   one workgroup per (tile, map): resolve the tile's list into an
//                 LDS tile with ds_min on the FP32 depth bits (non-negative
//                 floats order like uint32) or on 64-bit (depth, id) keys,
//                 then write the tile to HBM once with 16-byte stores
//                 (k_raster_split: a long list's tile in regions).
// atomicMin makes the result independent of list order, so the output is
// deterministic.  When a map's lists would exceed the workspace, that map falls
// back to every workgroup scanning the whole mesh (slower, same result).
//
// Raster rules (the choices the GL spec leaves to the implementation):
//   clip near (z >= -w), far (z <= w) and a guard band |x|,|y| <= 4w with
//   Sutherland-Hodgman (intersection taken from the inside vertex, so a shared
//   edge clips identically in both triangles), fan triangulation; window
//   coordinates snapped to 1/256 pixel with round-to-nearest-even; pixel
//   centres at (i+.5, j+.5); top-left tie rule in GL's y-up window space;
//   window depth linear in screen space, evaluated as an FP32 plane about
//   vertex 0, z = z0 + (A*(Px-X0) + B*(Py-Y0)), whose slopes are derived in
//   FP64 from the exact integer geometry and rounded once; clamped to [0, 1];
//   optional polygon offset factor*max|dz/dx|,|dz/dy| + units*2^(e-23).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/gi.h"
#include "gi_device.hpp"
#include "gi_internal.hpp"
#include "raster_kernels.hpp"

namespace gi {

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
namespace {

// Tiles of a launch up to which every workgroup is resident at once.
constexpr size_t kSpreadTiles = 2048;

// Whether a depth pass of nmaps maps splits long tile lists (k_raster_split):
// where its long lists are few beside what the GPU holds.  The maps of a pass
// show one mesh, so each brings long lists of its own, and from some number of
// maps on they fill the GPU without being split, while k_raster_split keeps 6
// workgroups per CU where k_raster keeps 8, and its regions read each list 16
// times.  Depth passes with and without splitting, us (a 32,002- and a
// 98,002-triangle body, soups of 50,000 and 200,000):
//   maps            tiles     body        body        soup        soup
//   1 of 512^2         64   48   77     69  126     54   97    105  259
//   4 of 512^2        256   55   79     79  136     99  104    203  279
//   8 of 350^2        288   69  108     99  159    107  119    288  354
//   9 of 512^2        576   64   88    101  145    115  113    303  297
//   16 of 256^2       256   74   87    114  106    131  132    533  406
//   16 of 512^2     1,024   84   94    161  158    120  117    336  327
//   25 of 512^2     1,600  106   98    241  168    148  143    414  389
//   9 of 1024^2     2,304   77   73    112  103    152  144    331  343
//   64 of 256^2     1,024  153  110    282  166    178  169    580  568
//   64 of 512^2     4,096  148  132    274  249    284  273    860  808
// Five to eight maps of 900^2 to 1800^2 take 1% more to 8% less without, in the
// mean of seven meshes (19% more to 21% less with one), and stay split, and so do
// the nine corner maps of an adaptive frame, whose light stands further away (maps
// of 1721^2, 38,722 triangles, the whole frame: 391 us with, 426 without).
// Few maps split, some more while their tiles are few, and large ones, whose one
// long list stands against 1,024 tiles or more.
constexpr size_t kSplitTiles = 12288;
constexpr int kSplitFew = 9;
constexpr int kSplitSome = 16;
constexpr size_t kSplitSomeTiles = 1024;
constexpr int kSplitLarge = 1024;  // tiles of a map
static_assert(kSplitTiles / kSplitLarge <= 64 && kSplitSome <= 64, "the workers hold a map's task count per lane");
bool splits_lists(int ntiles, int nmaps) {
    const size_t tiles = (size_t)ntiles * nmaps;
    return tiles <= kSplitTiles &&
           (nmaps <= kSplitFew || (nmaps <= kSplitSome && tiles <= kSplitSomeTiles) || ntiles >= kSplitLarge);
}

// Into how many shares a launch of `tiles` tiles is thought to be cut, a list
// longer than one being split (split_bound): a share per CU, or smaller ones
// while the tiles leave the GPU room.  Depth passes with 1,024, 512 and 256, us:
// one 512^2 map (64 tiles) of a 50,000-triangle soup 55, -, 80, of a 200,000-
// triangle soup 105, -, 148; one 2048^2 map (1,024 tiles) of these 113, 96, 96
// and 228, 189, 186; three of 900^2 (675) of a 4,830-triangle scene 55, 55, 63.
// More tiles: one 4096^2 map of 100,822 triangles 58 with 1,024, 48 with 256.  A
// CU holds 4 workgroups of a visibility pass: 510 tiles of a 200,000-triangle
// soup's G-buffer 67 us with 1,024, 83 with 256 (the raster alone); 4,096 tiles of
// 16 maps of 50,002 triangles 235 and 138.
template <bool kVis>
uint32_t split_shares(size_t tiles) {
    return tiles <= 256 ? 1024u : tiles <= 1024 ? (kVis ? 1024u : 512u) : 256u;
}

// Binning of every map (count, clip, scan, scatter) and the raster of the
// maps whose lists overflowed the workspace.
template <bool kVis>
int bin_stage(const MeshView& mesh, const MvpSource& mvps, int nmaps, const RasterCfg& cfg, const Workspace& ws,
              void* out, hipStream_t s) {
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    const BinBufs& b = ws.bins;
    size_t nz = zero_words(nmaps, cfg);
    size_t fb = (nz + 255) / 256;
    unsigned fill_blocks = (unsigned)(fb < 4096 ? fb : 4096);
    hipLaunchKernelGGL(k_fill_u32, dim3(fill_blocks), dim3(256), 0, s, b.counts, nz, 0u);
    dim3 gb((mesh.nt + 255) / 256, nmaps);
    dim3 gw(kWideBlocks, nmaps);
    if (mesh.nt > 0) {
        hipLaunchKernelGGL((k_bin<kTile, false>), gb, dim3(256), 0, s, mesh, mvps, cfg, b);
        if (b.attrs)
            hipLaunchKernelGGL(k_clip<6>, dim3(kClipBlocks, nmaps), dim3(kClipThreads), 0, s, mesh, mvps, cfg, b);
        else
            hipLaunchKernelGGL(k_clip<0>, dim3(kClipBlocks, nmaps), dim3(kClipThreads), 0, s, mesh, mvps, cfg, b);
        hipLaunchKernelGGL((k_bin_wide<kTile, false>), gw, dim3(256), 0, s, cfg, b);
    }
    hipLaunchKernelGGL(k_scan, dim3(nmaps), dim3(kScanThreads), 0, s, b, ntiles,
                       splits_lists(ntiles, nmaps) ? nmaps : 0,
                       split_shares<kVis>((size_t)ntiles * nmaps));
    if (mesh.nt > 0) {
        if constexpr (wide_span<kTile>() <= 4) {
            // triangles' appends and the wide records' appends in one launch
            const int tri_blocks = (mesh.nt + 256 * kScatterTris - 1) / (256 * kScatterTris);
            hipLaunchKernelGGL((k_bin_scatter<kTile, kScatterTris>), dim3(tri_blocks + kWideBlocks, nmaps), dim3(256),
                               0, s, mesh, cfg, b, tri_blocks);
        } else {
            hipLaunchKernelGGL((k_bin<kTile, true>), gb, dim3(256), 0, s, mesh, mvps, cfg, b);
            hipLaunchKernelGGL((k_bin_wide<kTile, true>), gw, dim3(256), 0, s, cfg, b);
        }
    }
    hipLaunchKernelGGL((k_raster_fallback<kTile, kVis>), dim3(ntiles), dim3(kRasterThreads), 0, s, mesh, mvps, cfg, b,
                       out, nmaps);
    return hipGetLastError() == hipSuccess ? GI_OK : GI_EDEVICE;
}

// Tile raster of maps [map_begin, map_begin + map_count) from the lists the
// bin stage left in the workspace (maps that overflowed are skipped: the bin
// stage rastered them).
template <bool kVis>
int raster_stage(const MeshView& mesh, const MvpSource& mvps, int nmaps, int map_begin, int map_count,
                 const RasterCfg& cfg, const Workspace& ws, void* out, hipStream_t s, hipEvent_t ev_begin = nullptr,
                 hipEvent_t ev_end = nullptr) {
    const int ntiles = cfg.tiles_x * cfg.tiles_y;
    if (ev_begin && hipEventRecord(ev_begin, s) != hipSuccess) return GI_EDEVICE;
    const unsigned tiles = (unsigned)(ntiles * map_count);
    const dim3 block(kRasterThreads);
    const bool spread = tiles <= kSpreadTiles;
    if (splits_lists(ntiles, nmaps))
        hipLaunchKernelGGL((k_raster_split<kTile, kVis>), dim3(tiles + kSplitWorkers), block, 0, s, mesh, mvps, cfg,
                           ws.bins, out, map_begin, map_count);
    else
        hipLaunchKernelGGL((k_raster<kTile, kVis>), dim3(tiles), block, 0, s, mesh, mvps, cfg, ws.bins, out, map_begin,
                           map_count, spread);
    if (ev_end && hipEventRecord(ev_end, s) != hipSuccess) return GI_EDEVICE;
    return hipGetLastError() == hipSuccess ? GI_OK : GI_EDEVICE;
}

template <bool kVis>
int run_raster(const MeshView& mesh, const MvpSource& mvps, int nmaps, const RasterCfg& cfg, const Workspace& ws,
               void* out, hipStream_t s, hipEvent_t ev_begin = nullptr, hipEvent_t ev_end = nullptr) {
    int rc = bin_stage<kVis>(mesh, mvps, nmaps, cfg, ws, out, s);
    if (rc != GI_OK) return rc;
    return raster_stage<kVis>(mesh, mvps, nmaps, 0, nmaps, cfg, ws, out, s, ev_begin, ev_end);
}

}  // namespace

namespace internal {

size_t vis_raster_workspace_size(int ntris, int nmaps, int w, int h) {
    if (ntris < 0 || nmaps <= 0 || !size_ok(w, h)) return 0;
    return layout(ntris, nmaps, w, h, false, nullptr, nullptr);
}

int vis_raster(const float* pos, int nverts, const int32_t* idx, int ntris, const float* mvps_dev, int nmaps, int w,
               int h, unsigned long long* vis_out, void* ws, size_t ws_bytes, hipStream_t s) {
    if (!pos || (!idx && ntris > 0) || !mvps_dev || !vis_out || !ws || nverts <= 0 || ntris < 0 || nmaps <= 0)
        return GI_EINVAL;
    if (ntris >= (1 << 28)) return GI_ENOTSUP;
    if (!size_ok(w, h)) return GI_ENOTSUP;
    Workspace wsp;
    size_t need = layout(ntris, nmaps, w, h, false, &wsp, reinterpret_cast<char*>(ws));
    if (ws_bytes < need) return GI_ENOSPACE;
    MeshView mesh{pos, nullptr, idx, ntris};
    MvpSource mvps{};
    mvps.dev = mvps_dev;
    RasterCfg cfg{w, h, (w + kTile - 1) / kTile, (h + kTile - 1) / kTile, 0.0f, 0.0f};
    return run_raster<true>(mesh, mvps, nmaps, cfg, wsp, vis_out, s);
}

}  // namespace internal
}  // namespace gi

using namespace gi;

extern "C" {

size_t gi_depth_pass_workspace_size(int ntris, int nmaps, int width, int height) {
    if (ntris < 0 || nmaps <= 0 || !size_ok(width, height)) return 0;
    return layout(ntris, nmaps, width, height, false, nullptr, nullptr);
}

}  // extern "C"

namespace {

struct DepthCall {
    MeshView mesh;
    MvpSource mvps;
    RasterCfg cfg;
    Workspace ws;
};

// Argument checks and workspace layout shared by the depth-pass entry points.
int depth_setup(const float* positions_dev, int nverts, const int32_t* indices_dev, int ntris,
                const float* mvps_dev, int nmaps, int width, int height, const gi_raster_opts* opts,
                float* depth_out_dev, void* workspace_dev, size_t workspace_bytes, DepthCall& d) {
    if (!positions_dev || (!indices_dev && ntris > 0) || !mvps_dev || !depth_out_dev || !workspace_dev)
        return GI_EINVAL;
    if (nverts <= 0 || ntris < 0 || nmaps <= 0) return GI_EINVAL;
    if (ntris >= (1 << 28)) return GI_ENOTSUP;
    if (!size_ok(width, height)) return GI_ENOTSUP;
    if ((reinterpret_cast<uintptr_t>(depth_out_dev) & 15u) != 0) return GI_EINVAL;
    float off_f = opts ? opts->polygon_offset_factor : 0.0f;
    float off_u = opts ? opts->polygon_offset_units : 0.0f;
    if (!std::isfinite(off_f) || !std::isfinite(off_u)) return GI_ENONFINITE;
    size_t need = layout(ntris, nmaps, width, height, false, &d.ws, reinterpret_cast<char*>(workspace_dev));
    if (workspace_bytes < need) return GI_ENOSPACE;
    d.mesh = MeshView{positions_dev, nullptr, indices_dev, ntris};
    d.mvps = MvpSource{};
    d.mvps.dev = mvps_dev;
    d.cfg = RasterCfg{width, height, (width + kTile - 1) / kTile, (height + kTile - 1) / kTile, off_f, off_u};
    return GI_OK;
}

}  // namespace

extern "C" {

int gi_depth_pass(const float* positions_dev, int nverts, const int32_t* indices_dev, int ntris,
                  const float* mvps_dev, int nmaps, int width, int height, const gi_raster_opts* opts,
                  float* depth_out_dev, void* workspace_dev, size_t workspace_bytes, gi_stream stream) {
    DepthCall d;
    int rc = depth_setup(positions_dev, nverts, indices_dev, ntris, mvps_dev, nmaps, width, height, opts,
                         depth_out_dev, workspace_dev, workspace_bytes, d);
    if (rc != GI_OK) return rc;
    return run_raster<false>(d.mesh, d.mvps, nmaps, d.cfg, d.ws, depth_out_dev, reinterpret_cast<hipStream_t>(stream),
                             opts ? reinterpret_cast<hipEvent_t>(opts->raster_begin_event) : nullptr,
                             opts ? reinterpret_cast<hipEvent_t>(opts->raster_end_event) : nullptr);
}

int gi_depth_pass_bin(const float* positions_dev, int nverts, const int32_t* indices_dev, int ntris,
                      const float* mvps_dev, int nmaps, int width, int height, const gi_raster_opts* opts,
                      float* depth_out_dev, void* workspace_dev, size_t workspace_bytes, gi_stream stream) {
    DepthCall d;
    int rc = depth_setup(positions_dev, nverts, indices_dev, ntris, mvps_dev, nmaps, width, height, opts,
                         depth_out_dev, workspace_dev, workspace_bytes, d);
    if (rc != GI_OK) return rc;
    return bin_stage<false>(d.mesh, d.mvps, nmaps, d.cfg, d.ws, depth_out_dev, reinterpret_cast<hipStream_t>(stream));
}

int gi_depth_pass_raster(const float* positions_dev, int nverts, const int32_t* indices_dev, int ntris,
                         const float* mvps_dev, int nmaps, int width, int height, const gi_raster_opts* opts,
                         int map_begin, int map_count, float* depth_out_dev, void* workspace_dev,
                         size_t workspace_bytes, gi_stream stream) {
    DepthCall d;
    int rc = depth_setup(positions_dev, nverts, indices_dev, ntris, mvps_dev, nmaps, width, height, opts,
                         depth_out_dev, workspace_dev, workspace_bytes, d);
    if (rc != GI_OK) return rc;
    if (map_begin < 0 || map_count <= 0 || map_begin > nmaps - map_count) return GI_EINVAL;
    return raster_stage<false>(d.mesh, d.mvps, nmaps, map_begin, map_count, d.cfg, d.ws, depth_out_dev,
                               reinterpret_cast<hipStream_t>(stream),
                               opts ? reinterpret_cast<hipEvent_t>(opts->raster_begin_event) : nullptr,
                               opts ? reinterpret_cast<hipEvent_t>(opts->raster_end_event) : nullptr);
}

size_t gi_gbuffer_pass_workspace_size(int ntris, int width, int height) {
    if (ntris < 0 || !size_ok(width, height)) return 0;
    return layout(ntris, 1, width, height, true, nullptr, nullptr);
}

int gi_gbuffer_pass(const float* positions_dev, const float* normals_dev, int nverts, const int32_t* indices_dev,
                    int ntris, const float mvp[16], int width, int height, float* position_out_dev,
                    float* normal_out_dev, float* facing_out_dev, void* workspace_dev, size_t workspace_bytes,
                    gi_stream stream) {
    if (!positions_dev || !normals_dev || (!indices_dev && ntris > 0) || !mvp || !position_out_dev ||
        !normal_out_dev || !workspace_dev)
        return GI_EINVAL;
    if (nverts <= 0 || ntris < 0) return GI_EINVAL;
    if (ntris >= (1 << 28)) return GI_ENOTSUP;
    if (!size_ok(width, height)) return GI_ENOTSUP;
    for (int i = 0; i < 16; ++i)
        if (!std::isfinite(mvp[i])) return GI_ENONFINITE;
    Workspace ws;
    size_t need = layout(ntris, 1, width, height, true, &ws, reinterpret_cast<char*>(workspace_dev));
    if (workspace_bytes < need) return GI_ENOSPACE;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    MeshView mesh{positions_dev, normals_dev, indices_dev, ntris};
    MvpSource mvps{};
    mvps.dev = nullptr;
    for (int i = 0; i < 16; ++i) mvps.single.m[i] = mvp[i];
    RasterCfg cfg{width, height, (width + kTile - 1) / kTile, (height + kTile - 1) / kTile, 0.0f, 0.0f};
    int rc = run_raster<true>(mesh, mvps, 1, cfg, ws, ws.vis, s);
    if (rc != GI_OK) return rc;
    hipLaunchKernelGGL(k_gbuffer_resolve, dim3((unsigned)((width + 63) / 64), (unsigned)((height + 3) / 4)),
                       dim3(256), 0, s, mesh, mvps.single, cfg, ws.bins,
                       reinterpret_cast<const unsigned long long*>(ws.vis), position_out_dev, normal_out_dev,
                       facing_out_dev);
    if ((uint32_t)ntris > ws.bins.acap)
        hipLaunchKernelGGL(k_gbuffer_resolve_rest, dim3(256), dim3(256), 0, s, mesh, mvps.single, cfg, ws.bins,
                           reinterpret_cast<const unsigned long long*>(ws.vis), position_out_dev, normal_out_dev,
                           facing_out_dev);
    return hipGetLastError() == hipSuccess ? GI_OK : GI_EDEVICE;
}

}  // extern "C"
