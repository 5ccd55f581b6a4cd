"""Shared helpers of the parity tests: build workloads, run the HIP path and
the oracle on identical inputs."""
from __future__ import annotations

import numpy as np


def light_mvps(workload) -> np.ndarray:
    from globalillumination_amd import passes

    return np.stack([passes.view_matrices(v)[2] for v in workload.lights])


def camera_mvp(workload) -> np.ndarray:
    from globalillumination_amd import passes

    return passes.view_matrices(workload.camera)[2]


def bits_equal(a: np.ndarray, b: np.ndarray) -> bool:
    a = np.ascontiguousarray(a)
    b = np.ascontiguousarray(b)
    return a.shape == b.shape and bool((a.view(np.uint32) == b.view(np.uint32)).all())


def mismatch_report(a: np.ndarray, b: np.ndarray, name: str = "") -> str:
    d = a.view(np.uint32) != b.view(np.uint32)
    idx = np.argwhere(d)
    n = int(d.sum())
    head = idx[:5].tolist()
    vals = [(float(a[tuple(i)]), float(b[tuple(i)])) for i in idx[:5]]
    return f"{name}: {n} of {d.size} differ; first {head} values {vals}"


def shrink_soup(n: int, seed: int = 1):
    from globalillumination_amd import scenes

    soup = scenes.triangle_soup(n, seed=seed)
    return scenes.Mesh.concat(soup, scenes.ground_quad(40.0, 40.0, 0.0))


def clip_heavy_mesh(n_small: int = 8000, n_clip: int = 200, seed: int = 3):
    """n_small tiny triangles under a light at (0, 10, 0.1) and n_clip large
    ones around the light's eye, most of which straddle the near plane or the
    guard band and are cut into fan pieces by the clip kernel."""
    from globalillumination_amd import scenes

    rng = np.random.default_rng(seed)
    eye = np.array([0.0, 10.0, 0.1], np.float32)
    big = eye + rng.uniform(-15, 15, size=(n_clip, 3, 3))
    cen = np.c_[rng.uniform(-3, 3, n_small), rng.uniform(0, 2, n_small), rng.uniform(-3, 3, n_small)]
    small = cen[:, None, :] + rng.uniform(-0.05, 0.05, size=(n_small, 3, 3))
    pos = np.concatenate([small, big]).astype(np.float32)
    n = n_small + n_clip
    nrm = np.tile(np.array([0, 1, 0], np.float32), (3 * n, 1))
    mesh = scenes.Mesh(pos.reshape(-1, 3), nrm, np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    light = scenes.View((0.0, 10.0, 0.1), (0.0, 0.0, 0.0), 128, 128, fov=60.0)
    return mesh, light


def overflow_mesh(n: int = 64, seed: int = 7, size: int = 1024):
    """n large overlapping triangles under a light at (0, 50, 0.1), fov 90:
    every one touches every tile, so the tile lists exceed the workspace
    bound and the map goes through the fallback raster."""
    from globalillumination_amd import scenes

    rng = np.random.default_rng(seed)
    pos = rng.uniform(-30, 30, size=(n, 3, 3)).astype(np.float32)
    pos[:, :, 1] = rng.uniform(0.0, 2.0, size=(n, 3))
    nrm = np.tile(np.array([0, 1, 0], np.float32), (3 * n, 1))
    mesh = scenes.Mesh(pos.reshape(-1, 3), nrm, np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    light = scenes.View((0.0, 50.0, 0.1), (0.0, 0.0, 0.0), size, size, fov=90.0)
    return mesh, light


def wide_overflow_mesh(n: int = 3000, seed: int = 11, size: int = 512):
    """n mid-sized triangles under a light at (0, 40, 0.1), each wider than
    the binning's per-thread span: more setup records than the workspace
    holds, so the map goes through the fallback raster."""
    from globalillumination_amd import scenes

    rng = np.random.default_rng(seed)
    cen = rng.uniform(-6, 6, size=(n, 1, 3))
    pos = (cen + rng.uniform(-3, 3, size=(n, 3, 3))).astype(np.float32)
    pos[:, :, 1] = rng.uniform(0.0, 3.0, size=(n, 3))
    nrm = np.tile(np.array([0, 1, 0], np.float32), (3 * n, 1))
    mesh = scenes.Mesh(pos.reshape(-1, 3), nrm, np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    light = scenes.View((0.0, 40.0, 0.1), (0.0, 0.0, 0.0), size, size, fov=45.0)
    return mesh, light


def clipped_count(mesh, mvp, guard=4.0):
    """Triangles the depth pass lists for clipping: not outside any of the six
    planes (z + w, w - z, x + g w, g w - x, y + g w, g w - y >= 0, g the guard
    band) and not inside all of them."""
    M = np.asarray(mvp, np.float64).reshape(4, 4).T
    h = np.c_[mesh.positions.astype(np.float64), np.ones(mesh.nverts)] @ M.T
    x, y, z, w = h.T
    d = np.stack([z + w, w - z, x + guard * w, guard * w - x, y + guard * w, guard * w - y], 1)[mesh.indices]
    reject = (d < 0).all(axis=1).any(axis=1)
    inside = (d >= 0).all(axis=(1, 2))
    return int((~reject & ~inside).sum())


def longest_edge(tri, mvp, w, h):
    """The longest edge, in x and units of 1/256 pixel, of one triangle's clipped
    pieces in a w x h view, among those between two heights of the view: the
    raster rules (clip planes, intersection from the inside vertex, fan,
    snapping) restated in FP32."""
    f = np.float32
    m = np.asarray(mvp, f).reshape(4, 4)

    def dist(c, p):
        return [c[2] + c[3], c[3] - c[2], c[0] + f(4) * c[3], f(4) * c[3] - c[0], c[1] + f(4) * c[3],
                f(4) * c[3] - c[1]][p]

    poly = [((m[0] * v[0] + m[1] * v[1]) + m[2] * v[2]) + m[3] * f(1) for v in np.asarray(tri, f)]
    for p in range(6):
        out = []
        for k in range(len(poly)):
            prev, cur = poly[k - 1], poly[k]
            dp, dc = dist(prev, p), dist(cur, p)
            if (dc >= 0) != (dp >= 0):
                a, b, da, db = (cur, prev, dc, dp) if dc >= 0 else (prev, cur, dp, dc)
                out.append(a + da / (da - db) * (b - a))
            if dc >= 0:
                out.append(cur)
        poly = out
    best = 0
    for j in range(1, len(poly) - 1):
        piece = [poly[0], poly[j], poly[j + 1]]
        if min(c[3] for c in piece) > 0:
            xy = [[int(np.rint((c[i] / c[3] * f(s * 0.5) + f(s * 0.5)) * f(256))) for i, s in ((0, w), (1, h))]
                  for c in piece]
            for (xa, ya), (xb, yb) in zip(xy, xy[1:] + xy[:1]):
                if 0 <= min(ya, yb) and max(ya, yb) <= 256 * h:
                    best = max(best, abs(xa - xb))
    return best


def horizon_scene(n_long, n_small, w, h, extent, seed=2):
    """n_long triangles that reach `extent` units to the left and right of a
    camera, each with a clipped edge of 32,768 pixels or more (its ends lie
    outside the guard band) across the w x h view, and n_small little ones in
    front.  Returns (mesh, mvp)."""
    from globalillumination_amd import passes, scenes

    view = scenes.View((0.0, 1.0, 0.0), (0.0, 0.95, -3.0), w, h, fov=60.0, znear=0.1, zfar=1000.0, up=(0, 1, 0))
    mvp = passes.view_matrices(view)[2]
    rng = np.random.default_rng(seed)
    tris = []
    for _ in range(20000):
        if len(tris) == n_long:
            break
        side, y, z = rng.uniform(0.1, 1.0, size=2), rng.uniform(-1.0, 2.5, size=3), -rng.uniform(3.0, 8.0, size=3)
        t = np.array([[-extent * side[0], y[0], z[0]], [extent * side[1], y[1], z[1]], [0.0, y[2] * 4.0, z[2]]],
                     np.float32)
        if longest_edge(t, mvp, w, h) >= 1 << 23:
            tris.append(t)
    assert len(tris) == n_long
    cen = np.c_[rng.uniform(-60, 60, n_small), rng.uniform(0.5, 1.0, n_small), rng.uniform(-6, -2, n_small)]
    small = cen[:, None, :] + rng.uniform(-0.03, 0.03, size=(n_small, 3, 3))
    pos = np.concatenate([np.reshape(tris, (-1, 3, 3)), small]).astype(np.float32)
    nt = len(pos)
    nrm = rng.normal(size=(3 * nt, 3)).astype(np.float32)
    return scenes.Mesh(pos.reshape(-1, 3), nrm, np.arange(3 * nt, dtype=np.int32).reshape(nt, 3)), mvp


def fence_mesh(n, w, h, length, thick, seed=4):
    """n thin triangles of about `length` x `thick` pixels for a w x h view and
    an identity matrix, upright and level in turn, each within one column or row
    of 64-pixel tiles where it fits one, over the whole view."""
    from globalillumination_amd import scenes

    rng = np.random.default_rng(seed)
    long = length * rng.uniform(0.9, 1.1, size=n)
    pos = np.empty((n, 3, 3))
    for k in range(n):
        a, b = (h, w) if k % 2 else (w, h)  # across, along
        tile = 64 * rng.integers(0, (a + 63) // 64)
        c = tile + 1 + rng.uniform(0, max(min(62, a - tile - 2) - thick, 0))
        s = rng.uniform(-0.6 * long[k], b - 0.4 * long[k])
        px = np.array([[c, s], [c + thick, s + 0.1 * long[k]], [c + 0.3 * thick, s + long[k]]])
        pos[k, :, :2] = (px[:, ::-1] if k % 2 else px) * [2.0 / w, 2.0 / h] - 1.0
        pos[k, :, 2] = rng.uniform(-0.9, 0.9, size=3)
    nrm = rng.normal(size=(3 * n, 3)).astype(np.float32)
    return scenes.Mesh(pos.reshape(-1, 3).astype(np.float32), nrm, np.arange(3 * n, dtype=np.int32).reshape(n, 3))
