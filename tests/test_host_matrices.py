"""Array-at-a-time host matrices against the one-at-a-time functions."""
import numpy as np
import pytest

from globalillumination_amd import camera, passes
from globalillumination_amd.diff import AreaLight, _dot, _normalize, lookat64, perspective64


@pytest.mark.parametrize("n,zbias", [(1, 0.0), (2, 0.005), (64, -0.25), (289, 0.0)])
def test_biased_samples_bits(gi, n, zbias):
    rng = np.random.default_rng(n)
    m = (rng.normal(size=(n, 16)) * 10.0 ** rng.integers(-6, 7, size=(n, 16))).astype(np.float32)
    m[0, :4] = [0.0, -0.0, 1e30, -1e-42]
    got = passes.biased_samples(m, zbias)
    want = np.stack([camera.mat4_mul(camera.bias_matrix(zbias), x) for x in m])
    assert got.shape == (n, 16) and (got.view(np.uint32) == want.view(np.uint32)).all()
    assert all((passes.biased(x, zbias).view(np.uint32) == w.view(np.uint32)).all() for x, w in zip(m, want))
    common, trans = passes.soft_uniforms(m, zbias)
    assert (common.view(np.uint32) == want[-1].view(np.uint32)).all()
    assert (trans.view(np.uint32) == want[:, 12:16].copy().view(np.uint32)).all()


@pytest.mark.parametrize("n", [1, 3, 16])
def test_area_light_matrices(n):
    """All samples at once against a view at a time (1-D lookAt, as glm
    writes it); FP64 sums of three terms, so 8 ulp of the entries' scale."""
    rng = np.random.default_rng(n)
    light = AreaLight((0.1, -0.2, 0.3), rng.uniform(-1, 1, (n, 2)), 64)
    L, r = np.array([3.0, 7.0, 2.0]), 0.25
    P = perspective64(45.0, 1.0, 1.0, 1000.0)
    want = []
    for ox, oy in light.offsets:
        d = r * np.array([ox, oy, 0.0])
        eye, at, up = L + d, np.asarray(light.at) + d, np.asarray(light.up)
        f = _normalize(at - eye)
        s = _normalize(np.cross(f, up))
        u = np.cross(s, f)
        V = np.eye(4)
        V[:3, :3] = s, u, -f
        V[:3, 3] = -_dot(s, eye), -_dot(u, eye), _dot(f, eye)
        want.append(P @ V)
    got = light.matrices(L, r)
    assert got.shape == (n, 4, 4) and got.dtype == np.float64
    np.testing.assert_allclose(got, np.stack(want), rtol=0, atol=8 * 2.0 ** -52 * np.abs(want).max())
    J, h = light.jacobian(L, r), 1e-6
    assert J.shape == (n, 4, 4, 4)
    for k in range(4):
        e = h * np.eye(4)[k]
        fd = (light.matrices(L + e[:3], r + e[3]) - light.matrices(L - e[:3], r - e[3])) / (2 * h)
        # central differences: rounding eps * 10 / h, truncation h^2 times third derivatives of order 1
        np.testing.assert_allclose(J[..., k], fd, rtol=0, atol=1e-7)


@pytest.mark.gpu
@pytest.mark.parametrize("side_stream", [False, True])
def test_host_matrices_may_change_after_the_call(gi, cuda, side_stream):
    """The light matrix is taken when the call is made: earlier work on the
    stream is still running when the host array is overwritten."""
    import torch

    wl = gi.scenes.config3(nsamples=4, view_w=64, view_h=64, sm=256, freq=20)
    dm = gi.DeviceMesh.from_mesh(wl.mesh)
    mvps = np.stack([passes.view_matrices(v)[2] for v in wl.lights])
    want = gi.render_shadow_map(dm, torch.from_numpy(mvps).cuda(), 256, 256)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream() if side_stream else None
    a = torch.randn(2048, 2048, device="cuda")
    outs = []
    for _ in range(4):
        host = mvps.copy()
        a = a @ a * 1e-3
        outs.append(gi.render_shadow_map(dm, host, 256, 256, stream=stream))
        if stream is not None:
            stream.synchronize()
        host[:] = 0.0
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o.view(torch.int32), want.view(torch.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("wrapped", [False, True])
def test_uploads_of_calls_on_another_stream(gi, cuda, wrapped):
    """Passes on a stream that is not torch's current one, several in a row
    with other matrices each, behind work that is still running there: each
    reads its own, though the tensors of the calls before have been dropped.
    Also with an object that only names the stream's handle."""
    import types

    import torch

    wl = gi.scenes.config3(nsamples=4, view_w=64, view_h=64, sm=256, freq=20)
    dm = gi.DeviceMesh.from_mesh(wl.mesh)
    mvps = np.stack([passes.view_matrices(v)[2] for v in wl.lights])
    frames = [np.roll(mvps, k, axis=0) * np.float32(1.0 + 0.05 * k) for k in range(4)]
    g = gi.render_gbuffer(dm, passes.view_matrices(wl.camera)[2], 64, 64)
    soft = passes.SoftParams()
    want = []
    for k, m in enumerate(frames):
        maps = gi.render_shadow_map(dm, torch.from_numpy(m).cuda(), 256, 256)
        trans = torch.from_numpy(passes.soft_uniforms(m, 0.01 * k)[1]).cuda()
        want.append((maps, gi.render_monte_carlo(g, maps, m, soft, zbias=0.01 * k, trans_dev=trans)))
    assert not torch.equal(want[0][0], want[1][0])
    outs = [(torch.empty_like(m), torch.empty_like(s)) for m, s in want]
    a = torch.randn(4096, 4096, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(20):
            a = a @ a * 1e-3
    for k, (m, (maps, out)) in enumerate(zip(frames, outs)):
        handle = types.SimpleNamespace(cuda_stream=stream.cuda_stream) if wrapped else stream
        gi.render_shadow_map(dm, m, 256, 256, out=maps, stream=handle)
        gi.render_monte_carlo(g, maps, m, soft, zbias=0.01 * k, out=out, stream=handle)
    stream.synchronize()
    for (maps, out), (wm, wo) in zip(outs, want):
        assert torch.equal(maps.view(torch.int32), wm.view(torch.int32))
        assert torch.equal(out.view(torch.int32), wo.view(torch.int32))


@pytest.mark.parametrize("r", [0.25, np.float32(0.25), np.array(0.25), np.array([0.25]), np.array([0.25, 0.5, 2.0])])
def test_area_light_radius_forms(r):
    """The radius may be one number or one per axis, as an array too: (N, 4, 4)
    matrices, each that of the light moved by r * (ox, oy, 0)."""
    light = AreaLight((0.1, -0.2, 0.3), np.array([[0.5, -0.25], [-1.0, 0.75]]), 64)
    L = np.array([3.0, 7.0, 2.0])
    got = light.matrices(L, r)
    assert got.shape == (2, 4, 4)
    for m, (ox, oy) in zip(got, light.offsets):
        d = r * np.array([ox, oy, 0.0])
        still = AreaLight(tuple(np.asarray(light.at) + d), np.zeros((1, 2)), 64)
        assert (m == still.matrices(L + d, 0.0)[0]).all()


@pytest.mark.parametrize("L,r", [(np.ones(3), np.ones(2)), (np.ones(3), np.ones((2, 3))), (np.ones(3), np.ones((2, 1))),
                                 (np.ones((1, 3)), 0.5), (np.ones(2), 0.5)])
def test_area_light_refuses_other_shapes(L, r):
    with pytest.raises(ValueError):
        AreaLight((0.1, -0.2, 0.3), np.array([[0.5, -0.25], [-1.0, 0.75]]), 64).matrices(L, r)


def test_area_light_and_views_refuse_other_counts():
    with pytest.raises(ValueError):
        AreaLight((0.1, -0.2, 0.3), np.zeros((0, 2)), 64).matrices(np.ones(3), 0.5)
    with pytest.raises(ValueError):
        lookat64(np.ones((2, 3)), np.zeros((2, 3)), (0.0, 0.0, 1.0))


def test_no_light_matrices_are_refused():
    for f in (passes.soft_uniforms, lambda m: passes.adaptive_trans(m, [])):
        with pytest.raises(ValueError):
            f(np.zeros((0, 16), np.float32))
