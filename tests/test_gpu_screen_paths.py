"""Screen-pass kernels at the sizes where their tables and index arithmetic can
go wrong, bit for bit against the CPU oracle (the same FP32 expressions in the
same order)."""
import numpy as np
import pytest

from helpers import bits_equal, camera_mvp, light_mvps, mismatch_report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("search,kernel", [(2, 2), (3, 64), (64, 3), (8, 31), (63, 16)])
def test_pcss_table_sizes(gi, oracle_lib, cuda, search, kernel):
    """The blocker search's offsets and the kernel's, from one tap per axis
    to the largest sizes the pass takes, odd and even."""
    sm = 300
    wl = gi.scenes.config3(nsamples=1, view_w=161, view_h=91, sm=sm, freq=20)
    wl.lights = [gi.scenes.View((120.0, 280.0, 80.0), (0.0, 0.0, 0.0), sm, sm, fov=5.0)]
    dm = gi.DeviceMesh.from_mesh(wl.mesh)
    g = gi.render_gbuffer(dm, camera_mvp(wl), 161, 91)
    mvps = light_mvps(wl)
    depth = gi.render_shadow_map(dm, mvps, sm, sm, polygon_offset=(4.0, 20.0))
    MV, nm, lpos = gi.phong_uniforms(wl.camera, wl.lights[0].eye)
    p = gi.PCSSParams(lightMVP=mvps[0], shadowMapWidth=sm, shadowMapHeight=sm, lightSourceRadius=64,
                      blockerSearchSize=search, kernelSize=kernel, preEvaluation=True, MV=MV, normalMatrix=nm,
                      lightPosition=lpos)
    got = gi.render_soft_shadows(g, depth[0], p).cpu().numpy()
    op = oracle_lib.make_params(gi.biased(mvps[0]), sm, sm, "naive", shadow_intensity=0.25, pre_evaluation=True, mv=MV,
                                normal_matrix=nm, light_position=lpos)
    want = oracle_lib.pcss(g.position.cpu().numpy(), g.normal.cpu().numpy(), depth[0].cpu().numpy(), op,
                           blocker_search_size=search, kernel_size=kernel, light_source_radius=64, z_near=1)
    assert bits_equal(got, want), mismatch_report(got, want, f"search {search} kernel {kernel}")


@pytest.mark.parametrize("w,h,div", [(64, 48, 1), (129, 67, 1), (129, 67, 2), (100, 75, 4), (127, 33, 33), (16, 16, 16)])
def test_node_test_grids(gi, oracle_lib, cuda, w, h, div):
    """Evaluation.frag's reduced grids: full, divisors that do and do not
    divide the view, down to one cell per axis."""
    wl = gi.scenes.config3(nsamples=4, view_w=w, view_h=h, sm=128, freq=20)
    dm = gi.DeviceMesh.from_mesh(wl.mesh)
    g = gi.render_gbuffer(dm, camera_mvp(wl), w, h)
    mvps = light_mvps(wl)
    maps = gi.render_shadow_map(dm, mvps, 128, 128)
    biased = np.stack([gi.biased(m) for m in mvps])
    img, count = gi.passes.quadtree_node_test(g, maps, [0, 1, 2, 3], biased, div)
    want_img, want_count = oracle_lib.qt_node_test(g.position.cpu().numpy(), maps.cpu().numpy(), [0, 1, 2, 3], biased,
                                                   div)
    assert bits_equal(img.cpu().numpy(), want_img)
    assert count == want_count
