"""The raster's dispatch and kernels at the sizes where they can go wrong,
bit for bit against the CPU oracle (coverage is integer arithmetic and depth
one fixed FP32 expression, so no tolerance is due)."""
import numpy as np
import pytest

from helpers import bits_equal, clip_heavy_mesh, clipped_count, mismatch_report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_small,n_clip,listed", [(50, 1, (0, 1)), (300, 5, (1, 5)), (8000, 200, (100, 200)),
                                                   (16, 3000, (1213, 3000)), (16, 24000, (16385, 24000))])
def test_gbuffer_of_clipped_triangles(gi, oracle_lib, cuda, n_small, n_clip, listed):
    """Pixels of clipped triangles read their piece's attributes from the clip
    kernel's table; the last mesh lists more triangles than the table's
    16,384, so the others are clipped again."""
    mesh, view = clip_heavy_mesh(n_small, n_clip)
    rng = np.random.default_rng(5)
    mesh.normals[:] = rng.normal(size=mesh.normals.shape).astype(np.float32)
    mvp = gi.passes.view_matrices(view)[2]
    assert listed[0] <= clipped_count(mesh, mvp) <= listed[1]
    w, h = 131, 67
    g = gi.render_gbuffer(gi.DeviceMesh.from_mesh(mesh), mvp, w, h)
    pos, nrm, fac = oracle_lib.gbuffer(mesh.positions, mesh.normals, mesh.indices, mvp, w, h)
    for name, got, want in (("position", g.position, pos), ("normal", g.normal, nrm), ("facing", g.facing, fac)):
        got = got.cpu().numpy()
        assert bits_equal(got, want), mismatch_report(got, want, name)
