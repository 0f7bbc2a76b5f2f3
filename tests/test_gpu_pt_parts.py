"""The Projection renderer's waves of 4x4 pixels (small viewports) against the wave per 8x8 tile that 64 segments per
pass always takes: the same fragments per pixel in the same order, so images are bit-identical, and gradients equal up
to the order of their float sums (1e-5, as for the tile renderer's parts)."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import FOVY, rel_l2

pytestmark = pytest.mark.gpu


# viewports of 1, 1, 6, 12, 750, 3,072 (4x4 waves), 3,136, 5,120 (4x4 in the adjoint only) and 5,184 tiles
@pytest.mark.parametrize("size", [(1, 1), (8, 8), (17, 9), (25, 23), (200, 240), (512, 384), (512, 392),
                                  (640, 512), (648, 512)])
@pytest.mark.parametrize("kind", ["vertex", "cell", "dense", "abs"])
def test_parts_equal_whole_tiles(gpu, size, kind):
    _compare(size, kind, 14)


# faces that cover whole tiles: batches with more fragments than the whole tile's list of 1,024 (listed in several
# goes), and around its edge; 2,304 tiles (4x4 waves, whose lists always fit)
@pytest.mark.parametrize("n", [2, 3, 5, 9])
def test_lists_in_several_goes(gpu, n):
    _compare((384, 384), "vertex", n, (0.5, 0.4, 0.9))


def _compare(size, kind, n, eye=(0.7, -0.5, 1.6)):
    import difftetvr_amd as d
    W, H = size
    w = meshgen.grid_workload(n, seed=5)
    mesh = d.TetMesh()
    mesh.set_use_gradients(True)
    if kind in ("cell", "abs"):
        mesh.set_tet_mesh_data(w["cells"], w["pos"], cell_colors=w["col"][w["cells"]].mean(axis=1))
        col = mesh.get_cell_colors()
    else:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
        col = mesh.get_vertex_colors()
    r = d.Renderer(renderer_type=d.RendererType.PROJECTION)
    r.set_tet_mesh(mesh)
    r.set_attenuation(200.0 if kind == "dense" else 1.0)
    r.set_viewport_size(W, H)
    r.set_camera_fovy(FOVY)
    r.set_view_matrix(meshgen.look_at_view_matrix(eye))
    dimg = torch.from_numpy(np.random.default_rng(1).standard_normal((H, W, 4)).astype(np.float32)).cuda()
    got = []
    for spp in (128, 64):
        r.set_segments_per_pass(spp)
        mesh.get_vertex_positions().grad.zero_()
        col.grad.zero_()
        img = r.render()
        cnt = r.get_fragment_counts()
        r.render_adjoint(dimg, kind == "abs")
        got.append((img, cnt, mesh.get_vertex_positions().grad.cpu().numpy().copy(), col.grad.cpu().numpy().copy()))
    (img, cnt, gp, gc), (img8, cnt8, gp8, gc8) = got
    assert torch.equal(img, img8) and torch.equal(cnt, cnt8)
    assert int(cnt.sum()) > 0
    ep, ec = rel_l2(gp, gp8), rel_l2(gc, gc8)
    print(f"{W}x{H} {kind}: gradients rel L2 pos {ep:.1e} col {ec:.1e}", flush=True)
    assert ep < 1e-5 and ec < 1e-5
