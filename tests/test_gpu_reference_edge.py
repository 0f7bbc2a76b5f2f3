"""The reference adjoint on either side of 3,200 tiles, from where it takes whole tiles behind a forward of 4x4-pixel
waves, against a render of whole tiles (64 segments per pass): the same fragments, so gradients agree up to the order of
their float sums (1e-5, as for the parts of tiles).  Uneven viewports, a batch, and tiles in row order among them."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import FOVY, rel_l2

pytestmark = pytest.mark.gpu


# 3,200; 3,264; 63 x 52 = 3,276 uneven; a batch of 2,501 + 783 = 3,284 tiles
@pytest.mark.parametrize("sizes", [[(512, 400)], [(512, 408)], [(500, 411)], [(481, 321), (230, 209)]])
@pytest.mark.parametrize("order", ["cost", "row-major"])
def test_lines(gpu, sizes, order):
    import difftetvr_amd as d
    w = meshgen.grid_workload(12, seed=6)
    mesh = d.TetMesh()
    mesh.set_use_gradients(True)
    mesh.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
    r = d.BatchRenderer(renderer_type=d.RendererType.INTERSECTION)
    r.set_camera_fovy(FOVY)
    r.set_attenuation(1.0)  # (the reference inverts 'over' by 1 - alpha: NaN behind opaque sub-segments)
    r.set_adjoint_mode("reference")
    r.set_tile_order(order)
    views = [meshgen.look_at_view_matrix((0.7, -0.5 + 0.3 * i, 1.6)) for i in range(len(sizes))]
    r.set_items([(mesh, v, W, H) for v, (W, H) in zip(views, sizes)])
    rng = np.random.default_rng(2)
    dimg = [torch.from_numpy(rng.standard_normal((H, W, 4)).astype(np.float32)).cuda() for W, H in sizes]
    got = []
    for spp in (128, 64):
        r.set_segments_per_pass(spp)
        mesh.get_vertex_positions().grad.zero_()
        mesh.get_vertex_colors().grad.zero_()
        images = r.render()
        r.render_adjoint(dimg)
        got.append(([i.clone() for i in images], mesh.get_vertex_positions().grad.cpu().numpy().copy(),
                    mesh.get_vertex_colors().grad.cpu().numpy().copy()))
    assert all(torch.equal(a, b) for a, b in zip(got[0][0], got[1][0]))
    assert np.linalg.norm(got[0][1]) > 0 and np.isfinite(got[0][1]).all()
    assert rel_l2(got[0][1], got[1][1]) < 1e-5 and rel_l2(got[0][2], got[1][2]) < 1e-5
