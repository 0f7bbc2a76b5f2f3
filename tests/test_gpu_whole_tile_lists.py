"""The default forward (128 segments per pass) rendering whole 8x8 tiles whose batches hold more fragments than its list
(1,024: faces that cover whole tiles, up to 32 x 64 fragments a batch), in several goes, against the waves of 4x4
pixels, whose lists always fit.  Alone a 512 x 512 view takes the latter (4,096 tiles), and a second item moves the batch
beyond 5,120 tiles, from where it takes whole ones (Projection: 384 x 384, 2,304 tiles, and 3,072).  Images and counts bit
for bit, gradients 1e-5 (float sums)."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import FOVY, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 5, 9, 20])
@pytest.mark.parametrize("projection,cell,ert", [(False, False, False), (False, True, False), (False, False, True),
                                                 (True, False, False), (True, True, False)])
def test_lists_in_several_goes(gpu, n, projection, cell, ert):
    import difftetvr_amd as d
    w, other = meshgen.grid_workload(n, seed=3), meshgen.grid_workload(2, seed=4)
    mesh, filler = d.TetMesh(), d.TetMesh()
    for m in (mesh, filler):
        m.set_use_gradients(True)
    if cell:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], cell_colors=w["col"][w["cells"]].mean(axis=1))
    else:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
    filler.set_tet_mesh_data(other["cells"], other["pos"], other["col"])
    pos, col = mesh.get_vertex_positions(), mesh.get_cell_colors() if cell else mesh.get_vertex_colors()
    view = meshgen.look_at_view_matrix((0.5, 0.4, 1.1))
    rng = np.random.default_rng(n)
    size = 384 if projection else 512
    dimg = [torch.from_numpy(rng.standard_normal((s, s, 4)).astype(np.float32)).cuda() for s in (size, 264)]
    got = []
    for items in ([(mesh, view, size, size)], [(mesh, view, size, size), (filler, view, 264, 264)]):  # 1,089 tiles more
        b = d.BatchRenderer(renderer_type=d.RendererType.PROJECTION if projection else d.RendererType.INTERSECTION)
        b.set_camera_fovy(FOVY)
        b.set_attenuation(20.0 if ert else 0.5)
        b.set_use_early_ray_termination(ert)
        b.set_items(items)
        pos.grad.zero_()
        col.grad.zero_()
        image = b.render()[0].clone()
        counts = b.get_fragment_counts()[0].clone()
        b.render_adjoint(dimg[:len(items)])
        got.append((image, counts, pos.grad.cpu().numpy().copy(), col.grad.cpu().numpy().copy()))
    (image, counts, gp, gc), (image8, counts8, gp8, gc8) = got
    assert int(counts.sum()) > 0
    assert torch.equal(image, image8) and torch.equal(counts, counts8)
    assert rel_l2(gp8, gp) < 1e-5 and rel_l2(gc8, gc) < 1e-5
