"""Batches with more fragments than the forward's list holds (1,024: faces that cover whole 8x8 tiles, up to 32 x 64
fragments a batch) and around its edge, against the waves of 4x4 pixels, whose lists always fit: the same fragments in
the same order, so images, counts and transmittance checkpoints' gradients agree (images bit for bit, gradients 1e-5)."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import make_renderer, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 5, 9, 20])
@pytest.mark.parametrize("cell,ert", [(False, False), (True, False), (False, True)])
def test_lists_in_several_goes(gpu, n, cell, ert):
    import difftetvr_amd as d
    w = meshgen.grid_workload(n, seed=3)
    mesh, r = make_renderer(d, w["cells"], w["pos"], w["col"], 512, 512, eye=(0.5, 0.4, 1.1),
                            attenuation=20.0 if ert else 0.5, use_ert=ert)
    if cell:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], cell_colors=w["col"][w["cells"]].mean(axis=1))
    col = mesh.get_cell_colors() if cell else mesh.get_vertex_colors()
    dimg = torch.from_numpy(np.random.default_rng(n).standard_normal((512, 512, 4)).astype(np.float32)).cuda()
    got = []
    for spp in (128, 64, 256):  # 4,096 tiles: 128 renders waves of 4x4 pixels, the others whole tiles
        r.set_segments_per_pass(spp)
        mesh.get_vertex_positions().grad.zero_()
        col.grad.zero_()
        img = r.render()
        r.render_adjoint(dimg)
        got.append((img, r.get_fragment_counts(), mesh.get_vertex_positions().grad.cpu().numpy().copy(),
                    col.grad.cpu().numpy().copy()))
    assert int(got[0][1].sum()) > 0
    for g in got[1:]:
        assert torch.equal(g[0], got[0][0]) and torch.equal(g[1], got[0][1])
        assert rel_l2(g[2], got[0][2]) < 1e-5 and rel_l2(g[3], got[0][3]) < 1e-5
