"""Batches of 1 to 18 meshes whose vertex gradients are folded in launches of up to eight, and meshes that share one
colour gradient buffer (folded one after the other), against each mesh's own adjoint: the same fragments' gradients in
another order of float sums, 1e-5 relative L2."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import FOVY, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,shared", [(1, False), (2, True), (8, False), (9, True), (18, False)])
def test_folds_of_several_meshes(gpu, count, shared):
    import difftetvr_amd as d
    items, meshes, works = [], [], []
    common = None
    for i in range(count):
        w = meshgen.grid_workload(4, seed=40 + i) if shared else meshgen.grid_workload(2 + i % 5, seed=40 + i)
        m = d.TetMesh()
        m.set_use_gradients(True)
        m.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
        if shared:
            common = m.get_vertex_colors().grad if common is None else common
            m.get_vertex_colors().grad = common
        works.append(w)
        meshes.append(m)
        items.append((m, meshgen.look_at_view_matrix((0.3, 0.2 + 0.05 * i, 2.0)), 40 + 3 * i, 33))
    br = d.BatchRenderer()
    br.set_attenuation(1.0)
    br.set_camera_fovy(FOVY)
    br.set_items(items)
    images = br.render()
    rng = np.random.default_rng(count)
    dimgs = [torch.from_numpy(rng.standard_normal(tuple(im.shape)).astype(np.float32)).cuda() for im in images]
    br.render_adjoint(dimgs)
    total = 0.0
    for m, w, (_, view, width, height), g in zip(meshes, works, items, dimgs):
        one = d.TetMesh()
        one.set_use_gradients(True)
        one.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
        r = d.Renderer(renderer_type=d.RendererType.INTERSECTION)
        r.set_tet_mesh(one)
        r.set_attenuation(1.0)
        r.set_viewport_size(width, height)
        r.set_camera_fovy(FOVY)
        r.set_view_matrix(view)
        r.render()
        r.render_adjoint(g)
        assert rel_l2(m.get_vertex_positions().grad.cpu().numpy(), one.get_vertex_positions().grad.cpu().numpy()) < 1e-5
        want = one.get_vertex_colors().grad.double().cpu().numpy()
        if shared:
            total = total + want
        else:
            assert rel_l2(m.get_vertex_colors().grad.cpu().numpy(), want) < 1e-5
    if shared:
        assert rel_l2(common.cpu().numpy(), total) < 1e-5
