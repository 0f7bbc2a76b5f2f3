"""The Projection renderer between 3,073 and 5,120 tiles, where the forward renders whole tiles and the adjoint 4x4-pixel
parts, whose coverage masks it derives again: planned rendering (the record count stays on the device, here below, at and
above the room for it), one call and captured in a graph, against eager rendering.  Images are bit-identical, gradients
equal up to the order of their float sums (1e-5, as for the parts)."""
import numpy as np
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import FOVY, rel_l2

pytestmark = pytest.mark.gpu


def _setup(d, n, W, H, cell):
    w = meshgen.grid_workload(n, seed=9)
    mesh = d.TetMesh()
    mesh.set_use_gradients(True)
    if cell:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], cell_colors=w["col"][w["cells"]].mean(axis=1))
    else:
        mesh.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
    r = d.Renderer(renderer_type=d.RendererType.PROJECTION)
    r.set_tet_mesh(mesh)
    r.set_attenuation(1.0)
    r.set_viewport_size(W, H)
    r.set_camera_fovy(FOVY)
    r.set_view_matrix(meshgen.look_at_view_matrix((0.7, -0.5, 1.6)))
    return mesh, r, mesh.get_cell_colors() if cell else mesh.get_vertex_colors()


@pytest.mark.parametrize("size", [(512, 392), (507, 421), (640, 512)])  # 3,136, 3,392 and 5,120 tiles
@pytest.mark.parametrize("cell", [False, True])
def test_planned_equals_eager(gpu, size, cell):
    import difftetvr_amd as d
    W, H = size
    mesh, r, col = _setup(d, 12, W, H, cell)
    pos = mesh.get_vertex_positions()
    dimg = torch.from_numpy(np.random.default_rng(3).standard_normal((H, W, 4)).astype(np.float32)).cuda()

    def step():
        pos.grad.zero_()
        col.grad.zero_()
        img = r.render()
        r.render_adjoint(dimg)
        return img

    def result(img):
        torch.cuda.synchronize()
        return img.clone(), pos.grad.cpu().numpy().copy(), col.grad.cpu().numpy().copy()

    def check(got):
        assert torch.equal(got[0], eager[0])
        assert rel_l2(got[1], eager[1]) < 1e-5 and rel_l2(got[2], eager[2]) < 1e-5

    eager = result(step())
    assert np.linalg.norm(eager[1]) > 0 and np.linalg.norm(eager[2]) > 0
    records = r.get_stats()["num_pairs"]
    for capacity in (records, records + 1, 3 * records):
        r.set_record_capacity(capacity)
        check(result(step()))
        assert r.records_overflowed() == (False, records)
    # captured, with eager work between the replays
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        img = step()
    for _ in range(3):
        pos.grad.fill_(7.0)
        img.fill_(-1.0)
        graph.replay()
        check(result(img))


def test_too_many_records_are_reported(gpu):
    import difftetvr_amd as d
    mesh, r, col = _setup(d, 12, 512, 392, False)
    r.render()
    records = r.get_stats()["num_pairs"]
    r.set_record_capacity(records - 5)
    img = r.render()
    r.render_adjoint(torch.ones_like(img))
    assert r.records_overflowed() == (True, records)
    assert bool(torch.isfinite(img).all()) and bool(torch.isfinite(mesh.get_vertex_positions().grad).all())
