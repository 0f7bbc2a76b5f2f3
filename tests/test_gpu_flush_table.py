"""The adjoint's per-batch vertex table: every tet of a mesh with vertices of its own (a batch of 32 records then has
up to 128 distinct vertices, more than the table holds) against the mesh that shares them.  Each pixel evaluates the
same fragments, so only the order of the gradient sums differs: within 1e-5 relative L2."""
import numpy as np
import pytest
import torch

from tests.helpers import grid_case, make_renderer, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width,height", [(2, 16, 16), (6, 64, 48), (12, 200, 168), (8, 608, 600)])
def test_tets_with_vertices_of_their_own(gpu, n, width, height):
    import difftetvr_amd as d
    w = grid_case(n=n, seed=31)
    flat = w["cells"].reshape(-1)
    own = np.arange(flat.size, dtype=w["cells"].dtype).reshape(-1, 4)
    eye = (0.4, -0.3, 2.0)
    m1, r1 = make_renderer(d, w["cells"], w["pos"], w["col"], width, height, eye=eye)
    m2, r2 = make_renderer(d, own, w["pos"][flat], w["col"][flat], width, height, eye=eye)
    a, b = r1.render(), r2.render()
    assert torch.equal(a, b)
    dimg = torch.from_numpy(np.random.default_rng(n).standard_normal(a.shape).astype(np.float32)).cuda()
    r1.render_adjoint(dimg)
    r2.render_adjoint(dimg)
    for get in ("get_vertex_positions", "get_vertex_colors"):
        want = getattr(m1, get)().grad.double().cpu().numpy()
        got = np.zeros_like(want)
        np.add.at(got, flat, getattr(m2, get)().grad.double().cpu().numpy())
        assert np.linalg.norm(want) > 0 and rel_l2(got, want) <= 1e-5
