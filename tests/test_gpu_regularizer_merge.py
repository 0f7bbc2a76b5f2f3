"""The regulariser's per-workgroup vertex sums at the edges of its tet ranges (1,024 tets, and 2,048 from 2^19 tets
on), with meshes in file order and shuffled (more distinct vertices than a range's table holds), against the FP64
oracle within the regulariser's 1e-5 relative L2."""
import numpy as np
import pytest

import oracle
from difftetvr_amd import meshgen
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tets", [1, 255, 1023, 1024, 1025, 4097, 2049, 2 ** 19 - 1, 2 ** 19 + 1])
@pytest.mark.parametrize("shuffled", [False, True])
def test_merge_ranges(gpu, tets, shuffled):
    import difftetvr_amd as d
    n = max(2, int(np.ceil((tets / 6.0) ** (1.0 / 3.0))))
    pos, cells = meshgen.hex_grid((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), n + 1, n + 1, n + 1)
    rng = np.random.default_rng(tets)
    pos = (pos + rng.uniform(-0.1 / n, 0.1 / n, size=pos.shape)).astype(np.float32)
    cells = (cells[rng.permutation(cells.shape[0])] if shuffled else cells)[:tets]
    mesh = d.TetMesh()
    mesh.set_use_gradients(True)
    mesh.set_tet_mesh_data(cells, pos, np.ones((pos.shape[0], 4), np.float32))
    d.TetRegularizer(mesh, 0.7, 3.0).compute_grad()
    want = oracle.tet_regularizer_grad(cells, pos.astype(np.float64), 0.7, 3.0, dtype=np.float64)
    assert rel_l2(mesh.get_vertex_positions().grad.cpu().numpy(), want) < 1e-5
