"""The binning pass and the record sort where their paths change: per-pixel fragment lists against the oracle
(bit-exact), eager and planned.

* a face in front of the near plane by a millionth: 27 bits of depth difference and 14 of tiles, so the sort's first
  passes carry 64-bit keys;
* one tet over the whole view: thousands of candidate tiles in one workgroup;
* workgroups of 64 and of 256 tets (more than 65,536 tets, below and above 1.25 pixels a tet), against the binning
  with 16-pixel tiles, whose coverage is tested per pixel: bit-identical images and lists."""
import numpy as np
import pytest
import torch

import oracle
from difftetvr_amd import meshgen
from tests.helpers import FOVY, ZFAR, ZNEAR, grid_case, make_renderer, view_from

pytestmark = pytest.mark.gpu


def _near_mesh():
    """A coarse grid seen from (0, 0, 1), and a tet whose front face lies 1e-6 behind the near plane."""
    w = grid_case(6, seed=4)
    z = 1.0 - np.array([0.010001, 0.0100011, 0.0100012, 0.0109])
    tet = np.stack([np.array([-0.002, 0.0021, 0.0002, 0.0001]), np.array([-0.0015, -0.0012, 0.0023, 0.0]), z], 1)
    V = w["pos"].shape[0]
    pos = np.concatenate([w["pos"], tet.astype(np.float32)])
    cells = np.concatenate([w["cells"], np.array([[V, V + 1, V + 2, V + 3]], np.int32)])
    col = np.concatenate([w["col"], np.full((4, 4), 0.5, np.float32)])
    return cells, pos, col, (0.0, 0.0, 1.0)


def _large_tet():
    pos = np.array([[-2.0, -1.5, 0.2], [2.0, -1.5, 0.1], [0.0, 2.5, 0.0], [0.0, 0.0, -0.7]], np.float32)
    return np.array([[0, 1, 2, 3]], np.int32), pos, np.full((4, 4), 0.6, np.float32), (0.1, 0.2, 1.4)


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("case,size", [("near", (1024, 1024)), ("near", (640, 480)), ("near", (33, 20)),
                                       ("large", (1024, 1024)), ("large", (1000, 72))])
def test_fragment_lists(gpu, case, size, planned):
    import difftetvr_amd as d
    W, H = size
    cells, pos, col, eye = _near_mesh() if case == "near" else _large_tet()
    _, r = make_renderer(d, cells, pos, col, W, H, eye=eye)
    if planned:  # the capacity is the record count itself
        r.render()
        r.set_record_capacity(r.get_stats()["num_pairs"])
    img = r.render()
    uf, _ = oracle.camera_uniforms(view_from(eye), FOVY, ZNEAR, ZFAR, W, H)
    fr = oracle.Fragments(cells, pos, uf, ZNEAR, W, H)
    off, ids = fr.lists()
    counts = np.diff(off)
    assert np.array_equal(r.get_fragment_counts().cpu().numpy().reshape(-1), counts) and counts.max() > 0
    if case == "near":
        assert (ids // 4 == cells.shape[0] - 1).any()  # the near tet is seen
    n = int(counts.max())
    got = r.get_fragment_ids(n).cpu().numpy().reshape(-1, n)
    want = np.full_like(got, -1)
    want[np.arange(n)[None, :] < counts[:, None]] = ids
    assert np.array_equal(got, want)
    assert bool(torch.isfinite(img).all())
    assert r.records_overflowed()[0] is False


@pytest.mark.parametrize("size", [(100, 90), (330, 300)])  # 0.12 and 1.36 pixels a tet of 73,002
def test_workgroup_sizes(gpu, size):
    import difftetvr_amd as d
    W, H = size
    w = meshgen.grid_workload(23, seed=2)
    assert w["cells"].shape[0] > 65536
    _, r = make_renderer(d, w["cells"], w["pos"], w["col"], W, H, eye=(0.9, 0.5, 1.3))
    img, ids = r.render(), r.get_fragment_ids(128)
    r.set_tile_size(16)
    assert torch.equal(r.render(), img) and torch.equal(r.get_fragment_ids(128), ids)
    assert int((ids >= 0).sum()) > 0
