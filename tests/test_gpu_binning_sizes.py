"""Workgroups of 64 and of 256 tets in the binning pass, against each other and against the oracle.

* A mesh of more than 65,536 tets takes 256 a workgroup when its view has fewer than 1.25 pixels a tet, and 64 when a
  second item of the batch (a toy mesh in a large viewport) moves the batch beyond that: image and fragment counts of the
  first are bit-identical.  Tile and Projection renderer, the mesh first and last in the batch.
* The same mesh alone at few pixels a tet against the oracle: the tile renderer's fragment lists (bit-exact) and the
  Projection renderer's counts and image (2e-5: the Projection tests' 16^3 grid has 1e-5, this one half as many triangles
  again per ray)."""
import numpy as np
import pytest
import torch

import oracle
from difftetvr_amd import meshgen
from tests.helpers import FOVY, ZFAR, ZNEAR, make_renderer, view_from

pytestmark = pytest.mark.gpu
EYE = (0.9, 0.5, 1.3)


def _large():
    w = meshgen.grid_workload(23, seed=2)
    assert w["cells"].shape[0] > 65536
    return w


def _mesh(d, w):
    mesh = d.TetMesh()
    mesh.set_tet_mesh_data(w["cells"], w["pos"], w["col"])
    return mesh


@pytest.mark.parametrize("projection", [False, True])
@pytest.mark.parametrize("first", [True, False])
def test_sizes_agree(gpu, projection, first):
    import difftetvr_amd as d
    large, small = _mesh(d, _large()), _mesh(d, meshgen.grid_workload(2, seed=1))
    view = meshgen.look_at_view_matrix(EYE)
    got = []
    for W, H in ((32, 24), (400, 300)):  # 0.1 and 1.7 pixels a tet in all
        b = d.BatchRenderer(renderer_type=d.RendererType.PROJECTION if projection else d.RendererType.INTERSECTION)
        b.set_camera_fovy(FOVY)
        b.set_attenuation(1.0)
        items = [(large, view, 97, 89), (small, view, W, H)]
        b.set_items(items if first else items[::-1])
        images, counts = b.render(), b.get_fragment_counts()
        got.append((images[0 if first else 1].clone(), counts[0 if first else 1].clone()))
    assert int(got[0][1].sum()) > 0
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_lists_against_oracle(gpu):
    import difftetvr_amd as d
    W, H = 100, 90
    w = _large()
    _, r = make_renderer(d, w["cells"], w["pos"], w["col"], W, H, eye=EYE)
    r.render()
    uf, _ = oracle.camera_uniforms(view_from(EYE), FOVY, ZNEAR, ZFAR, W, H)
    off, ids = oracle.Fragments(w["cells"], w["pos"], uf, ZNEAR, W, H).lists()
    counts = np.diff(off)
    n = int(counts.max())
    got = r.get_fragment_ids(n).cpu().numpy().reshape(-1, n)
    want = np.full_like(got, -1)
    want[np.arange(n)[None, :] < counts[:, None]] = ids
    assert n > 0 and np.array_equal(got, want)


def test_projection_against_oracle(gpu):
    import difftetvr_amd as d
    W, H = 61, 47
    w = _large()
    r = d.Renderer(renderer_type=d.RendererType.PROJECTION)
    r.set_tet_mesh(_mesh(d, w))
    r.set_attenuation(1.0)
    r.set_viewport_size(W, H)
    r.set_camera_fovy(FOVY)
    r.set_view_matrix(meshgen.look_at_view_matrix(EYE))
    img = r.render().cpu().numpy()
    uf, _ = oracle.camera_uniforms(view_from(EYE), FOVY, ZNEAR, ZFAR, W, H)
    fr = oracle.ProjFragments(w["cells"], w["pos"], w["col"], uf, ZNEAR, W, H)
    assert np.array_equal(r.get_fragment_counts().cpu().numpy(), fr.counts())
    want, _ = oracle.proj_forward(fr, w["pos"], w["col"], uf, 1.0)
    assert np.abs(img - want).max() < 2e-5
