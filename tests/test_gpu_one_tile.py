"""A view of one tile whose depth keys lie on either side of the sign bit (faces at the near plane, of which one's
centroid rounds to an NDC z below 0): the compact sort keys are all depth, 32 bits.  Fragment lists against the oracle
(bit-exact) and the image of dtv_render_noalloc against dtv_render's."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from tests.helpers import FOVY, ZFAR, ZNEAR, grid_case, make_renderer, view_from

EYE = (0.9, 0.7, 1.3)


def _mesh():
    """A coarse grid, a tet whose first three vertices have clip w >= znear and clip z < 0 in float32, and one whose
    first three have clip z = 0."""
    w = grid_case(6, seed=4)
    V = w["pos"].shape[0]
    tets = np.array([[0.89544189, 0.699063659, 1.29035854], [0.892488778, 0.693865538, 1.29520202],
                     [0.897938311, 0.693095922, 1.29184365], [0.892934501, 0.693012595, 1.28870213],
                     [0.891354978, 0.699039221, 1.29320109], [0.897143364, 0.697822452, 1.28984892],
                     [0.892996609, 0.692890465, 1.29537547], [0.890747488, 0.694876075, 1.2892127]], np.float32)
    return (np.concatenate([w["cells"], V + np.arange(8, dtype=np.int32).reshape(2, 4)]),
            np.concatenate([w["pos"], tets]), np.concatenate([w["col"], np.full((8, 4), 0.5, np.float32)]))


def _fragments(W, H):
    cells, pos, _ = _mesh()
    uf, _ = oracle.camera_uniforms(view_from(EYE), FOVY, ZNEAR, ZFAR, W, H)
    return oracle.Fragments(cells, pos, uf, ZNEAR, W, H)


@pytest.mark.parametrize("size", [(8, 8), (5, 3), (16, 16), (32, 20)])
def test_keys_span_32_bits(size):
    fr = _fragments(*size)
    keys, ids = fr.triangles()
    near = 4 * (_mesh()[0].shape[0] - 2)
    off, frag = fr.lists()
    seen = np.isin(ids, frag)
    assert (frag >= near).any() and (frag < near).any()
    assert int(keys[seen].max()) - int(keys[seen].min()) >= 1 << 31


@pytest.mark.gpu
@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("size,tile", [((8, 8), 8), ((5, 3), 8), ((16, 16), 16), ((32, 20), 32)])
def test_one_tile(gpu, size, tile, planned):
    import difftetvr_amd as d
    from difftetvr_amd import _lib
    W, H = size
    cells, pos, col = _mesh()
    _, r = make_renderer(d, cells, pos, col, W, H, eye=EYE)
    r.set_tile_size(tile)
    if planned:  # the capacity is the record count itself
        r.render()
        r.set_record_capacity(r.get_stats()["num_pairs"])
    img = r.render()
    off, ids = _fragments(W, H).lists()
    counts = np.diff(off)
    assert np.array_equal(r.get_fragment_counts().cpu().numpy().reshape(-1), counts)
    n = int(counts.max())
    got = r.get_fragment_ids(n).cpu().numpy().reshape(-1, n)
    want = np.full_like(got, -1)
    want[np.arange(n)[None, :] < counts[:, None]] = ids
    assert np.array_equal(got, want)
    assert r.records_overflowed()[0] is False
    if tile == 8:
        out = torch.full((H, W, 4), float("nan"), device="cuda")
        desc, cam, prm = r.get_tet_mesh()._desc(), r._camera(), r._params()
        rc = _lib.load().dtv_render_noalloc(
            d._ctx(), ctypes.byref(desc), ctypes.byref(cam), ctypes.byref(prm), ctypes.c_void_p(out.data_ptr()),
            ctypes.c_void_p(0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0 and torch.equal(out, img)
