"""The ordered fragment export at the edges of its batches of 32 records: stacks of tets that each show one face over the
whole view, so that every tile holds exactly as many records as the stack tets, with room for fewer, as many and more ids
per pixel, and behind early ray termination.  8-pixel tiles and 16-pixel ones (whose kernel tests the coverage itself)
against the oracle's lists."""
import numpy as np
import pytest

import oracle
from tests.helpers import FOVY, ZFAR, ZNEAR, make_renderer, view_from

EYE = (0.0, 0.0, 2.0)


def _stack(k):
    z = -0.01 * np.arange(k)
    front = np.array([[-9.0, -7.0], [9.0, -7.0], [0.0, 11.0]])
    pos = np.zeros((k, 4, 3))
    pos[:, :3, :2] = front
    pos[:, :3, 2] = z[:, None]
    pos[:, 3] = np.stack([0.0 * z, 0.0 * z, z - 0.005], axis=1)  # the apex behind: its three faces look away
    return (np.arange(4 * k, dtype=np.int32).reshape(-1, 4), pos.reshape(-1, 3).astype(np.float32),
            np.full((4 * k, 4), 0.5, np.float32))


def _lists(k, W, H):
    cells, pos, _ = _stack(k)
    uf, _ = oracle.camera_uniforms(view_from(EYE), FOVY, ZNEAR, ZFAR, W, H)
    return oracle.Fragments(cells, pos, uf, ZNEAR, W, H).lists()


@pytest.mark.parametrize("k", [1, 33])
def test_one_record_per_tet(k):
    off, ids = _lists(k, 20, 13)
    assert np.array_equal(np.diff(off), np.full(20 * 13, k))
    assert np.array_equal(ids.reshape(-1, k) // 4, np.broadcast_to(np.arange(k), (20 * 13, k)))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 31, 32, 33, 63, 64, 65, 97])
@pytest.mark.parametrize("tile", [8, 16])
@pytest.mark.parametrize("ert", [False, True])
def test_lists(gpu, k, tile, ert):
    import difftetvr_amd as d
    W, H = 20, 13
    cells, pos, col = _stack(k)
    # early ray termination after about 20 of the stack's segments of 0.005 (density 0.5 x attenuation)
    _, r = make_renderer(d, cells, pos, col, W, H, eye=EYE, attenuation=200.0 if ert else 1.0, use_ert=ert)
    r.set_tile_size(tile)
    r.render()
    counts = r.get_fragment_counts().cpu().numpy().reshape(-1)
    _, ids = _lists(k, W, H)
    ids = ids.reshape(-1, k)
    assert np.all(counts == k) if not ert or k == 1 else np.all((counts > 0) & (counts <= k))
    assert not ert or k < 63 or np.all(counts < k)
    for room in (1, max(k - 1, 1), k, k + 3):
        got = r.get_fragment_ids(room).cpu().numpy().reshape(-1, room)
        want = np.full_like(got, -1)
        n = min(room, k)
        want[:, :n] = np.where(np.arange(n) < counts[:, None], ids[:, :n], -1)
        assert np.array_equal(got, want)
