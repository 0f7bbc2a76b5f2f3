"""Waves that render a part of a tile (small viewports: 4x4 or 2x2 pixels a wave) against the wave per 8x8 tile that
64 segments per pass always takes: the same fragments per pixel in the same order, so images and fragment lists are
bit-identical, and gradients equal up to the order of their float sums (1e-5, as for the binning tile sizes)."""
import pytest
import torch

from difftetvr_amd import meshgen
from tests.helpers import make_renderer, rel_l2

pytestmark = pytest.mark.gpu


# viewports of 1, 1, 6, 12, 750 (2x2 waves to 768 tiles), 800, 5,120 (4x4 waves) and 5,184 tiles
@pytest.mark.parametrize("size", [(1, 1), (8, 8), (17, 9), (25, 23), (200, 240), (256, 200), (640, 512), (648, 512)])
@pytest.mark.parametrize("kind", ["vertex", "cell", "linear", "dense", "reference"])
def test_parts_equal_whole_tiles(gpu, size, kind):
    import difftetvr_amd as d
    W, H = size
    w = meshgen.grid_workload(14, seed=5)
    mesh, r = make_renderer(d, w["cells"], w["pos"], w["col"], W, H, eye=(0.7, -0.5, 1.6),
                            attenuation=30.0 if kind == "dense" else 1.0, use_ert=kind == "dense")
    if kind == "cell":
        mesh.set_tet_mesh_data(w["cells"], w["pos"], cell_colors=w["col"][w["cells"]].mean(axis=1))
    if kind == "linear":
        r._renderer_type = d.RendererType.PPLL
    if kind == "reference":
        r.set_adjoint_mode("reference")
    dimg = torch.randn(H, W, 4, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    col = mesh.get_cell_colors() if kind == "cell" else mesh.get_vertex_colors()
    got = []
    for spp in (128, 64):
        r.set_segments_per_pass(spp)
        mesh.get_vertex_positions().grad.zero_()
        col.grad.zero_()
        img = r.render()
        cnt, ids = r.get_fragment_counts(), r.get_fragment_ids(64)
        r.render_adjoint(dimg)
        got.append((img, cnt, ids, mesh.get_vertex_positions().grad.cpu().numpy().copy(), col.grad.cpu().numpy().copy()))
    (img, cnt, ids, gp, gc), (img8, cnt8, ids8, gp8, gc8) = got
    assert torch.equal(img, img8) and torch.equal(cnt, cnt8) and torch.equal(ids, ids8)
    assert int(cnt.sum()) > 0
    ep, ec = rel_l2(gp, gp8), rel_l2(gc, gc8)
    print(f"{W}x{H} {kind}: gradients rel L2 pos {ep:.1e} col {ec:.1e}", flush=True)
    assert ep < 1e-5 and ec < 1e-5
