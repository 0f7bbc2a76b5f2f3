"""The binning stage's timer covers the binning pass alone: not the host's read-back of the record count, nor the buffers
that a view's first render allocates and the pass it makes again.  Against planned rendering, which has none of these:
the host's part made it 1.6 times as long in a repeated render of a toy mesh and over 3 times in a first one of 384,000
tets."""
import statistics

import pytest

from difftetvr_amd import meshgen
from tests.helpers import make_renderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,size,first_only", [(3, 64, False), (40, 512, True)])
def test_binning_stage(gpu, n, size, first_only):
    import difftetvr_amd as d
    w = meshgen.grid_workload(n, seed=1)

    def renderer():
        _, r = make_renderer(d, w["cells"], w["pos"], w["col"], size, size, eye=(0.7, 0.4, 1.5))
        r.set_timing(True)
        return r

    def binning(r):
        r.render()
        return r.get_timings()["count_pairs"]

    binning(renderer())  # loads the kernels
    first = [binning(renderer()) for _ in range(5)]
    r = renderer()
    eager = [binning(r) for _ in range(16)][1:]
    r.set_record_capacity(r.get_stats()["num_pairs"])
    planned = statistics.median([binning(r) for _ in range(16)][1:])
    print(f"first {min(first):.4f} eager {min(eager):.4f} planned {planned:.4f} ms", flush=True)
    assert min(first) < 2.0 * planned
    if not first_only:
        assert min(eager) < 1.3 * planned
