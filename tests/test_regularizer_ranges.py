"""How the regulariser splits a mesh over workgroups (vertex_table.h, compiled here for the host), and its gradients at
the edges of each split's ranges, with vertices shared and of the tets' own, against the FP64 oracle within the
regulariser's 1e-5 relative L2.  A small mesh, and one whose tets share no vertex, must not make a thread search the table
more than 16 times in a row: the searches are its latency (3,072 tets with vertices of their own: 23 us with four tets a
thread and eight probes, 4.7 now, 4.3 with one atomic per value)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle
from difftetvr_amd import meshgen
from tests.helpers import rel_l2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include "vertex_table.h"
using namespace dtv;
int main() {
    for (int64_t T = 1; T <= (1 << 22); T = T < 64 ? T + 1 : T + T / 7)
        for (int k = 0; k < 4; k++) {
            const int64_t V = k == 0 ? T / 6 + 4 : k == 1 ? 2 * T - 1 : k == 2 ? 2 * T : 4 * T;
            const RegRange r = regularizer_range(T, V);
            const bool chain = (T < (1 << 17) || V >= 4 * T) && 4 * r.per * kRegProbes > 16;
            // the launch has a kernel for it, and large workgroups come only where every CU gets one
            const bool known = (r.threads == 128 && r.per == 1) || (r.threads == 256 && r.per == 2) ||
                               (r.threads == 512 && r.per == 4);
            if (chain || !known || (r.per == 4 && T < 256 * 512 * 4)) {
                printf("T %lld V %lld: %d x %d\n", (long long)T, (long long)V, r.threads, r.per);
                return 1;
            }
        }
    // every vertex of a range of tets of their own finds an entry or is turned away after kRegProbes
    int32_t keys[512];
    for (int32_t& k : keys) k = -1;
    int most = 0, found = 0;
    for (int32_t v = 0; v < 512; v++) {
        int probes = 0;
        const int e = grouped_entry<512, kRegProbes>(1000 + v, [&](int at, int32_t id) {
            probes++;
            const int32_t old = keys[at];
            if (old == -1) keys[at] = id;
            return old;
        });
        most = probes > most ? probes : most;
        found += e >= 0;
        if (e >= 0 ? keys[e] != 1000 + v : probes != kRegProbes) return printf("wrong entry\n"), 1;
    }
    return most > kRegProbes || found < 384;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_rule(tmp_path):
    src, exe = tmp_path / "ranges.cpp", tmp_path / "ranges"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "difftetvr_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("tets", [1, 127, 128, 129, 2 ** 17 - 1, 2 ** 17, 2 ** 17 + 511, 2 ** 17 + 513, 2 ** 19 + 2049])
@pytest.mark.parametrize("own", [False, True])
def test_gradients(gpu, tets, own):
    import difftetvr_amd as d
    n = max(2, int(np.ceil((tets / 6.0) ** (1.0 / 3.0))))
    pos, cells = meshgen.hex_grid((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), n + 1, n + 1, n + 1)
    pos = (pos + np.random.default_rng(tets).uniform(-0.1 / n, 0.1 / n, size=pos.shape)).astype(np.float32)
    cells = cells[:tets]
    if own:
        pos = pos[cells.reshape(-1)]
        cells = np.arange(cells.size, dtype=np.int32).reshape(-1, 4)
    mesh = d.TetMesh()
    mesh.set_use_gradients(True)
    mesh.set_tet_mesh_data(cells, pos, np.ones((pos.shape[0], 4), np.float32))
    d.TetRegularizer(mesh, 0.7, 3.0).compute_grad()
    want = oracle.tet_regularizer_grad(cells, pos.astype(np.float64), 0.7, 3.0, dtype=np.float64)
    assert rel_l2(mesh.get_vertex_positions().grad.cpu().numpy(), want) < 1e-5
