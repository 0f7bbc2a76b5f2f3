"""The vertex table of the adjoint's flush (vertex_table.h, compiled here for the host) over batches of 128 vertex slots:
no slot probes more than a few entries, the slots of a vertex share one entry, and in batches of up to 32 distinct
vertices (meshes that share them) fewer than one slot in a thousand is turned away.  Meshes whose tets share no vertex
fill the table: a slot must not walk all of it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include "vertex_table.h"
using namespace dtv;

static uint64_t seed = 88172645463325252ull;
static uint32_t rnd() { seed ^= seed << 13; seed ^= seed >> 7; seed ^= seed << 17; return (uint32_t)(seed >> 16); }

int main() {
    int most = 0, away = 0, few = 0, few_away = 0;
    for (int batch = 0; batch < 20000; batch++) {
        int32_t keys[kFlushTab], vertex[128], entry[128];
        for (int e = 0; e < kFlushTab; e++) keys[e] = -1;
        // the batch's distinct vertices: consecutive ids (tets of their own, up to 128), any ids (up to 128), or the
        // corners of consecutive cubes along an axis of a grid
        const int kind = batch % 3;
        int32_t ids[128];
        int distinct = kind == 2 ? 0 : 6 + (int)(rnd() % 123u);
        const int32_t first = (int32_t)(rnd() & 0x3FFFFFFFu);
        for (int i = 0; i < distinct; i++) ids[i] = kind == 0 ? first + i : (int32_t)(rnd() & 0x7FFFFFFFu);
        if (kind == 2) {
            const int32_t m = 2 + (int32_t)(rnd() % 200u), step[3] = {1, m, m * m}, axis = (int32_t)(rnd() % 3u);
            for (int c = 0; c < 4 + (int)(rnd() % 4u); c++)
                for (int q = 0; q < 8 && distinct < 32; q++) {
                    const int32_t id = first + c * step[axis] + (q & 1) + (q >> 1 & 1) * m + (q >> 2) * m * m;
                    bool known = false;
                    for (int i = 0; i < distinct; i++) known = known || ids[i] == id;
                    if (!known) ids[distinct++] = id;
                }
        }
        for (int s = 0; s < 128; s++) {
            vertex[s] = ids[s < distinct ? s : (int)(rnd() % (uint32_t)distinct)];
            int probes = 0;
            bool created;
            entry[s] = vertex_entry<kFlushTab, kFlushProbes>(vertex[s], created, [&](int e, int32_t v) {
                probes++;
                const int32_t old = keys[e];
                if (old == -1) keys[e] = v;
                return old;
            });
            most = probes > most ? probes : most;
            away += entry[s] < 0;
            if (entry[s] >= 0 && (entry[s] >= kFlushTab || keys[entry[s]] != vertex[s])) return printf("wrong entry\n"), 1;
            for (int r = 0; r < s; r++)
                if (vertex[r] == vertex[s] && entry[r] >= 0 && entry[r] != entry[s]) return printf("two entries\n"), 1;
            if (entry[s] < 0 && probes < kFlushProbes) return printf("turned away after %d probes\n", probes), 1;
            few += distinct <= 32;
            few_away += distinct <= 32 && entry[s] < 0;
        }
    }
    printf("most probes %d, turned away %d, of %d slots in batches of few vertices %d\n", most, away, few, few_away);
    return most > 16 || away == 0 || few_away * 1000 > few;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_probes_are_bounded(tmp_path):
    src, exe = tmp_path / "vertex_table.cpp", tmp_path / "vertex_table"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "difftetvr_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    print(run.stdout)
    assert run.returncode == 0, run.stdout
