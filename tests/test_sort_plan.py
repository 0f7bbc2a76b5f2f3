"""The record sort's compact keys (sort_plan.h, compiled here for the host): for every width of the tile number and of
the depth difference, the digits that the passes read from 64- and 32-bit keys are those of the compact key, and the
sorted 32-bit key gives the tile back, the view of one tile whose depth keys span 32 bits included (a shift by 32)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include "sort_plan.h"
using namespace dtv;

static uint32_t low_bits(int n) { return n >= 32 ? 0xFFFFFFFFu : (1u << n) - 1u; }

int main() {
    uint64_t seed = 88172645463325252ull;
    auto random = [&] { seed ^= seed << 13; seed ^= seed >> 7; seed ^= seed << 17; return (uint32_t)(seed >> 16); };
    int checked = 0;
    for (int tbits = 0; tbits <= 32; tbits++)
        for (int dbits = 0; dbits <= 32; dbits++) {
            const uint32_t dmin = dbits == 32 ? 5u : 0x3F000000u;
            const SortPlan p = plan_sort(dmin, dbits, tbits);
            if (p.passes > 8 || 8 * p.passes < p.total || p.tile_shift() > 32u) {
                printf("tbits %d dbits %d: %d passes, shift %u\n", tbits, dbits, p.passes, p.tile_shift());
                return 1;
            }
            for (int i = 0; i < 64; i++) {
                uint32_t tile = i & 1 ? random() : 0xFFFFFFFFu, depth = i & 2 ? random() : 0xFFFFFFFFu;
                if (i < 4) tile = 0u;
                tile &= low_bits(tbits);
                depth = dmin + (depth & low_bits(dbits));
                if (dbits == 32 && depth < dmin) continue;  // below the smallest depth key
                const uint64_t key = compact_key(((uint64_t)tile << 32) | depth, p);
                const uint32_t key32 = (uint32_t)(key >> p.drop);
                for (int pass = 0; pass < p.passes; pass++) {
                    const uint32_t want = (uint32_t)(key >> (8 * pass)) & 255u;
                    const uint32_t got = pass <= p.last_wide() ? want : (key32 >> (8 * pass - p.drop)) & 255u;
                    if (got != want || (p.total < 64 && (key >> p.total) != 0)) {
                        printf("tbits %d dbits %d pass %d: digit %u, not %u\n", tbits, dbits, pass, got, want);
                        return 1;
                    }
                }
                if (tile_of_key(key32, p.tile_shift()) != tile) {
                    printf("tbits %d dbits %d: tile %u, not %u\n", tbits, dbits, tile_of_key(key32, p.tile_shift()), tile);
                    return 1;
                }
                checked++;
            }
        }
    printf("checked %d\n", checked);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_compact_keys(tmp_path):
    src, exe = tmp_path / "sort_plan.cpp", tmp_path / "sort_plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "difftetvr_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
