"""The occupancy word of a pool slot (pbb_slot.h): over every interleaving of
workgroups that join and leave a running slot, the member indices inside it are
distinct.  A workgroup that reaches its deadline leaves while others stay, and one
that started later may find room in its place."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pbbperm_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is required")

MODEL = r"""
#include <cstdio>
#include <cstdlib>
#include "pbb_slot.h"
using namespace pbb;
static int G, W, epi;
static long joins, paths;
// a workgroup: 0 outside, 1 has read the word `seen`, 2 inside at `base`, 3 has closed the slot, 4 gone
struct Group { int st, seen, base; };
static void walk(const Group *g, int occ)
{
    bool moved = false;
    for (int i = 0; i < G; i++) {
        Group h[4];
        for (int k = 0; k < G; k++) h[k] = g[k];
        int o = occ;
        if (g[i].st == 0) { h[i].st = 1; h[i].seen = occ; }
        else if (g[i].st == 1) {
            // the compare-and-swap of pool_pick; it gives up on a word that admits no one
            if (!slot_open(g[i].seen, W, epi)) h[i].st = 4;
            else if (occ != g[i].seen) h[i].seen = occ;
            else {
                h[i].st = 2; h[i].base = occ & POOL_MEMBERS; o = occ + W;
                if ((o & POOL_MEMBERS) > epi) { printf("over the cap\n"); exit(1); }
                for (int k = 0; k < G; k++)
                    if (k != i && (g[k].st == 2 || g[k].st == 3) && abs(g[k].base - h[i].base) < W) {
                        printf("index %d given twice\n", h[i].base); exit(1);
                    }
                joins++;
            }
        }
        else if (g[i].st == 2) { h[i].st = 3; o = occ | POOL_CLOSING; }
        else if (g[i].st == 3) { h[i].st = 4; o = occ - W; }
        else continue;
        moved = true;
        // the last one out retires the slot
        if ((o & POOL_MEMBERS) == 0) { paths++; continue; }
        walk(h, o);
    }
    if (!moved) paths++;
}
int main(int argc, char **argv)
{
    G = atoi(argv[1]); W = atoi(argv[2]); epi = atoi(argv[3]);
    Group g[4] = {{2, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}};  // group 0 admitted the request
    walk(g, POOL_RUNNING + W);
    printf("%ld joins over %ld paths\n", joins, paths);
    return joins > 0 && paths > 0 ? 0 : 1;
}
"""


@pytest.mark.parametrize("groups,waves,cap", [(3, 4, 8), (4, 4, 12), (4, 1, 4), (4, 2, 4)])
def test_member_indices_are_distinct_whatever_the_order(tmp_path, groups, waves, cap):
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe), str(groups), str(waves), str(cap)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
