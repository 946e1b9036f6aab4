"""The rules that give a decode GEMM launch's tiles to its blocks (umdk_amd/csrc/gmm_plan.h), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "umdk_amd", "csrc")
SOURCE = """
#include "gmm_plan.h"
extern "C" int rows32(int n32, int n64, int tall, int G) { return cam::small_rows32(n32, n64, tall, G); }
extern "C" int blocks(int n, int G) { return cam::plan_blocks(n, G); }
extern "C" void gmm2(int b, int G, int t1, int ge, int t2, int c1, int c2, int *out)
{
    const cam::ChainGmm2 p = cam::plan_chain_gmm2(b, G, t1, ge, t2, c1, c2);
    out[0] = p.run, out[1] = p.rn, out[2] = p.next;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    so = str(d / "plan.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(d / "plan.cpp"), "-o", so],
                   check=True)
    return ctypes.CDLL(so)


def tiles(counts, ntn):
    """32-row tiles of a GEMM with ntn N-tiles, its tiles with 64-row ones for the experts of more than 32 rows, and these."""
    tall = sum(-(-c // 64) for c in counts if c > 32)
    return sum(-(-c // 32) for c in counts) * ntn, (tall + sum(0 < c <= 32 for c in counts)) * ntn, tall * ntn


def test_64_row_tiles_only_where_they_save_rounds(plan):
    ragged = [20, 36, 62, 40, 66, 33, 40, 34, 15, 14, 53, 45, 22, 33, 28, 14]
    n32, n64, tall = tiles(ragged, 18)  # 486 and 306 tiles on 256 blocks: two rounds either way
    assert -(-n32 // 256) == -(-n64 // 256) == 2 and plan.rows32(n32, n64, tall, 256)
    assert not plan.rows32(*tiles([45] * 16, 32), 256)   # 1024 -> 512 tiles
    assert not plan.rows32(*tiles([47] * 8, 56), 256)    # 896 -> 448
    assert plan.rows32(*tiles([45] * 8, 16), 256)        # one round
    assert plan.rows32(*tiles([20] * 64, 56), 256)       # no expert of more than 32 rows
    assert not plan.rows32(*tiles([4] * 32 + [128], 16), 256)  # 576 -> 544, three rounds either way, 32 of them tall
    assert not plan.rows32(*tiles([20] * 48 + [45] * 14 + [70] * 2, 36), 256)  # twelve rounds to ten
    for n32 in range(1, 3000, 7):  # rounds, a tall one weighted by a 64-row tile's time, unless few are tall
        for n64 in range(max(1, n32 // 2), n32 + 1, 13):
            for tall in range(0, n64 + 1, 61):
                if not plan.rows32(n32, n64, tall, 256):
                    assert 4 * tall <= n64 or -(-n64 // 256) + 0.25 * -(-tall // 256) <= -(-n32 // 256)


@pytest.mark.parametrize("G", [256, 304, 250])
@pytest.mark.parametrize("t1,t2,c1,c2", [(192, 432, 2304, 512), (200, 1024, 4096, 768), (255, 256, 1024, 512),
                                         (256, 900, 2048, 1024), (8, 16, 1024, 256), (1, 1, 7168, 1024), (0, 0, 512, 512),
                                         (330, 700, 2048, 704), (700, 2000, 14336, 1024), (1144, 2300, 512, 4096)])
def test_chained_decode_gmm2_tiles(plan, G, t1, t2, c1, c2):
    ge = plan.blocks(t1, G) if t1 < G else G
    out, seen, per_block = (ctypes.c_int * 3)(), [], []
    for b in range(G):
        plan.gmm2(b, G, t1, ge, t2, c1, c2, out)
        run, rn, nxt = out
        mine = [t for t in list(range(run, run + rn)) + list(range(nxt, t2, G)) if t < t2]
        assert mine == sorted(mine)  # the first index past the tiles ends a block's sequence
        seen += mine
        per_block.append(len(mine))
    assert sorted(seen) == list(range(t2))  # every tile once
    if t1 <= G:  # no block may start GMM2 before the others: even shares
        assert max(per_block) <= -(-t2 // G)
