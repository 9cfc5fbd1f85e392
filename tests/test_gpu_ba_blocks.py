"""The block LDL^T pose solve (more than 20 free poses) at the edges of its
64-row blocks: the solution of the system that the GPU assembled against
numpy's fp64 solve of the same S and b, and a pivot that fails in a later
block.

Bound: both solves are backward stable, so they differ by at most about
2 n eps cond(S) of the solution's norm.
"""
import numpy as np
import pytest

from helpers import announce, gpu_or_fail, norm_rel
import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def slk():
    return gpu_or_fail()


def _run(slk, p, lm, ep):
    d = {k: slk.DeviceArray.from_host(p[k])
         for k in ("poses", "disps", "intr", "target", "weight", "eta", "ii", "jj")}
    ctx = slk.Context(p["h"], p["w"], max_batch=1, levels=1)
    ctx.ba_iterate(d["poses"], d["disps"], d["intr"], d["target"], d["weight"], d["eta"], d["ii"],
                   d["jj"], p["ii"], p["jj"], p["t0"], p["t1"], lm, ep)
    return ctx, d


# n = 126 (2 blocks, 2 padded rows), 132 (3 blocks, 4 rows in the last), 192
# (3 whole blocks), 198, 384 (6 whole blocks), 390 (6 rows in the seventh)
@pytest.mark.parametrize("P", [21, 22, 32, 33, 64, 65])
def test_solution_at_block_edges(slk, P):
    announce(f"ba block solve n={6 * P}")
    p = wl.ba_problem(n=P + 2, h=6, w=8, seed=70 + P)
    ctx, _ = _run(slk, p, 1e-4, 1e-2)
    assert ctx.ba_status() == slk.SLK_OK
    S, b, dx = ctx.ba_last_system()
    ctx.close()
    n = 6 * P
    assert S.shape == (n, n)
    assert norm_rel(dx, np.linalg.solve(S, b)) < 2 * n * np.finfo(float).eps * np.linalg.cond(S)


@pytest.mark.parametrize("frame", [2, 20, 34])
def test_failed_pivot_in_a_later_block(slk, frame):
    """33 free poses (n = 198, 4 blocks) with no damping and the edges of one
    frame at zero weight: the first pivot of that pose is zero (pivot 0, in
    the first panel; 108, in the second block; 192, at the fourth block's
    start)."""
    announce(f"ba block solve, zero pose {frame}")
    p = wl.ba_problem(n=35, h=6, w=8, seed=90)
    p["weight"][(p["ii"] == frame) | (p["jj"] == frame)] = 0.0
    ctx, d = _run(slk, p, 0.0, 0.0)
    assert ctx.ba_status() == slk.SLK_E_NOT_SPD
    np.testing.assert_array_equal(d["poses"].to_host(), p["poses"])
    np.testing.assert_array_equal(d["disps"].to_host(), p["disps"])
    ctx.close()
