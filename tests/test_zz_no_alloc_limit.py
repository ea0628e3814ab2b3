"""The allocation-free step at the very limit of its working memory.

What a case takes of the 64 MiB is an account of its blocks, cells and faces
that programs may rely on (a case accepted once stays accepted).  Seven channel
blocks of 160 x 64 cells with WENO5's ghost width take exactly all of it; one
cell more per row does not fit, and the refusal states the account.
"""
import copy

import numpy as np
import pytest

from pyugks_amd import cases

pytestmark = pytest.mark.gpu


def account(widths, height, ghost):
    """Bytes of a channel case: regions of 256 bytes, in the order of the working memory."""
    n = len(widths)
    faces = sum(w * (height - 1) + (w + 1) * height for w in widths)       # south and north are walls
    cells = sum((w + 2 * ghost) * (height + 2 * ghost) for w in widths)
    regions = [1168 * n, 8 * 4 * (n + 1), 16 * 4 * n, 16 * 4 * n, 4 * n, 4 * 2, 80, 8 * n, 8 * n,
               32 * cells, 128 * faces, 256 * faces, 64 * faces, 4 * faces]
    return sum((r + 255) // 256 * 256 for r in regions)


def test_noalloc_takes_the_case_that_fills_its_working_memory(hip):
    from pyugks_amd import lib as L
    from pyugks_amd.fused import StepPlan, run_noalloc
    from pyugks_amd.sim import UGKSim
    cap = L.load().ugks_step_noalloc_capacity()
    widths, height = [160] * 7, 64
    assert account(widths, height, 3) == cap
    g = cases.cfg5_channel(widths=widths, height=height, nc=8, Kn=0.05)
    print("[gpu] noalloc at its limit", flush=True)
    a, b = UGKSim(copy.deepcopy(g)), UGKSim(copy.deepcopy(g))
    plan = StepPlan(a, "fp64")
    plan.run(1)
    run_noalloc(b, "fp64", 1)
    for x, y in zip(a.blocks, b.blocks):
        assert np.array_equal(x.f(), y.f())
        assert np.array_equal(x.macro(), y.macro())
        assert np.array_equal(x.Q_D.download(), y.Q_D.download())
    plan.close()
    widths[0] += 1
    need = account(widths, height, 3)
    assert need > cap
    over = UGKSim(cases.cfg5_channel(widths=widths, height=height, nc=8, Kn=0.05))
    f0 = [x.f() for x in over.blocks]
    with pytest.raises(L.UGKSError, match=f"needs {need} bytes"):
        run_noalloc(over, "fp64", 1)
    assert all(np.array_equal(x.f(), y) for x, y in zip(over.blocks, f0))
