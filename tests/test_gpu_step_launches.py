"""The step as it runs (wall faces beside the face states, ghost cells beside
the time step, whose last workgroup sets the cases' dt) against the same parts
in launches of their own, as the per-kernel timer runs them.  Both run the same
code per face, cell and case, and a maximum does not depend on its order, so
every result is the same to the last bit, step after step.  The large batch has
more cases than the workgroup that sets dt has threads, and more wall faces
than go beside the face states.
"""
import copy

import numpy as np
import pytest

from pyugks_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("ncases", [1, 300])
def test_joint_launches_are_bitwise_the_separate_ones(hip, ncases, precision):
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] step launches {ncases} cases {precision}", flush=True)
    gs = [cases.cavity(5 + k % 2, ("NC", 8), "vanLeer", 0.05 * (1 + k % 7), n_cells_j=4, rho_perturb=0.01 * (1 + k % 3))
          for k in range(ncases)]
    joint, apart = ([UGKSim(copy.deepcopy(g)) for g in gs] for _ in range(2))
    pj, pa = StepPlan(joint, precision), StepPlan(apart, precision)
    for _ in range(3):
        pj.run(2)
        pa.run_timed(2)
        for a, b in zip(pj.states(), pa.states()):
            assert (a.dt, a.time, a.step) == (b.dt, b.time, b.step)
    assert len({s.gdata.dt for s in joint}) == len({s.gdata.dt for s in apart}) >= min(ncases, 2)
    for a, b in zip(joint, apart):
        for name in ("f_D", "macro_D", "Q_D", "wall_fluxes_D"):
            if hasattr(a.blocks[0], name):
                x, y = getattr(a.blocks[0], name).download(), getattr(b.blocks[0], name).download()
                assert np.array_equal(x, y), name
    pj.close()
    pa.close()


@pytest.mark.parametrize("precision,copies", [("fp64", 3), ("mixed", 6)])
@pytest.mark.parametrize("method", ["WENO5", "vanLeer", "minmod"])
@pytest.mark.parametrize("bent", [False, True])
def test_kept_and_streamed_fluxes_are_bitwise_alike(hip, bent, method, precision, copies):
    """A case alone keeps its 56 MB (28 in mixed mode) of face fluxes in the
    caches; a plan of copies has more than 144 MB and streams them.  The stores
    differ, the values do not."""
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] flux stores {method} bent={bent} {precision}", flush=True)
    g = cases.cavity(40, ("NC", 32), method, 0.05, n_cells_j=41, rho_perturb=0.01)
    if bent:
        cases.curvilinear(g, 0.05)
    one, many = UGKSim(copy.deepcopy(g)), [UGKSim(copy.deepcopy(g)) for _ in range(copies)]
    pairs = 2 * 40 * 41 * 33 * 33 * (16 if precision == "fp64" else 8)
    assert pairs < 144 << 20 < copies * pairs * 39 / 40
    po, pm = StepPlan(one, precision), StepPlan(many, precision)
    po.run(3)
    pm.run(3)
    for sim in (many[0], many[-1]):
        for name in ("macro_D", "Q_D", "wall_fluxes_D"):
            assert np.array_equal(getattr(one.blocks[0], name).download(), getattr(sim.blocks[0], name).download()), name
    po.close()
    pm.close()
