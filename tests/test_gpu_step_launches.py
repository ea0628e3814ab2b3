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
