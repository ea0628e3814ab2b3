"""One plan over cases with different reconstructions and velocity sets.

Its face passes read the method from each block instead of being built for one,
and their tables are sized by the longest velocity axis of any block, tensor
grid or not.  FP64 within 1e-12 of the oracle per step and of each case in a plan
of its own; mixed within 1e-5 in rho, U, T: the bounds of test_gpu_fused.py.
"""
import copy

import numpy as np
import pytest

from helpers import SCALE_FLOOR, field_errors, rel_err
from pyugks_amd import cases

pytestmark = pytest.mark.gpu

STEPS = 3


def shuffled(g):
    """The same velocities in another order: a velocity set that is no tensor grid."""
    h = copy.deepcopy(g)
    h.init_ref_values()
    order = np.random.default_rng(5).permutation(h.Nv)
    g.quad_type, g.quad, g.weight = "defined", h.quad[order], h.weight[order]
    return g


def case(method, n, nj, nc, bend=False, shuffle=False, nb=(1, 1)):
    g = cases.cavity(n, ("NC", nc), method, 0.05, n_cells_j=nj, nb=nb, rho_perturb=0.01)
    if bend:
        cases.curvilinear(g, 0.05)
    return shuffled(g) if shuffle else g


PLANS = {
    "axis_aligned": [("WENO5", 9, 7, 12), ("vanLeer", 8, 10, 16), ("minmod", 11, 6, 8)],
    "bent": [("minmod", 9, 7, 8, True), ("WENO5", 10, 9, 16, True, False, (2, 1)), ("vanLeer", 6, 8, 12, True)],
    "with_a_set_that_is_no_tensor_grid": [("vanLeer", 9, 7, 12, False, True), ("WENO5", 8, 8, 36),
                                          ("minmod", 7, 9, 8, True), ("WENO5", 7, 6, 8, False, True)],
    "one_velocity_a_lane": [("WENO5", 5, 4, 4), ("minmod", 4, 5, 4, True)],
}


@pytest.mark.parametrize("name", list(PLANS))
def test_each_case_steps_as_the_oracle_and_as_alone(hip, name):
    from oracle import OracleSim
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] plan of several limiters {name}", flush=True)
    gs = [case(*a) for a in PLANS[name]]
    oracles = [OracleSim(copy.deepcopy(g), threads=4) for g in gs]
    for o in oracles:
        o.run(STEPS)
    for precision in ("fp64", "mixed"):
        sims = [UGKSim(copy.deepcopy(g)) for g in gs]
        plan = StepPlan(sims, precision)
        plan.run(STEPS)
        for k, (sim, ora) in enumerate(zip(sims, oracles)):
            if precision == "mixed":
                e = field_errors([b.macro_D.download() for b in sim.blocks], [o["macro"] for o in ora.blocks])
                assert max(e[q] for q in ("rho_linf", "U_linf", "T_linf")) <= 1e-5, (k, e)
                continue
            alone = UGKSim(copy.deepcopy(gs[k]))
            own = StepPlan(alone, precision)
            own.run(STEPS)
            for b, o, c in zip(sim.blocks, ora.blocks, alone.blocks):
                for field, key in (("f_D", "f"), ("macro_D", "macro"), ("Q_D", "Q"), ("wall_fluxes_D", "wall_fluxes")):
                    x, floor = getattr(b, field).download(), SCALE_FLOOR.get(key, 0.0)
                    assert rel_err(x, o[key], floor) <= STEPS * 1e-12, (k, key)
                    assert rel_err(x, getattr(c, field).download(), floor) <= STEPS * 1e-12, (k, key)
            own.close()
        plan.close()
