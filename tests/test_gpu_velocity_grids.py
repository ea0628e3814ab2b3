"""The fused step on velocity sets at the edges of the flux pass's tables.

Its per-face tables are built in one go up to 32 values per axis and in two
beyond, and a velocity set that is no tensor grid (here a shuffled one) or a
face normal off the axes takes the general loop.  FP64 within 1e-12 of the
oracle per step, mixed within 1e-5 in rho, U, T, the bounds of
test_gpu_fused.py.
"""
import copy

import numpy as np
import pytest

from helpers import SCALE_FLOOR, field_errors, rel_err
from pyugks_amd import cases

pytestmark = pytest.mark.gpu


def grid(kind, method):
    g = cases.cavity(9, ("NC", 12), method, 0.05, n_cells_j=7, rho_perturb=0.01)
    if kind == "gh31":
        cases.gauss_hermite(g, 31)
    elif kind == "gh32":
        cases.gauss_hermite(g, 32)
    elif kind == "nc5x61":
        g.u_num, g.v_num = 4, 60
    elif kind == "nc41x13":
        g.u_num, g.v_num = 40, 12
    elif kind == "nc61x33":
        g.u_num, g.v_num = 60, 32
    elif kind == "shuffled":
        h = copy.deepcopy(g)
        h.init_ref_values()
        order = np.random.default_rng(5).permutation(h.Nv)
        g.quad_type, g.quad, g.weight = "defined", h.quad[order], h.weight[order]
    elif kind == "bent":
        cases.curvilinear(g, 0.05)
    return g


@pytest.mark.parametrize("method", ["WENO5", "vanLeer", "minmod"])
@pytest.mark.parametrize("kind", ["gh31", "gh32", "nc5x61", "nc41x13", "nc61x33", "shuffled", "bent"])
def test_velocity_grids_match_oracle(hip, kind, method):
    from oracle import OracleSim
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] velocity grid {kind} {method}", flush=True)
    g = grid(kind, method)
    ora = OracleSim(copy.deepcopy(g), threads=4)
    ora.run(3)
    for precision in ("fp64", "mixed"):
        gpu = UGKSim(copy.deepcopy(g))
        plan = StepPlan(gpu, precision)
        plan.run(3)
        b, o = gpu.blocks[0], ora.blocks[0]
        if precision == "fp64":
            assert rel_err(b.f_D.download(), o["f"]) <= 3e-12
            assert rel_err(b.macro_D.download(), o["macro"]) <= 3e-12
            assert rel_err(b.Q_D.download(), o["Q"], SCALE_FLOOR["Q"]) <= 3e-12
            assert rel_err(b.wall_fluxes_D.download(), o["wall_fluxes"]) <= 3e-12
        else:
            e = field_errors([b.macro_D.download()], [o["macro"]])
            assert max(e[k] for k in ("rho_linf", "U_linf", "T_linf")) <= 1e-5, e
        plan.close()
