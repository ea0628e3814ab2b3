"""Every field a step leaves, ghost cells and per-velocity fluxes included, on
the routes a step can take: joint launches against launches of their own, and
face fluxes stored through the caches against streamed ones.  The routes run
the same code per face, cell and case, so every field is the same to the last
bit, in mixed mode in the FP32 state the step advances.
"""
import copy

import numpy as np
import pytest

from pyugks_amd import bc as bcd
from pyugks_amd import cases

pytestmark = pytest.mark.gpu


def open_cavity(k, method, across):
    """Inflow and outflow (whose ghosts are built from the cell's new state) across two opposite faces."""
    g = cases.cavity(7 + k % 3, ("NC", 8), method, 0.05 * (1 + k % 4), n_cells_j=6, rho_perturb=0.01)
    inflow, outflow = bcd.InflowBC(D=1.1, T=1.05), bcd.OutflowBC(P=0.9, D=1.0)
    wall, moving = bcd.DiffuseBC(D=1.0, T=0.9), bcd.DiffuseBC(D=1.0, T=1.0, U=0.1)
    g.blocks[0].bc_list = [outflow, wall, inflow, moving] if across == "NS" else [wall, outflow, moving, inflow]
    return g


def channel(k, reflect):
    return cases.cfg5_channel(widths=[9, 12 + k % 3], height=6, nc=8, Kn=0.05 * (1 + k % 4), reflect_type=reflect,
                              alpha_n=0.8, alpha_t=0.7)


GROUPS = {
    "open_NS": lambda: [open_cavity(k, "WENO5", "NS") for k in range(3)],
    "open_EW": lambda: [open_cavity(k, "vanLeer", "EW") for k in range(3)],
    "adsorbing_diffuse": lambda: [channel(k, "D") for k in range(2)],
    "adsorbing_specular": lambda: [channel(k, "S") for k in range(2)],
    "adsorbing_CL": lambda: [channel(k, "CL") for k in range(2)],
    "bent_joined": lambda: [cases.curvilinear(cases.cavity(14, ("NC", 8), "minmod", 0.1, nb=(2, 1), n_cells_j=9), 0.05)],
    # 110 x 2 x (21 to 23) wall faces: more than go beside the face states
    "many_adsorbing": lambda: [channel(k, "D") for k in range(110)],
}
FIELDS = ("macro_D", "Q_D", "residual_D", "time_step_D", "flux_macro_S_D", "flux_macro_W_D", "wall_prop_D",
          "wall_cover_D", "wall_fluxes_D", "flag_D")
STATE = {"fp64": ("f_D", "flux_f_S_D", "flux_f_W_D"), "mixed": ("f32_D", "fluxS32_D", "fluxW32_D")}


def assert_same_fields(a, b, precision):
    for name in STATE[precision] + FIELDS:
        x, y = getattr(a, name).download(), getattr(b, name).download()
        assert np.array_equal(x, y), name
        if name in STATE[precision] or name in ("macro_D", "Q_D"):
            assert np.isfinite(x).all(), name


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("group", list(GROUPS))
def test_joint_and_separate_launches_leave_the_same_fields(hip, group, precision):
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] step fields {group} {precision}", flush=True)
    gs = GROUPS[group]()
    joint, apart = ([UGKSim(copy.deepcopy(g)) for g in gs] for _ in range(2))
    pj, pa = StepPlan(joint, precision), StepPlan(apart, precision)
    start = pj.f64(joint[0].blocks[0])
    for _ in range(2):
        pj.run(2)
        pa.run_timed(2)
        for x, y in zip(pj.states(), pa.states()):
            assert (x.dt, x.time, x.step) == (y.dt, y.time, y.step)
        for a, b in zip(joint, apart):
            for x, y in zip(a.blocks, b.blocks):
                assert_same_fields(x, y, precision)
    assert not np.array_equal(pj.f64(joint[0].blocks[0]), start)
    pj.close()
    pa.close()


@pytest.mark.parametrize("precision,copies", [("fp64", 3), ("mixed", 6)])
@pytest.mark.parametrize("method", ["WENO5", "vanLeer", "minmod"])
@pytest.mark.parametrize("bent", [False, True])
def test_kept_and_streamed_fluxes_leave_the_same_fields(hip, bent, method, precision, copies):
    """One case's face fluxes (56 MB, 28 in mixed mode) stay in the caches, those of a plan of copies (more than
    144 MB) are streamed past them."""
    from pyugks_amd.fused import StepPlan
    from pyugks_amd.sim import UGKSim
    print(f"[gpu] flux store fields {method} bent={bent} {precision}", flush=True)
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
        assert_same_fields(one.blocks[0], sim.blocks[0], precision)
    po.close()
    pm.close()
