"""bench.py's per-step traffic and instruction totals against the counter tables they come from.

A step is every launch between two time steps: the walls are a launch of their
own behind the flux pass where they do not go beside the face states (more than
4096 workgroups together, as on the 64-case batch), so k_wallS counts twice there.
"""
import os

import pytest

import bench

PROFILES = os.path.join(bench.ROOT, "profiles")
# wall faces and workgroups of 256 interior faces
WALLS_BEHIND = {"batch64_cavities_weno5": True, "cavity_2x2x128sq_nc32_weno5": False}


def rows(table, tag):
    """kernel -> (launches per step, total per step) by the table's own column names"""
    out, names = {}, None
    with open(os.path.join(PROFILES, table)) as fh:
        for line in fh:
            if line.startswith("# kernel "):
                names = line[1:].split()
            elif not line.startswith("#") and line.split()[1] == tag:
                r = dict(zip(names, line.split()))
                total = next(v for k, v in r.items() if k in ("hbm_bytes_per_step", "valu_insts_per_step"))
                out[r["kernel"]] = (int(r["launches_per_step"]), float(total))
    return out


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("workload", list(WALLS_BEHIND))
@pytest.mark.parametrize("table", ["hbm_traffic", "valu"])
def test_totals_are_those_of_every_launch_of_a_step(table, workload, precision):
    fname, tag = f"{table}_per_kernel_{workload}.txt", f"{workload}_{precision}"
    r = rows(fname, tag)
    want = {"k_faceA": 1, "k_wallS": 2 if WALLS_BEHIND[workload] else 1, "k_faceC": 1, "k_update": 1, "k_end": 1}
    assert {k: n for k, (n, _) in r.items()} == want
    per_step, commit = bench.read_profile_table(fname, tag)
    assert commit
    assert per_step == {k: total for k, (_, total) in r.items()}


def test_unknown_workload_has_no_totals():
    assert bench.read_profile_table("valu_per_kernel_batch64_cavities_weno5.txt", "no_such_workload")[0] == {}
    assert bench.read_profile_table("no_such_table.txt", "any") == ({}, None)
