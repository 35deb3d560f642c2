"""Small lattices advance several steps per launch in overlapping tiles (k_tile): whatever
the block and the steps per launch, with launches that end short of a whole one, every
field follows the oracle and equals the fused passes' bit for bit (the node arithmetic is
shared).  Blocks that do not divide the box, single nodes, blocks as wide as the box (the
halo wraps onto itself), walls inside the halo.  Bar against the oracle: the FP64 mode's
1e-12."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import max_rel, pair, sphere_fields
from test_gpu_parity import CASES, FIELDS, TOL

pytestmark = pytest.mark.gpu

PLANS = {
    "d2q9_droplet_nht": ["8,8,1,2", "5,7,1,3", "1,1,1,4", "32,1,1,1"],
    "d2q9_bubble_thermal": ["6,5,1,2", "24,1,1,1"],
    "d2q9_column_fixedT": ["5,7,1,3", "2,9,1,2", "5,1,1,8"],
    "d2q9_column_liTempMRT": ["5,16,1,4"],
    "d2q9_surface_tension": ["6,6,1,2", "24,2,1,1"],
    "d2q9_carnahan_starling_keys_first": ["7,7,1,3"],
    "d2q9_column_two_frdt": ["5,8,1,5", "3,4,1,1"],
    "d3q15_bubble_nht": ["3,2,3,1", "2,2,2,1"],
    "d3q15_surface_tension": ["1,2,2,1"],
    "d3q15_thermal_column": ["6,6,1,1"],
    "d3q15_column_frdt_nopert": ["6,3,1,1"],
}


@pytest.mark.parametrize("name,plan", [(n, p) for n, v in PLANS.items() for p in v])
def test_tiles_equal_the_passes_and_follow_the_oracle(name, plan, monkeypatch):
    spec, fk, ht, frozen, steps = CASES[name]
    print("case", name, plan, flush=True)
    fields = sphere_fields(spec, seed=7, **fk)
    monkeypatch.setenv("MPLB_TILES", "0")
    a, o = pair(spec, fields, precision=M.FP64, ht=ht)
    monkeypatch.setenv("MPLB_TILES", plan)
    b, _ = pair(spec, fields, precision=M.FP64, ht=ht)
    # a run of its own length first: write steps and the end of a call cut launches short
    done, _, kern = b.time_steps(7)
    assert done == 7 and set(kern) == {"collide"}, kern
    assert a.step(7) == 7
    assert a.step(steps - 7) == b.step(steps - 7) == steps - 7
    o.run(steps)
    for f in FIELDS:
        if f == "p" and spec.write_interval > steps:
            continue
        x, y = a.get(f), b.get(f)
        assert np.array_equal(x, y), f
        assert max_rel(y, o.get(f)) <= TOL, f
