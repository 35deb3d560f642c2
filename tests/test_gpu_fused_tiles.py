"""Small D2Q9 lattices advance several fused steps per launch in overlapping tiles
(k_fused_tile).  Whatever the block and the steps per launch, the fields follow the FP64
oracle to the fused kernels' FP32 bar (2e-5 on rho, T and f) and the pass kernels to FP32
rounding (1e-5, ten times that with FP16 storage, where a rounding difference can change a
stored value).  How a run is cut into launches, write steps and read-backs changes
nothing: bit for bit.  Blocks that do not divide the box, single nodes, blocks as wide as
the box (the halo wraps onto itself), walls inside the halo, one and all sizes of
workgroup."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import pair, sphere_fields
from test_gpu_fused import rel
from test_gpu_parity import CASES

pytestmark = pytest.mark.gpu

PLANS = {
    "d2q9_droplet_nht": ["8,8,1,2", "5,7,1,3", "1,1,1,4", "20,19,1,2"],
    "d2q9_bubble_thermal": ["6,5,1,2", "24,1,1,1", "13,13,1,2"],
    "d2q9_column_fixedT": ["5,7,1,3", "2,9,1,2", "5,1,1,8"],
    "d2q9_column_liTempMRT": ["5,16,1,4", "5,5,1,1"],
    "d2q9_surface_tension": ["6,6,1,2", "24,2,1,1"],
    "d2q9_carnahan_starling_keys_first": ["7,7,1,3"],
    "d2q9_column_two_frdt": ["5,8,1,5", "3,4,1,1"],
}


@pytest.mark.parametrize("name,plan", [(n, p) for n, v in PLANS.items() for p in v])
def test_tiles_follow_the_oracle_and_the_passes(name, plan, monkeypatch):
    spec, fk, ht, frozen, steps = CASES[name]
    print("case", name, plan, flush=True)
    fields = sphere_fields(spec, seed=7, **fk)
    monkeypatch.setenv("MPLB_TILES", plan)
    a, o = pair(spec, fields, precision=M.FP32, ht=ht, fused=True)
    done, _, kern = a.time_steps(3)
    assert done == 3 and set(kern) == {"fused"}, kern
    assert a.step(steps - 3) == steps - 3
    monkeypatch.setenv("MPLB_TILES", "0")
    b, _ = pair(spec, fields, precision=M.FP32, ht=ht, fused=True)
    assert b.step(steps) == steps
    o.run(steps)
    for f in ("rho", "T", "f"):
        assert rel(a.get(f), o.get(f)) < 2e-5, f
        assert rel(a.get(f), b.get(f)) < 1e-5, f
    assert np.max(np.abs(a.get("U") - b.get("U"))) < 1e-6


@pytest.mark.parametrize("precision", [M.FP32, M.FP16S, M.FP16N], ids=["fp32", "fp16s", "fp16n"])
@pytest.mark.parametrize("name,plan", [("d2q9_droplet_nht", "8,8,1,4"), ("d2q9_bubble_thermal", "13,13,1,2"),
                                       ("d2q9_column_liTempMRT", "5,16,1,4"), ("d2q9_column_two_frdt", "5,8,1,5")])
def test_launches_leave_no_trace(name, plan, precision, monkeypatch):
    spec, fk, ht, frozen, steps = CASES[name]
    print("case", name, plan, precision, flush=True)
    fields = sphere_fields(spec, seed=5, **fk)
    monkeypatch.setenv("MPLB_TILES", plan)
    a, _ = pair(spec, fields, precision=precision, ht=ht, fused=True)
    b, _ = pair(spec, fields, precision=precision, ht=ht, fused=True)
    monkeypatch.setenv("MPLB_TILES", "0")
    p, _ = pair(spec, fields, precision=precision, ht=ht, fused=True)
    assert a.step(31) == b.step(1) + b.step(2) + b.step(7) + b.step(11) + (b.get("rho") is None) + b.step(10) == 31
    p.step(31)
    names = ("rho", "U", "f") + (("T", "g", "ss") if ht else ())
    for f in names:
        assert np.array_equal(a.get(f), b.get(f)), f
    for f in ("rho", "f"):
        assert rel(a.get(f), p.get(f)) < (1e-5 if precision == M.FP32 else 1e-4), f
