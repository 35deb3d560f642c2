"""The fused pass kernels index nodes in 32 bits up to 2^30 of them and in 64 beyond.  Both
forms follow each other to FP32 rounding (1e-5, ten times that with FP16 storage, where a
rounding difference can change a stored value), on boxes whose faces wrap, on walls read
through the neighbour table, and on nodes that end inside a workgroup."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import pair, sphere_fields
from test_gpu_fused import rel
from test_gpu_parity import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [M.FP32, M.FP16S, M.FP16N], ids=["fp32", "fp16s", "fp16n"])
@pytest.mark.parametrize("name", ["d2q9_droplet_nht", "d2q9_column_fixedT", "d2q9_surface_tension", "d3q15_bubble_nht",
                                  "d3q15_bubble_thermal", "d3q15_thermal_column", "d3q15_surface_tension"])
def test_both_index_widths_agree(name, precision, monkeypatch):
    spec, fk, ht, frozen, steps = CASES[name]
    print("case", name, precision, flush=True)
    fields = sphere_fields(spec, seed=3, **fk)
    monkeypatch.setenv("MPLB_TILES", "0")
    monkeypatch.setenv("MPLB_FUSED_KERNEL", "twopass")
    a, _ = pair(spec, fields, precision=precision, ht=ht, fused=True)
    monkeypatch.setenv("MPLB_INDEX64", "1")
    b, _ = pair(spec, fields, precision=precision, ht=ht, fused=True)
    assert a.step(30) == b.step(30) == 30
    for f in ("rho", "f") + (("T", "g") if ht else ()):
        assert rel(a.get(f), b.get(f)) < (1e-5 if precision == M.FP32 else 1e-4), f
    assert np.max(np.abs(a.get("U") - b.get("U"))) < (1e-6 if precision == M.FP32 else 1e-5)
