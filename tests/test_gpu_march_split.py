"""The z-marches split a box into chunks of planes and store the new populations either
non-temporally or not, by the rows' size and the populations' total; whether a box takes
the march or the two passes follows from its size too.  Neither of the first two changes a
node's arithmetic: whatever the number of chunks (one, the default, one per plane) the
fields are equal bit for bit, and boxes on both sides of the store rule (rows that end
inside a 64-byte sector, whole sectors in populations of less and of more than 256 MiB)
follow the two-pass kernels to FP32 rounding, ten times that with FP16 storage, where a
rounding difference can change a stored value."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import make_case_dir, sphere_fields
from test_gpu_fused import rel
from test_gpu_parity import TC, d3

pytestmark = pytest.mark.gpu


def run(spec, precision, thermal, steps):
    c = M.Case(make_case_dir(spec), precision=precision, heat_transfer=thermal, fused=True)
    rho, U, T = sphere_fields(spec, seed=5, T=0.85 * TC, r_in=0.16, r_out=0.03, radius=4.0)
    c.set("rho", rho)
    c.set("U", U)
    c.set("T", T)
    c.init()
    assert c.step(steps) == steps
    return {f: c.get(f) for f in ("rho", "U", "f") + (("T", "g") if thermal else ())}


@pytest.mark.parametrize("precision,thermal,variant", [
    (M.FP32, False, ""), (M.FP32, False, "MPLB_MARCH_LDS"), (M.FP32, False, "MPLB_MARCH_PF"), (M.FP16S, False, ""),
    (M.FP16N, False, ""), (M.FP32, True, "MPLB_THERMAL_MARCH"), (M.FP16N, True, "MPLB_THERMAL_MARCH")])
@pytest.mark.parametrize("box", [(33, 10, 11), (64, 9, 6), (66, 5, 3)])
def test_chunks_leave_the_fields_unchanged(box, precision, thermal, variant, monkeypatch):
    print("box", box, "precision", precision, "thermal", thermal, variant, flush=True)
    spec = d3(nx=box[0], ny=box[1], nz=box[2], btype=5)
    monkeypatch.setenv("MPLB_FUSED_KERNEL", "march")
    if variant:
        monkeypatch.setenv(variant, "1")
    out = []
    for chunks in ("", "1", str(box[2])):
        if chunks:
            monkeypatch.setenv("MPLB_MARCH_CHUNKS", chunks)
        out.append(run(spec, precision, thermal, 6))
    for other in out[1:]:
        for f in out[0]:
            assert np.array_equal(out[0][f], other[f]), f


@pytest.mark.parametrize("precision", [M.FP32, M.FP16S, M.FP16N], ids=["fp32", "fp16s", "fp16n"])
@pytest.mark.parametrize("box", [(97, 10, 11), (64, 9, 6), (192, 160, 160)], ids=["ragged", "small", "large"])
def test_both_kinds_of_stores_follow_the_two_pass_kernels(box, precision, monkeypatch):
    print("box", box, "precision", precision, flush=True)
    spec = d3(nx=box[0], ny=box[1], nz=box[2], btype=5)
    picked = run(spec, precision, False, 6)          # whichever the box's size calls for
    monkeypatch.setenv("MPLB_FUSED_KERNEL", "march")
    one = run(spec, precision, False, 6)
    monkeypatch.setenv("MPLB_FUSED_KERNEL", "twopass")
    two = run(spec, precision, False, 6)
    tol = 1e-5 if precision == M.FP32 else 1e-4
    assert rel(one["rho"], two["rho"]) < tol
    assert rel(one["f"], two["f"]) < tol
    assert np.max(np.abs(one["U"] - two["U"])) < 0.1 * tol
    assert any(all(np.array_equal(picked[f], o[f]) for f in picked) for o in (one, two))
