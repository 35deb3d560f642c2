"""Fully periodic isothermal D3Q15 boxes of whole 32-wide columns and more than 2^19 nodes run
in one pass over the populations in the per-routine arithmetic: the fields follow the oracle
to the parity mode's 1e-12 over one step, over several, and after a read-back, with and
without surface tension and gravity, on a box whose y and z do not divide the columns and
chunks.  In FP32 the same kernel follows the FP64 run to FP32 rounding."""
import pytest

import multiphaselb_amd as M
from _cases import max_rel, pair, sphere_fields
from test_gpu_fused import rel
from test_gpu_parity import TC, TOL, d3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [{}, dict(f_st=1, f_kappa=0.3, g=(1e-6, 0.0, -2e-6))], ids=["plain", "surface-gravity"])
@pytest.mark.parametrize("box", [(96, 75, 74), (32, 129, 130)])
def test_one_pass_over_the_populations_follows_the_oracle(box, extra):
    print("box", box, extra, flush=True)
    spec = d3(nx=box[0], ny=box[1], nz=box[2], btype=5, **extra)
    fields = sphere_fields(spec, seed=3, T=0.85 * TC, r_in=0.03, r_out=0.16, radius=10.0)
    c, o = pair(spec, fields, precision=M.FP64, ht=False)
    s, _ = pair(spec, fields, precision=M.FP32, ht=False)
    done, _, kern = c.time_steps(1)
    assert done == 1 and set(kern) == {"collide"}, kern
    o.run(1)
    for steps in (0, 5):
        assert c.step(steps) == steps
        o.run(steps)
        for f in ("rho", "U", "f", "Fi", "Ft"):
            assert max_rel(c.get(f), o.get(f)) <= TOL, f
    assert s.step(6) == 6
    assert rel(s.get("rho"), o.get("rho")) < 2e-5 and rel(s.get("f"), o.get("f")) < 2e-5
