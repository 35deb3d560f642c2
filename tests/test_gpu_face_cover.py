"""The faces that the fused kernels read through the neighbour table are the cheapest set
that covers every node with an odd link or a boundary condition; all other surface nodes
use the computed wrap.  Boxes whose covers differ (walls on one axis, four odd corners,
closed boxes), a few nodes wider than a wavefront, against the FP64 oracle.  Tolerance: the
fused FP32 kernels' own bound against the oracle over a comparable number of steps."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import pair, sphere_fields
from multiphaselb_amd.casefiles import BC
from test_gpu_fused import rel
from test_gpu_parity import TC, d2, d3

pytestmark = pytest.mark.gpu

WALL_F = {"Z0": BC("bounceBack"), "Z1": BC("bounceBack")}
CASES = {
    "column3d": (d3(nx=67, ny=5, nz=18, btype=3, g=(0.0, 0.0, -1e-6), f_bc=WALL_F,
                    g_bc={"Z0": BC("fixedRandomT", (0.95 * TC,), pert=0.5, duration=30),
                          "Z1": BC("fixedT", (0.8 * TC,))}), dict(radius=0, column=6.0)),
    "column2d": (d2(nx=67, ny=21, btype=1, f_bc={"Y0": BC("bounceBack"), "Y1": BC("bounceBack")},
                    g_bc={"Y0": BC("fixedT", (0.95 * TC,)), "Y1": BC("fixedT", (0.8 * TC,))}),
                 dict(radius=0, column=8.0)),
    "periodic2d": (d2(nx=67, ny=19, btype=3), dict(radius=5.0)),
    "closed3d": (d3(nx=66, ny=6, nz=7, btype=0, f_bc={p: BC("bounceBack") for p in ("X0", "X1", "Y0", "Y1", "Z0", "Z1")},
                    g_bc={p: BC("bounceBack") for p in ("X0", "X1", "Y0", "Y1", "Z0", "Z1")}), dict(radius=2.5)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_fused_boxes_follow_the_oracle_whatever_faces_are_read_through_the_table(name):
    spec, fk = CASES[name]
    fields = sphere_fields(spec, seed=7, T=0.85 * TC, r_in=0.16, r_out=0.03, **fk)
    c, o = pair(spec, fields, precision=M.FP32, fused=True)
    assert c.get_info().fused_active == 1
    assert c.step(60) == 60
    o.run(60)
    for f in ("rho", "T", "f", "g"):
        assert rel(c.get(f), o.get(f)) < 2e-5, f
    assert np.max(np.abs(c.get("U") - o.get("U"))) < 2e-2 * np.max(np.abs(o.get("U")))
