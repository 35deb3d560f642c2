"""Boundary lists that leave the surface of a built box.  The 2D closed box fills its Y1 list
with j + (Nx - 1) Ny (genericBoundary.c:6-49): for Ny a multiple of Nx every one of these
nodes is inside the box, for other ratios some are.  bounceBack acts on them (it averages the
axis pairs of nodes that have all links), in the fused passes as in tiles, against the oracle
at the FP64 mode's 1e-12; in FP32 the two share their arithmetic and agree bit for bit."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import max_rel, pair, sphere_fields
from multiphaselb_amd.casefiles import BC
from test_gpu_parity import TC, TOL, d2

pytestmark = pytest.mark.gpu

ALL = {p: BC("bounceBack") for p in ("X0", "X1", "Y0", "Y1")}
WALLS = {"X0": BC("periodic"), "X1": BC("periodic"), "Y0": BC("bounceBack"), "Y1": BC("bounceBack")}
BOXES = {"20x40": (20, 40, ALL), "13x39": (13, 39, ALL), "20x30_open_sides": (20, 30, WALLS)}


def case(name, precision, ht):
    nx, ny, bc = BOXES[name]
    spec = d2(nx=nx, ny=ny, btype=0, write_interval=40, f_bc=bc, g_bc=bc)
    fields = sphere_fields(spec, T=0.85 * TC, r_in=0.16, r_out=0.03, radius=5.0, seed=7)
    return pair(spec, fields, precision=precision, ht=ht)


@pytest.mark.parametrize("ht", [False, True], ids=["nht", "thermal"])
@pytest.mark.parametrize("name", list(BOXES))
def test_lists_inside_the_box_are_applied(name, ht, monkeypatch):
    print("case", name, ht, flush=True)
    for tiles in ("0", "6,7,1,2"):
        monkeypatch.setenv("MPLB_TILES", tiles)
        c, o = case(name, M.FP64, ht)
        assert c.step(60) == o.run(60) == 60
        for f in ("rho", "U", "T", "f", "Fi", "Ft") + (("g", "ss") if ht else ()):
            assert max_rel(c.get(f), o.get(f)) <= TOL, (tiles, f)


def test_fp32_passes_equal_tiles(monkeypatch):
    got = []
    for tiles in ("0", "6,7,1,2"):
        monkeypatch.setenv("MPLB_TILES", tiles)
        c, _ = case("20x40", M.FP32, True)
        c.step(60)
        got.append({f: c.get(f) for f in ("rho", "U", "T", "f", "g")})
    for f in got[0]:
        assert np.array_equal(got[0][f], got[1][f]), f
