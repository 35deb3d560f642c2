"""Nodes inside a box that carry a boundary condition or have odd links, in the fused kernels:
the 2D closed box whose Y1 list lies inside it (Ny a multiple of Nx) against the oracle, and
a lattice read from files with a plate in the middle (links cut, its nodes listed) against
the FP64 per-routine arithmetic.  Tiles, passes and the populations that are read back all
apply them.  Bar: the fused kernels' FP32 bound (2e-5 on rho, T, f and g)."""
import os

import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import make_case_dir, pair, sphere_fields
from multiphaselb_amd.casefiles import BC
from test_gpu_fused import rel
from test_gpu_parity import TC, d2

pytestmark = pytest.mark.gpu

ALL = {p: BC("bounceBack") for p in ("X0", "X1", "Y0", "Y1")}
C9 = np.array([(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)])
PLANS = ["0", "7,6,1,2"]


def check(c, ref, fields):
    for f in fields:
        assert rel(c.get(f), ref.get(f)) < 2e-5, f
    assert np.max(np.abs(c.get("U") - ref.get("U"))) < 2e-2 * np.max(np.abs(ref.get("U")))


@pytest.mark.parametrize("ht", [False, True], ids=["nht", "thermal"])
@pytest.mark.parametrize("plan", PLANS)
def test_list_inside_a_closed_box(plan, ht, monkeypatch):
    monkeypatch.setenv("MPLB_TILES", plan)
    spec = d2(nx=20, ny=40, btype=0, write_interval=40, f_bc=ALL, g_bc=ALL)
    fields = sphere_fields(spec, T=0.85 * TC, r_in=0.16, r_out=0.03, radius=5.0, seed=7)
    c, o = pair(spec, fields, precision=M.FP32, ht=ht, fused=True)
    assert c.get_info().fused_active == 1
    assert c.step(60) == o.run(60) == 60
    check(c, o, ("rho", "T", "f") + (("g",) if ht else ()))


def plate_case(nx, ny):
    """A periodicX box as lattice files, rows 10 and 11 cut from each other over columns 6 to
    12 and those nodes listed as X0."""
    spec = d2(nx=nx, ny=ny, btype=1, write_interval=1000, f_bc=ALL, g_bc=ALL)
    d = make_case_dir(spec)
    h = M.Case(d, device=-1)
    nb = h.neighbours().copy()
    lists = h.boundaries()
    h.write_lattice(d)
    h.close()
    j, i = np.divmod(np.arange(nx * ny), nx)
    plate = (i >= 6) & (i <= 12) & ((j == 10) | (j == 11))
    for q in range(9):
        up = nb[:, q]
        cut = plate & (up >= 0) & plate[np.maximum(up, 0)] & (C9[q, 1] != 0)
        nb[cut, q] = -1
    base = os.path.join(d, "processor0", "lattice")
    with open(os.path.join(base, "neighbours"), "w") as fh:
        fh.write("%d 2 9\n" % (nx * ny) + "\n".join(" ".join(map(str, r)) for r in nb) + "\n")
    with open(os.path.join(base, "boundary"), "w") as fh:
        fh.write("%d\n" % len(lists))
        for name, ids in lists:
            ids = np.flatnonzero(plate) if name == "X0" else [] if name == "X1" else ids
            fh.write("%s\n%d\n%s\n" % (name, len(ids), "\n".join(map(str, ids))))
    return spec, d


@pytest.mark.parametrize("plan", PLANS)
def test_plate_inside_a_lattice_from_files(plan, monkeypatch):
    spec, d = plate_case(24, 22)
    rho, U, T = sphere_fields(spec, T=0.85 * TC, r_in=0.16, r_out=0.03, radius=5.0, seed=3)
    got = []
    for fused in (True, False):
        monkeypatch.setenv("MPLB_TILES", plan if fused else "0")
        c = M.Case(d, precision=M.FP32 if fused else M.FP64, fused=fused)
        assert c.get_info().fused_active == int(fused)
        for name, v in (("rho", rho), ("U", U), ("T", T)):
            c.set(name, v)
        c.init()
        assert c.step(60) == 60
        got.append(c)
    check(got[0], got[1], ("rho", "T", "f", "g"))
