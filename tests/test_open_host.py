"""What opening a case allocates, on a HIP runtime without a GPU (_fakehip)."""
import pytest

from _fakehip import run

KINDS = ["precision=M.FP64, heat_transfer=False", "precision=M.FP64", "precision=M.FP32, fused=True"]


@pytest.mark.parametrize("kind", KINDS)
def test_tiles_are_built_by_the_first_init(kind, tmp_path):
    """A small case that is opened and not run (its lattice or fields written, say) does not wait
    for tile tables; the first init builds them, the next one keeps them."""
    print(run(tmp_path, """
import os
n = []
for tiles in ("0", ""):
    os.environ["MPLB_TILES"] = tiles
    if not tiles:
        del os.environ["MPLB_TILES"]
    before = live.value
    c = M.Case(make_case_dir(d2(nx=128, ny=128, btype=3)), device=0, %s)
    opened = live.value - before
    for name in ("rho", "T"):
        c.set(name, np.ones(c.N))
    c.init()
    inited = live.value - before
    c.init()
    c.step(3)
    assert live.value - before == inited
    c.close()
    assert live.value == before
    n.append((opened, inited))
assert n[0][0] == n[0][1] == n[1][0] < n[1][1], n
""" % kind))


def test_isothermal_tiles_keep_no_second_temperature_and_heat_source(tmp_path):
    """Second copies are for the fields a launch writes: five of them beside the three tables
    without heat transfer, all seven with it."""
    print(run(tmp_path, """
for ht, extra in ((False, 3 + 5), (True, 3 + 7)):
    c = M.Case(make_case_dir(d2(nx=128, ny=128, btype=3)), device=0, heat_transfer=ht)
    opened = live.value
    for name in ("rho", "T"):
        c.set(name, np.ones(c.N))
    c.init()
    assert live.value - opened == extra, (ht, live.value - opened)
    c.step(9)
    c.close()
"""))
