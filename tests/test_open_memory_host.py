"""Opening a case when memory is short, on a HIP runtime without a GPU (_fakehip): what only
makes steps faster (tiles) is left out, and the case opens."""
import pytest

from _fakehip import run

SETUP = """
import os
def opened(tiles=True, **kw):
    os.environ.pop("MPLB_TILES", None)
    if not tiles:
        os.environ["MPLB_TILES"] = "0"
    peak.value = live.value
    c = M.Case(make_case_dir(d2(nx=128, ny=128, btype=3)), device=0, **kw)
    for name in ("rho", "T"):
        c.set(name, np.ones(c.N))
    c.init()
    c.step(3)
    c.close()
    assert live.value == 0
    return peak.value
"""
KINDS = ["precision=M.FP64, heat_transfer=False", "precision=M.FP64", "precision=M.FP32, fused=True"]


@pytest.mark.parametrize("kind", KINDS)
def test_no_device_memory_for_tiles(kind, tmp_path):
    print(run(tmp_path, SETUP + """
plain, tiled = opened(False, %s), opened(%s)
assert tiled > plain
for most.value in range(plain, tiled):
    opened(%s)
""" % (kind, kind, kind)))


@pytest.mark.parametrize("kind", KINDS)
def test_no_host_memory_for_tile_tables(kind, tmp_path):
    print(run(tmp_path, SETUP + """
opened(%s)
for limit in (1 << 20, 3 << 18):
    new_limit.value = limit
    opened(%s)
    new_limit.value = 0
""" % (kind, kind)))


def test_no_device_memory_for_the_passes(tmp_path):
    """The per-node list numbers and the new temperature of the fused passes: without them the
    case runs one kernel per routine."""
    print(run(tmp_path, """
from multiphaselb_amd.casefiles import BC
spec = d2(nx=5, ny=40, btype=1, f_bc={"Y0": BC("bounceBack"), "Y1": BC("bounceBack")},
          g_bc={"Y0": BC("fixedT", (0.95 * TC,)), "Y1": BC("fixedT", (0.8 * TC,))})
M.Case(make_case_dir(spec), device=0).close()
for most.value in range(peak.value - 3, peak.value + 1):
    c = M.Case(make_case_dir(spec), device=0)
    for name in ("rho", "T"):
        c.set(name, np.ones(c.N))
    c.init()
    assert c.step(3) == 3
    c.close()
    assert live.value == 0
"""))
