"""Large fields move through a ring of pinned buffers (2 MiB chunks, eight of them): what
is set comes back exactly (FP64) or as its FP32 rounding, for one, three and Q values per
node, below and above the size where the ring takes over (4 MiB of doubles), with whole
and ragged last chunks and more chunks than buffers."""
import numpy as np
import pytest

import multiphaselb_amd as M
from _cases import make_case_dir
from test_gpu_parity import d2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [M.FP64, M.FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny", [(723, 725), (1024, 512), (1024, 1024), (1500, 1409)])
def test_large_fields_round_trip(nx, ny, precision):
    c = M.Case(make_case_dir(d2(nx=nx, ny=ny, btype=3)), precision=precision, heat_transfer=False)
    rng = np.random.default_rng(nx)
    for name in ("rho", "U", "f"):
        a = rng.standard_normal(c._shape(name))
        c.set(name, a)
        want = a if precision == M.FP64 else a.astype(np.float32).astype(np.float64)
        assert np.array_equal(c.get(name), want), name
    c.close()
