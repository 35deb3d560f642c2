"""The two-launch network (k_rows: 16 rows per workgroup through every layer; k_weights: all
weight and bias gradients with Adam in the epilogue) at the edges of its tiles: one layer,
narrow and uneven widths, the smallest batch, row counts that leave a partial workgroup,
more iterations than one; and a network too wide for a row workgroup's LDS, which keeps one
launch per product.  Bars: those of the network's own tests against the CPU oracle."""
import os
import sys

import numpy as np
import pytest

import multiphaselb_amd as M

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as MO  # noqa: E402

pytestmark = pytest.mark.gpu

NETS = [([1, 32], 32), ([9, 32, 64, 32], 32), ([32, 96, 32], 96), ([9, 256, 256, 256, 128], 256), ([5, 320, 288], 64),
        ([7, 1024, 512, 64], 32)]


@pytest.mark.parametrize("widths,batch", NETS, ids=["-".join(map(str, w)) for w, _ in NETS])
def test_network_at_tile_edges(widths, batch):
    rng = np.random.default_rng(len(widths) * batch)
    net = M.Mlp(widths, batch)
    parts = []
    for a, b in zip(widths[:-1], widths[1:]):
        lim = np.sqrt(6.0 / (a + b))
        parts += [rng.uniform(-lim, lim, a * b), rng.uniform(-0.1, 0.1, b)]
    p = np.concatenate(parts).astype(np.float32)
    net.set_params(p)
    x = rng.uniform(-1, 1, (batch, widths[0])).astype(np.float32)
    t = rng.uniform(-1, 1, (batch, widths[-1])).astype(np.float32)
    for rows in (1, batch - 15, batch, 2 * batch + 17):
        xr = rng.uniform(-1, 1, (rows, widths[0])).astype(np.float32)
        y = net.forward(xr)
        ref = MO.forward(p, widths, xr.astype(np.float64))[2]
        assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref), rows
    loss, g = net.gradient(x, t)
    l16, g16 = MO.loss_grad(p, widths, x.astype(np.float64), t.astype(np.float64), bf16_ops=True)
    assert abs(loss - l16) < 1e-4 * l16
    assert np.linalg.norm(g - g16) < 5e-3 * np.linalg.norm(g16)
    # two iterations: the first is Adam's closed form on that gradient, the second moves on
    # from the refreshed BF16 copies
    idx = np.tile(np.arange(batch, dtype=np.int32), 2)
    net.train(x, t, idx[:batch], lr=1e-3)
    p1 = net.get_params()
    ref1, _, _ = MO.adam_step(p.astype(np.float64), g.astype(np.float64), 0, 0, 1, 1e-3)
    assert np.max(np.abs(p1 - ref1)) < 2e-6
    loss1, g1 = net.gradient(x, t)
    net.set_params(p)
    hist = net.train(x, t, idx, lr=1e-3)
    assert hist[0] == np.float32(loss) and hist[1] == np.float32(loss1)
    _, m, v = MO.adam_step(p.astype(np.float64), g.astype(np.float64), 0, 0, 1, 1e-3)
    ref2, _, _ = MO.adam_step(p1.astype(np.float64), g1.astype(np.float64), m, v, 2, 1e-3)
    assert np.max(np.abs(net.get_params() - ref2)) < 2e-6
