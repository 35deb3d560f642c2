"""mplb_mlp_tensor after a forward or training call: the activations, output and loss
gradients of that call's last batch, bit for bit those of a gradient call with the same
parameters on the same batch (rows beyond the data are zero); in the two-launch network and
in one that keeps a launch per product."""
import numpy as np
import pytest

import multiphaselb_amd as M

pytestmark = pytest.mark.gpu

NETS = [([9, 64, 96, 32], 32), ([7, 1024, 512, 64], 32)]


def tensors(net, widths, B, backward):
    L = len(widths) - 1
    wp = [32] + widths[1:]
    out = {"y": net.tensor("y", 0, (B, widths[-1]))}
    for j in range(L):
        out["a%d" % j] = net.tensor("a", j, (B, wp[j]))
        if j:
            out["a32_%d" % j] = net.tensor("a32", j, (B, wp[j]))
        if backward:
            out["dz%d" % (j + 1)] = net.tensor("dz", j + 1, (B, widths[j + 1]))
            out["dzb%d" % (j + 1)] = net.tensor("dzb", j + 1, (B, widths[j + 1]))
    return out


def same(got, want):
    for k in want:
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("widths,B", NETS, ids=["two-launch", "per-product"])
def test_tensors_belong_to_the_last_call(widths, B):
    rng = np.random.default_rng(3)
    net = M.Mlp(widths, B)
    p = np.concatenate([np.concatenate([rng.uniform(-1, 1, a * b) * np.sqrt(6.0 / (a + b)), rng.uniform(-0.1, 0.1, b)])
                        for a, b in zip(widths[:-1], widths[1:])]).astype(np.float32)
    X = rng.uniform(-1, 1, (3 * B, widths[0])).astype(np.float32)
    T = rng.uniform(-1, 1, (3 * B, widths[-1])).astype(np.float32)
    idx = rng.permutation(3 * B).astype(np.int32)
    for iters in (1, 3):
        net.set_params(p)
        if iters > 1:
            net.train(X, T, idx[:(iters - 1) * B], lr=1e-3)
        before = net.get_params()
        last = idx[(iters - 1) * B:iters * B]
        net.set_params(before)
        net.gradient(X[last], T[last])
        want = tensors(net, widths, B, True)
        net.set_params(p)
        net.gradient(X[:B], T[:B])
        net.train(X, T, idx[:iters * B], lr=1e-3)
        same(tensors(net, widths, B, True), want)
    for rows in (5, B, 2 * B + 17):
        x = np.zeros((B, widths[0]), np.float32)
        first = (rows - 1) // B * B
        x[:rows - first] = X[first:rows]
        net.gradient(x, T[:B])
        want = tensors(net, widths, B, False)
        net.gradient(X[B:2 * B], T[:B])
        y = net.forward(X[:rows])
        assert np.array_equal(y[first:], want["y"][:rows - first])
        same(tensors(net, widths, B, False), want)
