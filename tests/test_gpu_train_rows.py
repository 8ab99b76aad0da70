"""The training pass (k_net_pass, k_net_grad, k_net_reduce) at the edges of its tiles: workgroups
of 64 rows, chunks of 32, splits of the row sum from 2,048 rows on, windows that start inside the
data. Gradients against FP64 (oracle/mlp_ref.py), one Adam step against its formula on the
gradients, and the forward pass against the FP64 reference with the same bf16 roundings."""
import sys

import numpy as np
import pytest

from tests.test_gpu_learned import identity_norm, random_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 33, 63, 64, 65, 1000, 2047, 2048, 4100])
def test_gradients_and_adam_step(built, rows):
    from morphogenesis_amd.learned import Net
    from oracle import mlp_ref as R

    print("case: training rows", rows, flush=True)
    sys.stdout.flush()
    row0 = 37
    X, T, M = random_data(row0 + rows + 5, rows)
    M[row0] = 1.0  # at least one row counts
    mu, inv = identity_norm()
    net = Net(seed=rows)
    net.set_norm(mu, inv, 1.0)
    net.load_data(X, T, M)
    at = slice(row0, row0 + rows)
    p = net.get_params().astype(np.float64)
    xn = R.normalise(X[at], mu, inv)
    y = net.forward(row0, rows)
    ref = R.forward_bf16(p, xn)[:, :6]
    assert np.abs(y - ref).max() <= 2e-3 * np.abs(ref).max()
    loss, g = net.grad(row0, rows)
    ref_loss, ref_g = R.loss_and_grad(p, xn, T[at], M[at])
    assert abs(loss - ref_loss) <= 2e-2 * abs(ref_loss)
    # at most nine bf16 roundings of 2^-9 follow each other from an input to a gradient (0.2% each)
    for name, _ in R.SHAPES:
        a, b = R.unpack(g)[name], R.unpack(ref_g)[name]
        assert np.linalg.norm(a - b) < 5e-2 * np.linalg.norm(b), name
    loss2, g2 = net.grad(row0, rows)
    assert loss2 == loss and np.array_equal(g, g2), "gradients are deterministic"

    # one Adam step over the whole data: m / c1 = g, v / c2 = g^2 up to rounding
    net.load_data(X[at], T[at], M[at])
    lr = 1e-2
    l = net.train(1, rows, lr, seed=1)
    assert l[0] == loss
    g64 = g.astype(np.float64)
    want = p - lr * g64 / (np.abs(g64) + 1e-8)
    # the fp32 moments and constants: a few 2^-24 of the update, and the weight's own rounding
    assert np.abs(net.get_params() - want).max() <= lr * 1e-3 + 2 ** -24 * np.abs(want).max()
    # the bf16 copies follow: the next forward pass runs on the updated weights
    q = net.get_params().astype(np.float64)
    y = net.forward(0, rows)
    ref = R.forward_bf16(q, xn)[:, :6]
    assert np.abs(y - ref).max() <= 2e-3 * np.abs(ref).max()
    net.close()
