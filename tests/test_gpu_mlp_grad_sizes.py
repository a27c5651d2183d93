"""The device gradient at the sizes where its tiling can go wrong.

A block takes four tiles of 16 samples, at most 256 blocks run and then go
round again: one sample, a tile and its neighbours, a block and its
neighbours, one sample more than all blocks take in one round (16385), and an
offset into the data.  The CPU restatement rounds to BF16 at the same points;
an activation that falls on the other side of a rounding boundary there moves
a sample's share by up to 2^-8 of it, and with few samples such a share is not
averaged out, so each block of the gradient is held to 2^-7 of its norm.  The
sum over the batch has a fixed order: two calls give the same bits.
"""
import numpy as np
import pytest

import cueva
from cueva import learned_c2p as lc
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": (mo.OFF_W1, mo.OFF_B1), "b1": (mo.OFF_B1, mo.OFF_W2), "W2": (mo.OFF_W2, mo.OFF_B2),
          "b2": (mo.OFF_B2, mo.OFF_W3), "W3": (mo.OFF_W3, mo.OFF_B3), "b3": (mo.OFF_B3, mo.NPARAM)}


@pytest.mark.parametrize("off,cnt", [(0, 1), (3, 15), (0, 16), (5, 17), (0, 63), (1, 64), (0, 65), (7, 257),
                                     (2, 4099), (0, 16384), (11, 16385), (0, 20011)])
def test_gradient_sizes(off, cnt):
    rng = np.random.default_rng(cnt)
    n = 20032
    x = rng.normal(size=(n, 3)).astype(np.float32)
    t = rng.normal(size=(n, 2)).astype(np.float32)
    p = lc.pack(lc.init_weights(4) + rng.normal(scale=0.05, size=cueva.MLP_NPARAM).astype(np.float32), np.zeros(3),
                np.ones(3), np.zeros(2), np.ones(2))
    with cueva.Mlp(p) as m:
        m.set_data(x, t)
        g, loss = m.grad(off, cnt)
        g2, loss2 = m.grad(off, cnt)
    assert np.array_equal(g, g2) and loss == loss2
    want_loss, want = mo.loss_and_grad(p, x[off:off + cnt], t[off:off + cnt])
    assert abs(loss - want_loss) <= 2.0 ** -7 * want_loss
    for name, (a, b) in BLOCKS.items():
        rel = np.linalg.norm(g[a:b] - want[a:b]) / np.linalg.norm(want[a:b])
        print(off, cnt, name, "%.2e" % rel, flush=True)
        assert rel <= 2.0 ** -7, name
