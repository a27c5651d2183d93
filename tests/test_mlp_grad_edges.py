"""Which samples the device gradient takes: all of the range, none beside it.

test_gpu_mlp_grad_sizes.py holds each block of the gradient to 2^-7 of its
norm, which one sample of 16385 does not reach.  Here

- the samples at the edges of the range and of its tiles (16 samples), blocks
  (64) and rounds (256 blocks), and the neighbours outside the range, carry
  targets 1e4 times the others', so that one of them left out or taken in shows
  against the oracle.  An activation on the other side of a BF16 rounding
  boundary moves a sample's share by up to 2^-8 of it: each block of the
  gradient is held to 2^-7 of the sum of those samples' norms;
- the range cut in three adds up to the whole, where every error has one sign.
  The two sides round apart in FP32: at most 110 additions in a row (two rounds
  of 16 samples, four wavefronts, 64 partial sums and the ends) and 40
  operations within a sample's share, so each parameter is held to
  2 x 150 x 2^-24 of the sum of the magnitudes, and the loss (FP64, over an FP32
  1/n) to 2^-22.

The checks run on the device, and on the oracle with samples left out or taken
in, where they have to fail.
"""
import numpy as np
import pytest

import cueva
from cueva import learned_c2p as lc
from oracle import mlp_oracle as mo

N = 20032
SIZES = [(0, 1), (3, 15), (0, 16), (5, 17), (0, 63), (1, 64), (0, 65), (7, 257), (2, 4099), (0, 16384), (11, 16385),
         (0, 20011)]
CUTS = (0, mo.OFF_B1, mo.OFF_W2, mo.OFF_B2, mo.OFF_W3, mo.OFF_B3, mo.NPARAM)


def params(rng):
    return lc.pack(lc.init_weights(4) + rng.normal(scale=0.05, size=cueva.MLP_NPARAM).astype(np.float32), np.zeros(3),
                   np.ones(3), np.zeros(2), np.ones(2))


def edge_data(off, cnt):
    rng = np.random.default_rng(cnt)
    x = rng.normal(size=(N, 3)).astype(np.float32)
    t = rng.normal(size=(N, 2)).astype(np.float32)
    p = params(rng)
    edges = {0, cnt - 1} | {e for q in (16, 64, 16384) for e in (q - 1, q, (cnt - 1) // q * q - 1, (cnt - 1) // q * q)}
    edges = sorted(e for e in edges if 0 <= e < cnt)
    heavy = [off + e for e in edges] + [e for e in (off - 1, off + cnt) if 0 <= e < N]
    t[heavy] += 1.0e4
    return p, x, t, [off + e for e in edges]


def check_edges(off, cnt, data, grad):
    p, x, t, edges = data
    g, loss = grad(off, cnt)
    want_loss, want = mo.loss_and_grad(p, x[off:off + cnt], t[off:off + cnt])
    assert abs(loss - want_loss) <= 2.0 ** -7 * want_loss
    shares = np.stack([mo.loss_and_grad(p, x[e:e + 1], t[e:e + 1])[1] for e in edges]) / cnt
    for a, b in zip(CUTS, CUTS[1:]):
        assert np.linalg.norm(g[a:b] - want[a:b]) <= 2.0 ** -7 * np.linalg.norm(shares[:, a:b], axis=1).sum(), (a, b)


def sum_data(off, cnt):
    rng = np.random.default_rng(cnt + 1)
    x = rng.normal(size=(N, 3)).astype(np.float32)
    return params(rng), x, (100.0 + rng.normal(size=(N, 2))).astype(np.float32)


def magnitudes(p, x, t):
    """The gradient's sums with every term's magnitude in place of the term."""
    w1, _, w2, _, w3, _ = mo.unpack(p)
    y, (xb, h1, h1b, h2, h2b) = mo.forward(p, x)
    dy = np.abs(2.0 * (y - t) / len(x))
    dz2 = (dy @ np.abs(mo.bf16(w3))) * (1.0 - h2 * h2)
    dz1 = (dz2 @ np.abs(mo.bf16(w2))) * (1.0 - h1 * h1)
    xb, h1b, h2b = np.abs(xb), np.abs(h1b), np.abs(h2b)
    return np.concatenate([(dz1.T @ xb).ravel(), dz1.sum(0), (dz2.T @ h1b).ravel(), dz2.sum(0), (dy.T @ h2b).ravel(),
                           dy.sum(0)])


def check_sum(off, cnt, data, grad):
    p, x, t = data
    g, loss = grad(off, cnt)
    cut = [0, max(1, cnt // 3), max(2, cnt // 3 + cnt // 2), cnt] if cnt > 2 else [0, cnt]
    parts = [(grad(off + a, b - a), b - a) for a, b in zip(cut, cut[1:])]
    g3 = sum(np.asarray(q[0], dtype=np.float64) * n for q, n in parts) / cnt
    assert abs(sum(q[1] * n for q, n in parts) / cnt - loss) <= 2.0 ** -22 * loss
    bound = 300.0 * 2.0 ** -24 * magnitudes(p, x[off:off + cnt], t[off:off + cnt])
    assert (np.abs(g3 - g) <= bound).all(), float((np.abs(g3 - g) / bound).max())


CHECKS = {"edges": (edge_data, check_edges), "sum": (sum_data, check_sum)}


@pytest.mark.gpu
@pytest.mark.parametrize("check", sorted(CHECKS))
@pytest.mark.parametrize("off,cnt", SIZES)
def test_device_gradient(off, cnt, check):
    print("gradient", check, off, cnt, flush=True)
    make, test = CHECKS[check]
    data = make(off, cnt)
    with cueva.Mlp(data[0]) as m:
        m.set_data(data[1], data[2])
        test(off, cnt, data, m.grad)


# the samples that a gradient with a mistake takes of a range of n (of all N from its first one on)
MISTAKES = {
    "none": lambda n: range(0, n),
    "first_left_out": lambda n: range(1, n),
    "last_left_out": lambda n: range(0, n - 1),
    "one_past": lambda n: range(0, n + 1),
    "one_before": lambda n: range(-1, n),
    "no_ragged_tile": lambda n: range(0, n // 16 * 16),
    "no_ragged_block": lambda n: range(0, n // 64 * 64),
    "one_round": lambda n: range(0, min(n, 16384)),
}


@pytest.mark.parametrize("mistake", sorted(MISTAKES))
@pytest.mark.parametrize("off,cnt", [(5, 17), (7, 257), (11, 16385), (0, 20011)])
def test_oracle_with_a_mistake(off, cnt, mistake):
    def wrong(data):
        def grad(o, n):
            take = [o + s for s in MISTAKES[mistake](n) if 0 <= o + s < N]
            if not take:
                return np.zeros(mo.NPARAM), 0.0
            loss, g = mo.loss_and_grad(data[0], data[1][take], data[2][take])
            return g * len(take) / n, loss * len(take) / n
        return grad

    same = [off + s for s in MISTAKES[mistake](cnt) if 0 <= off + s < N] == list(range(off, off + cnt))
    caught = []
    for name in sorted(CHECKS):
        make, test = CHECKS[name]
        data = make(off, cnt)
        try:
            test(off, cnt, data, wrong(data))
        except AssertionError:
            caught.append(name)
    if mistake == "none":
        assert not caught
    elif not same:
        assert "edges" in caught, caught
        # a mistake that leaves nothing of the range adds up all the same
        assert "sum" in caught or not list(MISTAKES[mistake](cnt)), caught
