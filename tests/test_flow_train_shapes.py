"""Kernel shapes of the training gradient: a batch's gradient is the sum of its
configurations' own, whichever shape its size selects (the per-site factors are
the same bits, the FP32 sums run in another order), and it follows the FP32
twin's autograd for every number of spline bins, on both weight-gradient paths.

Sums of n FP32 terms of random sign: about sqrt(n) 2^-24 of their norm, n up to
81920 here: 2e-5, times 5 for the two sides and the tail: 1e-4.  Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from qcdgpu_amd import flow as QF  # noqa: E402

BLOCKS = (QF.W1N, QF.HIDDEN, QF.W2N, QF.COUT)


def _params(layers, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(layers):
        for n, s in zip(BLOCKS, (0.1, 0.1, 0.01, 0.3)):
            out.append(s * rng.standard_normal(n))
    return np.concatenate(out).astype(np.float32)


def _links(dims, count, seed):
    q = 0.45 * np.random.default_rng(seed).standard_normal((count, 4, int(np.prod(dims)), 4))
    q[..., 0] += 1.0
    return (q / np.linalg.norm(q, axis=-1, keepdims=True)).astype(np.float32)


def _blocks(g):
    """(layer, block, values)"""
    o = 0
    for l in range(len(g) // QF.LAYER_PARAMS):
        for b, n in enumerate(BLOCKS):
            yield l, b, g[o:o + n]
            o += n


@pytest.mark.parametrize("dims,batch,bins", [
    ((8, 8, 8, 4), 5, 4),      # 40 x-planes in segments of 64 rows
    ((8, 8, 8, 4), 40, 4),     # 320 x-planes on 256 workgroups
    ((6, 10, 12, 2), 3, 3),    # planes of 15 tiles: the last step half empty
    ((4, 4, 4, 4), 2, 5),      # two steps per plane
    ((4, 14, 14, 10), 2, 2),   # planes too large for LDS
    ((2, 2, 2, 2), 3, 1),      # planes of half a tile
])
def test_batch_is_the_sum(dims, batch, bins):
    print("[case]", dims, batch, bins, flush=True)
    links, p = _links(dims, batch, 1), _params(4, 2)
    with QF.Flow(dims=dims, layers=4, bins=bins, max_batch=batch) as f:
        f.set_params(p)
        loss, g = f.train_grad(links)
        one = [f.train_grad(links[k:k + 1]) for k in range(batch)]
    assert abs(loss - np.mean([o[0] for o in one])) <= 1e-6 * max(1.0, np.mean([abs(o[0]) for o in one]))
    want = np.sum([o[1].astype(np.float64) for o in one], axis=0)
    scale = np.sqrt(np.sum([o[1].astype(np.float64) ** 2 for o in one], axis=0))
    for (l, b, u), (_, _, v), (_, _, s) in zip(_blocks(g), _blocks(want), _blocks(scale)):
        assert np.linalg.norm(u - v) <= 1e-4 * np.linalg.norm(s), (l, b)


@pytest.mark.parametrize("dims,bins", [
    ((4, 6, 4, 2), 1), ((4, 6, 4, 2), 2), ((4, 6, 4, 2), 3), ((4, 6, 4, 2), 4), ((4, 6, 4, 2), 5),   # planes of 3 tiles
    ((8, 2, 6, 2), 3),   # planes of 24 rows: by chunks of rows
])
def test_bins_against_autograd(dims, bins):
    import torch

    print("[case]", dims, bins, flush=True)
    links, p = _links(dims, 3, 4), _params(4, 5)
    m = QF.FlowModel(dims=dims, layers=4, bins=bins, device="cpu")
    with torch.no_grad():
        m.params.copy_(torch.from_numpy(p))
    m.local_nll(torch.from_numpy(links)).sum().backward()
    want = m.params.grad.numpy()
    with QF.Flow(dims=dims, layers=4, bins=bins, max_batch=3) as f:
        f.set_params(p)
        _, g = f.train_grad(links)
    # BF16 operands: the bounds of the existing comparison with autograd
    for (l, b, u), (_, _, v) in zip(_blocks(g), _blocks(want)):
        cos = float(np.dot(u, v) / (np.linalg.norm(u) * np.linalg.norm(v)))
        assert cos >= 0.99 and np.linalg.norm(u - v) <= 0.1 * np.linalg.norm(v), (l, b, cos)


@pytest.mark.parametrize("below", [0.0, 2e-6])
def test_gradient_at_a_knot(below):
    """Links whose loop angle lies on the knot pi/2 of a spline with two equal
    heights, or a part of a step below it: the gradient is the symmetric
    difference's.  One value on all active sites; BF16 keeps 8 bits of it (2^-8),
    and the knots' FP32 constants move the step's parts by 1e-3 at most."""
    import math
    import os
    import sys

    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
    import flow_ref as FR

    print("[case] knot", below, flush=True)
    dims, K = (4, 4, 4, 4), 2
    r = np.array([0.7, -0.4, 0.2, 0.2, -0.5, 0.9, 0.3])
    th = math.pi / 2 - below
    links = np.zeros((1, 4, 256, 4), dtype=np.float32)
    links[..., 0] = 1.0
    for s in range(256):   # sites run y fastest, then z, t, x; direction x is active where y + z + t is even
        y, z, t = s % 4, (s // 4) % 4, (s // 16) % 4
        if (y + z + t) % 2 == 0:
            links[0, 0, s] = (math.cos(th), 0.0, 0.0, math.sin(th))
    p = np.zeros(QF.LAYER_PARAMS, dtype=np.float32)
    p[-QF.COUT:-QF.COUT + 7] = r
    with QF.Flow(dims=dims, layers=1, bins=K, max_batch=1) as f:
        f.set_params(p)
        loss, g = f.train_grad(links)

    th = math.atan2(float(links[0, 0, 0, 3]), float(links[0, 0, 0, 0]))
    r = p[-QF.COUT:-QF.COUT + 7].astype(np.float64)

    def nll(q):
        x, dlog = FR.spline(q, K, th, inverse=True)
        return dlog + 2 * math.log(math.sin(th) / math.sin(x))

    want = np.array([(nll(r + 1e-5 * e) - nll(r - 1e-5 * e)) / 2e-5 for e in np.eye(7)])
    got = g[-QF.COUT:-QF.COUT + 7] / 128.0
    print("  ", got, want)
    assert abs(loss - 128 * nll(r)) <= 1e-4 * 128
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 1e-3 * np.abs(want).max())
