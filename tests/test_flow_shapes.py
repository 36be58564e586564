"""Kernel shapes of the flow's convolutions and couplings: a batch gives every
configuration the bits it gets alone, whichever shape its size selects, and
one configuration agrees with the FP32 twin for every number of spline bins.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from qcdgpu_amd import flow as QF  # noqa: E402


def _params(layers, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(layers):
        for n, s in ((QF.W1N, 0.05), (QF.HIDDEN, 0.1), (QF.W2N, 0.006), (QF.COUT, 0.1)):
            out.append(s * rng.standard_normal(n))
    return np.concatenate(out).astype(np.float32)


def _links(dims, count, seed):
    q = 0.45 * np.random.default_rng(seed).standard_normal((count, 4, int(np.prod(dims)), 4))
    q[..., 0] += 1.0
    return (q / np.linalg.norm(q, axis=-1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("dims,batch,bins", [
    ((8, 8, 8, 4), 16, 4),     # 128 x-planes of 256 sites: eight wavefronts per plane
    ((8, 8, 8, 4), 40, 4),     # 320 x-planes: four wavefronts
    ((6, 10, 12, 2), 20, 3),   # planes of 15 tiles
    ((4, 14, 14, 10), 2, 2),   # planes too large for LDS, one tile per wavefront
    ((4, 14, 14, 10), 9, 5),   # 4410 tiles: four per wavefront, the last two alone
    ((2, 2, 2, 2), 3, 1),      # one tile per configuration
])
def test_batch_equals_alone(dims, batch, bins):
    print("[case]", dims, batch, bins, flush=True)
    links, p = _links(dims, batch, 1), _params(5, 2)
    with QF.Flow(dims=dims, layers=5, bins=bins, max_batch=batch) as f:
        f.set_params(p)
        lq, S = f.evaluate(links, 2.2)
        for k in sorted({0, batch // 2, batch - 1}):
            lq1, S1 = f.evaluate(links[k:k + 1], 2.2)
            assert lq1[0] == lq[k] and S1[0] == S[k]


@pytest.mark.parametrize("bins", [1, 2, 3, 4, 5])
def test_bins_against_twin(bins):
    import torch

    print("[case] bins", bins, flush=True)
    dims = (4, 6, 4, 2)
    links, p = _links(dims, 3, 4), _params(4, 5)
    m = QF.FlowModel(dims=dims, layers=4, bins=bins)
    with torch.no_grad():
        m.params.copy_(torch.from_numpy(p))
        want = m.log_q(torch.from_numpy(links)).numpy()
    with QF.Flow(dims=dims, layers=4, bins=bins, max_batch=3) as f:
        f.set_params(p)
        got, _ = f.evaluate(links, 2.2)
    # BF16 activations and weights, the bound of the existing comparison: 0.3 % of |log q|'s scale
    assert np.abs(got - want).max() <= 0.003 * max(np.abs(want).max(), 50.0)
