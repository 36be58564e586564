"""Export and import of the links: every site's link lands in its own place for
each stored form, lattices of one partial block to several transfer slots, and
transfers from several threads at once.  The values are exact: doubles carry the
stored type, the parts that are not stored follow from it in double precision.

Skips without a GPU."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402


def _stored(links, sun, storage, precision):
    """links as they come back: rounded to the stored type, the rest rebuilt."""
    a = np.asarray(links, dtype=np.float64)
    if precision == "fp32":
        a = a.astype(np.float32).astype(np.float64)
    m = a.reshape(-1, sun, sun, 2)
    if sun == 2:
        m[:, 1, 0, 0], m[:, 1, 0, 1] = -m[:, 0, 1, 0], m[:, 0, 1, 1]
        m[:, 1, 1, 0], m[:, 1, 1, 1] = m[:, 0, 0, 0], -m[:, 0, 0, 1]
    elif storage == 12:
        def mul(p, q):
            return p[:, 0] * q[:, 0] - p[:, 1] * q[:, 1], p[:, 0] * q[:, 1] + p[:, 1] * q[:, 0]

        u, v = m[:, 0], m[:, 1]
        for k in range(3):
            i, j = (k + 1) % 3, (k + 2) % 3
            (ar, ai), (br, bi) = mul(u[:, i], v[:, j]), mul(u[:, j], v[:, i])
            m[:, 2, k, 0], m[:, 2, k, 1] = ar - br, -(ai - bi)
    return a


def _links(lat, seed):
    return np.random.default_rng(seed).standard_normal(lat.link_shape())


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("sun,storage", [(2, 4), (3, 12), (3, 18)])
@pytest.mark.parametrize("dims", [
    (2, 2, 2, 2),        # a quarter of a block
    (6, 10, 2, 4),       # 240 pairs: the last block is half full
    (14, 6, 10, 22),     # slots that end inside a row
    (16, 12, 20, 18),    # more chunks than slots, the last one short
])
def test_round_trip(dims, sun, storage, precision):
    print("[case]", dims, sun, storage, precision, flush=True)
    with Q.Lattice(sun=sun, dims=dims, precision=precision, storage_reals=storage, max_measurements=2) as lat:
        a = _links(lat, 3)
        lat.import_links(a)
        assert np.array_equal(lat.export_links(), _stored(a, sun, storage, precision))


def test_threads():
    print("[case] threads", flush=True)
    lats = [Q.Lattice(sun=3, dims=(16, 12, 12, 8), precision="fp32", max_measurements=2) for _ in range(3)]
    bad = []

    def turn(k):
        for r in range(4):
            a = _links(lats[k], 10 * k + r)
            lats[k].import_links(a)
            if not np.array_equal(lats[k].export_links(), _stored(a, 3, 18, "fp32")):
                bad.append((k, r))

    th = [threading.Thread(target=turn, args=(k,)) for k in range(3)]
    [t.start() for t in th]
    [t.join() for t in th]
    [lat.close() for lat in lats]
    assert not bad
