"""RANLUX produce() with its blocks in parallel: quads and streams equal the
oracle's number for number, for every luxury level, at every position inside a
block, for stream counts around a wavefront, on both sides of the length the
jump tables reach, and for the states whose product needs its last reduction.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402

B = 1 << 24
M = B ** 24 - B ** 10 + 1
SKIP = {0: 24, 1: 48, 2: 97, 3: 223, 4: 389}


def _digits(v):
    return [(v >> (24 * j)) & (B - 1) for j in range(24)]


def _state_of(X):
    """Ring x_{n-24} .. x_{n-1} and borrow of the state X_n = X: the 24 numbers
    that follow X_{n-24} = X b^24."""
    Y = X * pow(B, 24, M) % M
    d, r, c = _digits(Y), [], 0
    for j in range(24):
        t = (r[j - 10] if j >= 10 else 0) - d[j] - c
        c = int(t < 0)
        r.append(t % B)
    return r, c


def _table(states):
    """7 float4 per stream at the end of a block (position 23 the oldest)."""
    t = np.zeros((7, len(states), 4), dtype=np.float32)
    for g, (ring, c) in enumerate(states):
        for j, x in enumerate(ring):
            p = 23 - j
            t[p // 4, g, p % 4] = np.float32(x) * np.float32(2.0 ** -24)
        t[6, g] = (23.0, 9.0, 6.0, 2.0 ** -24 if c else 0.0)
    return t


def _check(O, table, samples, lux):
    want_t = table.copy()
    want = O.ranlux_produce(want_t, samples, SKIP[lux])
    got = Q.prng_produce("RANLUX", table, samples, luxury=lux)
    assert np.array_equal(got.view(np.uint32), np.asarray(want, dtype=np.float32).reshape(got.shape).view(np.uint32))
    assert np.array_equal(table, want_t)


@pytest.mark.parametrize("lux", range(5))
@pytest.mark.parametrize("n", [1, 64, 65, 200])
def test_produce_at_every_position(O, lux, n):
    print("[case]", lux, n, flush=True)
    t = O.ranlux_seed_table(17 + n, n).astype(np.float32).reshape(7, n, 4)
    for samples in (33, 1, 5, 6, 7, 2, 33, 41, 48, 49, 72, 73, 33):   # 49 and more: stepped through
        _check(O, t, samples, lux)


@pytest.mark.parametrize("lux", [0, 3])
def test_produce_from_edge_states(O, lux):
    print("[case] edge states", lux, flush=True)
    P = SKIP[lux]
    states = [([0] * 24, 0), ([B - 1] * 24, 1), ([0] * 24, 1), ([B - 1] * 24, 0)]
    for t in (1, 2):   # block t's product comes out as 0 .. b^10: below and above the second form + m
        N = t * P + (t - 1) * 24
        for want in (1, 2, B - 1, B, B ** 10 - 2, B ** 10 - 1, B ** 10, M - 1):
            states.append(_state_of(want * pow(B, N - 24, M) % M))
    _check(O, _table(states), 33, lux)
