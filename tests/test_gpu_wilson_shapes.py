"""Wilson loops on lattices of both kernel shapes (a thread per site and direction
up to 256 workgroups of sites, a thread per site beyond) against the loops of the
exported links in double precision: lines of one link, lines around the lattice,
several lengths.

A loop is 2 (R + T) products of SU(2) matrices, each off by a few 2^-52, summed
over 3 V sites and directions: 3 V 2 (R + T) 8 2^-52 bounds the difference.
Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402


def _loops(links, dims, N, R, T):
    """Sum of ReTr over sites and spatial directions; sites run y fastest, then z, t, x."""
    u = links.reshape(dims[0], dims[3], dims[2], dims[1], 4, N, N, 2)
    U = (u[..., 0] + 1j * u[..., 1]).transpose(4, 0, 3, 2, 1, 5, 6)   # [dir][x][y][z][t]

    def line(d, n):
        P = U[d]
        for k in range(1, n):
            P = P @ np.roll(U[d], -k, axis=d)
        return P

    Lt, s = line(3, T), 0.0
    for d in range(3):
        Ld = line(d, R)
        W = Lt @ np.roll(Ld, -T, axis=3)
        V = Ld @ np.roll(Lt, -R, axis=d)
        s += np.einsum("...ij,...ij->...", W, V.conj()).real.sum()
    return s


@pytest.mark.parametrize("sun,dims,R,T", [
    (2, (2, 2, 2, 2), 1, 1),
    (2, (6, 4, 10, 2), 5, 3),         # around y and t
    (2, (16, 16, 16, 16), 10, 3),     # 256 workgroups
    (2, (16, 16, 16, 18), 7, 2),      # 288: a thread per site
    (3, (6, 4, 10, 2), 7, 13),
])
def test_wilson(sun, dims, R, T):
    print("[case]", sun, dims, R, T, flush=True)
    with Q.Lattice(sun=sun, dims=dims, beta=2.3 if sun == 2 else 5.8, precision="fp64", prng="XOR128", randseries=3,
                   max_measurements=2) as lat:
        lat.set_wilson(R, T)
        lat.prng_init()
        lat.init("hot")
        lat.sweep("hb")
        lat.measure(wilson=True)
        got = float(np.ravel(lat.wilson_measurements(raw=True))[0])
        want = _loops(lat.export_links(), dims, sun, R, T)
    assert abs(got - want) <= 3 * np.prod(dims) * 2 * (R + T) * 8 * 2.0 ** -52 * sun
