"""Heatbath sweeps whose RANLUX quads are produced four half-steps at a time give
the bits of half-steps that produce for themselves, links and streams, eagerly and
replayed: every position inside a block, kept parts of one quad to all, stream
counts around a wavefront, long and short luxury skips, lattices on both sides of
the buffer's limit.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402


def _lattice(**kw):
    lat = Q.Lattice(beta=2.3 if kw["sun"] == 2 else 5.8, randseries=11, prng="RANLUX", max_measurements=16, **kw)
    lat.prng_init()
    lat.init("cold")
    return lat


def _by_halfsteps(lat):
    for parity in (1, 0):
        for mu in range(4):
            lat.halfstep(parity, mu, "hb")


@pytest.mark.parametrize("kw", [
    dict(sun=2, dims=(2, 2, 2, 2)),                              # 8 streams
    dict(sun=2, dims=(4, 4, 4, 2), nhit=1),                      # one wavefront, 2 of 6 quads kept
    dict(sun=2, dims=(6, 2, 6, 4), precision="fp64"),            # 144 streams, 11 of 33 kept
    dict(sun=3, dims=(6, 4, 2, 4), storage_reals=12),            # all 33 kept
    dict(sun=3, dims=(4, 4, 4, 4), nhit=3, ranlux_luxury=0),     # 12 of 12
    dict(sun=3, dims=(4, 4, 4, 4), nhit=2, ranlux_luxury=4),     # 9 of 9: blocks shared by half-steps
    dict(sun=2, dims=(4, 4, 4, 4), nhit=11),                     # 36 quads
    dict(sun=3, dims=(8, 12, 8, 22), storage_reals=12),          # 132 units: two in turn, the last workgroups one
    dict(sun=2, dims=(32, 16, 32, 34)),                          # 197 MB: half-steps produce for themselves
])
def test_sweeps_equal_halfsteps(kw):
    print("[case]", kw, flush=True)
    a, b = _lattice(**kw), _lattice(**kw)
    small = np.prod(kw["dims"]) < 1 << 16
    for n in range(7 if small else 2):
        a.sweep("hb")
        _by_halfsteps(b)
        if n == 2:   # the streams go on from a half-step of their own
            a.halfstep(0, 1, "hb")
            b.halfstep(0, 1, "hb")
        assert np.array_equal(a.save_state(), b.save_state())
    if small:
        a.capture_cycle(n_hb=3, n_or=1, plaquette=False, polyakov=False)
        for _ in range(3):
            a.launch_cycle(2)
            a.sync()
            for _ in range(2):
                for _ in range(3):
                    _by_halfsteps(b)
                b.sweep("or")
            assert np.array_equal(a.export_links(), b.export_links())
            a.sweep("hb")
            _by_halfsteps(b)
            assert np.array_equal(a.save_state(), b.save_state())
    a.close()
    b.close()


def test_beside_a_recording():
    """A first sweep and an export of one lattice while another one's graph is recorded: both give
    what they give alone."""
    print("[case] beside a recording", flush=True)
    kw = dict(sun=3, dims=(4, 4, 4, 4))
    a, b, c = _lattice(**kw), _lattice(**kw), _lattice(**kw)
    a.graph_begin()
    a.sweep("hb")
    b.sweep("hb")
    links = b.export_links()
    a.sweep("or")
    a.graph_end()
    for _ in range(3):
        a.launch_cycle(1)
        a.sync()
        _by_halfsteps(c)
        if _ == 0:
            assert np.array_equal(links, c.export_links())
        c.sweep("or")
        assert np.array_equal(a.export_links(), c.export_links())
    for lat in (a, b, c):
        lat.close()
