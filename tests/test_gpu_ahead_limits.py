"""RANLUX quads made ahead, at the places test_gpu_ranlux_ahead.py does not reach: a
lattice whose quads exceed the buffer's 192 MiB (half-steps produce for themselves),
and workgroups of several units of which the last has one less.  Sweeps give the bits
of half-steps that produce for themselves, links and streams.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402
from test_gpu_ranlux_ahead import _by_halfsteps, _lattice  # noqa: E402


@pytest.mark.parametrize("kw", [
    dict(sun=2, dims=(32, 16, 32, 34)),                         # 4 x 11 quads of 278528 streams: 187 MiB
    dict(sun=2, dims=(32, 16, 32, 36)),                         # 198 MiB
    dict(sun=3, dims=(8, 6, 4, 86), storage_reals=12),          # 129 units: 64 workgroups of two, one of one
    dict(sun=3, dims=(2, 10, 10, 86), ranlux_luxury=4),         # 8600 streams: 135 units, the last one partly filled
])
def test_sweeps_equal_halfsteps(kw):
    print("[case]", kw, flush=True)
    a, b = _lattice(**kw), _lattice(**kw)
    for _ in range(2):
        a.sweep("hb")
        _by_halfsteps(b)
        assert np.array_equal(a.save_state(), b.save_state())
    a.close()
    b.close()
