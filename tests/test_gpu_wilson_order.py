"""Wilson loops of FP64 SU(3) links on both sides of the rule for the order of the
workgroups (one x-slab per XCD; hardware order for long lines on planes that lie
powers of two apart), against the loops of the exported links, with the bound of
test_gpu_wilson_shapes.py.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402
from test_gpu_wilson_shapes import _loops  # noqa: E402


@pytest.mark.parametrize("storage", [18, 12])
@pytest.mark.parametrize("dims,R,T", [
    ((8, 32, 32, 8), 4, 2),    # slabs
    ((8, 32, 32, 8), 5, 2),    # hardware order
    ((2, 32, 32, 8), 7, 1),    # hardware order, around x
    ((8, 32, 32, 6), 5, 2),    # planes of 6144 sites: slabs
    ((4, 32, 30, 10), 5, 2),   # no power of two: slabs
])
def test_orders(dims, R, T, storage):
    print("[case]", dims, R, T, storage, flush=True)
    with Q.Lattice(sun=3, dims=dims, beta=5.8, precision="fp64", storage_reals=storage, prng="XOR128", randseries=3,
                   max_measurements=2) as lat:
        lat.set_wilson(R, T)
        lat.prng_init()
        lat.init("hot")
        lat.sweep("hb")
        lat.measure(wilson=True)
        got = float(np.ravel(lat.wilson_measurements(raw=True))[0])
        want = _loops(lat.export_links(), dims, 3, R, T)
    assert abs(got - want) <= 3 * np.prod(dims) * 2 * (R + T) * 8 * 2.0 ** -52 * 3
