"""Lattices whose z-groups are dispatched in several z-blocks (two or one z-row per
unit, more than 256 units from one z-group to the next, eight z-groups per XCD), in
every stored form: the same bytes as in hardware order.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402


def _run(sun, dims, precision, storage, mode):
    with Q.Lattice(sun=sun, dims=dims, beta=5.9 if sun == 3 else 2.3, precision=precision, storage_reals=storage, prng="PM",
                   randseries=5, max_measurements=4) as lat:
        lat.tune(xcd_map=mode)
        lat.init("cold")
        lat.prng_init()
        lat.run_cycle(n_hb=1, n_or=1)
        lat.sync()
        return lat.save_state()


@pytest.mark.parametrize("sun,dims,precision,storage", [
    (2, (24, 64, 16, 86), "fp32", 4),     # two z-rows per unit, two z-blocks
    (2, (8, 128, 16, 258), "fp64", 4),    # one z-row, four z-blocks
    (3, (24, 64, 16, 86), "fp32", 18),
    (3, (8, 128, 8, 258), "fp32", 12),    # one z-row, two z-blocks
    (3, (24, 64, 16, 86), "fp64", 18),
])
def test_same_bytes_as_hardware_order(sun, dims, precision, storage):
    print("[case]", sun, dims, precision, storage, flush=True)
    base = _run(sun, dims, precision, storage, 0)
    img = _run(sun, dims, precision, storage, 2)
    assert img.size == base.size and np.array_equal(img, base)
