"""Dispatch orders of the update kernels on extents where the XCD ranges are
uneven, hold x-values that are no whole units, or are walked in z-blocks: every
order must leave the same bytes (links, streams, records) as hardware order.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402

CASES = [
    # (sun, dims, precision, storage, prng)
    (3, (4, 4, 4, 4), "fp64", 18, "XOR128"),       # 2 units: most XCDs have none
    (3, (6, 10, 6, 4), "fp32", 18, "RANLUX"),      # 12 units, the last one partly filled
    (3, (8, 6, 4, 4), "fp32", 12, "PM"),           # N1 a multiple of 8, 48 links per x-value: under one unit
    (3, (16, 6, 10, 6), "fp64", 18, "XOR128"),     # 180 links per x-value, two x-values per XCD
    (2, (24, 24, 12, 4), "fp32", 4, "XOR128"),     # 9 whole units per x-value
    (2, (64, 64, 8, 64), "fp32", 4, "PM"),         # z-blocks of four z-groups
]


def _run(case, mode, phi):
    sun, dims, prec, storage, prng = case
    with Q.Lattice(sun=sun, dims=dims, beta=5.9 if sun == 3 else 2.3, precision=prec, storage_reals=storage, prng=prng,
                   randseries=5, max_measurements=4) as lat:
        lat.tune(xcd_map=mode)
        if phi:
            lat.set_twist(phi)
        lat.init("cold")
        lat.prng_init()
        lat.capture_cycle(n_hb=1, n_or=1, plaquette=True, polyakov=True)
        lat.launch_cycle(2)
        lat.sync()
        return lat.save_state()


@pytest.mark.parametrize("phi", [0.0, 0.7])
@pytest.mark.parametrize("case", CASES, ids=["su%d-%s-%s-%d-%s" % (c[0], "x".join(map(str, c[1])), c[2], c[3], c[4])
                                             for c in CASES])
def test_orders_leave_the_same_bytes(case, phi):
    print("[case]", case, phi, flush=True)
    base = _run(case, 0, phi)
    for mode in (1, 2, 3):
        img = _run(case, mode, phi)
        assert img.size == base.size
        assert int(np.count_nonzero(img != base)) == 0, mode
