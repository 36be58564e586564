"""A batch of FP64 18-real SU(3) chains whose links exceed the last-level cache takes
another overrelaxation kernel than a smaller one, 12 reals take that one always: every
chain is still bit for bit the chain run alone, links and records, with the plaquette
fused and without.

Skips without a GPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import qcdgpu_amd as Q  # noqa: E402


@pytest.mark.parametrize("storage,chains", [
    (18, [((24, 24, 24, 16), 5.9, 3), ((24, 24, 24, 18), 5.7, 4)]),   # 258 MiB
    (18, [((24, 24, 24, 16), 5.9, 3), ((24, 24, 24, 16), 5.7, 4)]),   # 243 MiB
    (12, [((12, 12, 12, 16), 5.9, 3), ((12, 16, 12, 6), 5.7, 4)]),
])
def test_chains_alone(storage, chains):
    print("[case]", storage, chains, flush=True)
    kw = dict(sun=3, precision="fp64", storage_reals=storage, prng="XOR128", max_measurements=4)
    got = []
    with Q.Batch(chains, **kw) as b:
        b.init("cold")
        b.sweep("hb")
        b.sweep("or")
        b.run_cycle(n_hb=0, n_or=1)
        b.sync()
        for k in range(len(chains)):
            got.append((b.chain(k).export_links(), b.chain(k).raw_measurements()))
    for (dims, beta, seed), (links, records) in zip(chains, got):
        with Q.Lattice(dims=dims, beta=beta, randseries=seed, **kw) as lat:
            lat.prng_init()
            lat.init("cold")
            lat.sweep("hb")
            lat.sweep("or")
            lat.run_cycle(n_hb=0, n_or=1)
            lat.sync()
            assert np.array_equal(lat.export_links(), links), dims
            for r, q in zip(lat.raw_measurements(), records):
                assert np.array_equal(r, q), dims
