"""The library's host side without a GPU: libqcdhip.so on a stand-in for the HIP
runtime (fake_hip.c: host memory for device memory, kernels not run, every call
noted, allocations that can be made to fail).  Each test is a program of its own,
since the stand-in has to be loaded before the library."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

pytestmark = [
    pytest.mark.skipif(not os.path.exists(os.path.join(REPO, "qcdgpu_amd", "libqcdhip.so")), reason="libqcdhip.so not built"),
    pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc missing"),
]

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_limits.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
ANY = 2 ** 64 - 1
sys.path[:0] = %r
def calls():
    lines = fake.fake_log().decode().splitlines()
    fake.fake_clear()
    return lines
import numpy as np
import qcdgpu_amd as Q
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    r = subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", out, os.path.join(HERE, "fake_hip.c"), "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


def _run(fake, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE % [REPO, HERE] + code, fake], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("sun,storage", [(2, 4), (3, 12), (3, 18)])
def test_links_without_pinned_memory(fake, sun, storage, precision):
    """Import and export need ordinary memory only: no slot can be pinned here."""
    _run(fake, """
from test_gpu_links_move import _links, _stored
fake.fake_limits(ANY, 0)
for dims in ((2, 2, 2, 2), (6, 10, 2, 4), (4, 6, 10, 6)):
    with Q.Lattice(sun=%d, dims=dims, precision="%s", storage_reals=%d, max_measurements=2) as lat:
        a = _links(lat, 3)
        lat.import_links(a)
        assert np.array_equal(lat.export_links(), _stored(a, %d, %d, "%s")), dims
        assert not any("launch" in c for c in calls())
""" % (sun, precision, storage, sun, storage, precision))


def test_links_with_little_pinned_memory(fake):
    """Where eight slots cannot be pinned, fewer are taken."""
    _run(fake, """
fake.fake_limits(ANY, 3 << 20)
with Q.Lattice(sun=3, dims=(16, 16, 16, 16), max_measurements=2) as lat:
    calls()
    lat.export_links()
    seen = calls()
pinned = [c for c in seen if c.startswith("hostmalloc")]
assert pinned and not pinned[-1].endswith("failed"), pinned
assert sum(c.startswith("launch") for c in seen) > 8 and not any(c.startswith("copy") for c in seen)
""")


def test_pinned_memory_outlives_a_lattice(fake):
    """A lattice per configuration: the pinned memory is had once and given back by
    qcd_device_close, not with every last lattice."""
    _run(fake, """
from qcdgpu_amd import _abi
calls()
for _ in range(3):
    with Q.Lattice(sun=2, dims=(16, 16, 16, 8), max_measurements=2) as lat:
        lat.import_links(lat.export_links())
seen = calls()
assert sum(c.startswith("hostmalloc") for c in seen) == 1, seen
assert "hostfree" not in seen
assert _abi.lib().qcd_device_close() == 0
assert calls().count("hostfree") == 1
""")


def test_pinned_memory_is_coherent(fake):
    """The transfer kernel's writes are read by the host after an event: the memory says
    so itself (hipHostMallocCoherent), not an environment variable's default."""
    _run(fake, """
with Q.Lattice(sun=3, dims=(4, 4, 4, 4), max_measurements=2) as lat:
    calls()
    lat.export_links()
    flags = [int(c.split()[3]) for c in calls() if c.startswith("hostmalloc")]
assert flags and all(f & 0x40000000 for f in flags), flags
""")


def test_sweeps_without_memory_for_quads_ahead(fake):
    """Where the quads of several half-steps find no memory, sweeps go on as before they
    were made ahead: no wait and no further attempt in each of them, and nothing kept."""
    _run(fake, """
with Q.Lattice(sun=3, dims=(8, 8, 8, 8), prng="RANLUX", max_measurements=2) as lat:
    lat.prng_init()
    lat.init("cold")
    calls()
    fake.fake_limits(4 << 20, ANY)
    lat.sweep("hb")
    first = calls()
    assert sum(c.startswith("malloc") and c.endswith("failed") for c in first) == 1, first
    for _ in range(3):
        lat.sweep("hb")
    lat.run_cycle(n_hb=1, n_or=0)
    seen = calls()
    assert not any(c.startswith(("malloc", "wait")) for c in seen), seen
    assert sum(c.startswith("launch") for c in seen) >= 4 * 16   # a produce() and an update per half-step
    fake.fake_limits(ANY, ANY)
    lat.sweep("hb")   # as before, ...
    assert sum(c.startswith("launch") for c in calls()) == 16
    lat.capture_cycle(n_hb=1, n_or=0)   # ... until a recording asks again
    assert sum(c.startswith("malloc") for c in calls()) == 2
    lat.sweep("hb")
    assert sum(c.startswith("launch") for c in calls()) == 10
""")


def test_flow_works_on_its_own_stream(fake):
    """The flow's stream does not wait for the null stream nor the null stream for it: what
    is cleared, packed and copied follows in one order, and a gradient is waited for before
    it is read, also when the loss is not asked for."""
    _run(fake, """
from qcdgpu_amd import flow as QF, _abi
f = QF.Flow(dims=(4, 4, 4, 4), layers=2, max_batch=2)
p = np.zeros(f.param_count(), np.float32)
f.set_params(p)
links = np.ones((2, 4, 256, 4), np.float32)
f.train_grad(links)
f.set_params(p)
f.train_step(links, 1e-3)
f.imh_counts(reset=True)
seen = calls()
assert not any(c.startswith("clear") and " on " not in c for c in seen), seen
g = np.empty_like(p)
P = ctypes.POINTER(ctypes.c_float)
assert _abi.lib().qcd_flow_train_grad(f._h, links.ctypes.data_as(P), 2, None, g.ctypes.data_as(P)) == 0
seen = calls()
copy = [i for i, c in enumerate(seen) if c.startswith("copy kind 2")][-1]
assert " on " in seen[copy] and seen[copy + 1].startswith("wait on"), seen[copy:]
""")


def test_training_without_memory(fake):
    """A gradient that finds no memory for its buffers is refused, each time, and works
    once there is memory: never a launch on buffers that were not had."""
    _run(fake, """
from qcdgpu_amd import flow as QF
f = QF.Flow(dims=(4, 4, 4, 4), layers=1, max_batch=64)
f.set_params(np.zeros(f.param_count(), np.float32))
links = np.ones((2, 4, 256, 4), np.float32)
calls()
fake.fake_limits(300000, ANY)   # parameters fit, the partial sums do not
for _ in range(2):
    try:
        f.train_grad(links)
        raise SystemExit("accepted")
    except Q.QCDError as e:
        assert "training buffers" in str(e)
assert not any(c.startswith("launch") for c in calls())
fake.fake_limits(ANY, ANY)
f.train_grad(links)
assert any(c.startswith("launch") for c in calls())
""")


def test_start_without_memory_for_quads(fake):
    """A hot start that finds no memory for its larger quad buffer is refused; so are
    half-steps after it, until a start finds memory: never an update on no buffer."""
    _run(fake, """
def refused(f):
    try:
        f()
    except Q.QCDError:
        return
    raise SystemExit("accepted")
with Q.Lattice(sun=3, dims=(8, 8, 8, 8), prng="RANLUX", max_measurements=2) as lat:
    lat.prng_init()
    lat.init("cold")
    fake.fake_limits(1200000, ANY)   # 33 quads per stream fit, 41 do not
    refused(lambda: lat.init("random"))
    calls()
    refused(lambda: lat.halfstep(1, 0, "hb"))
    refused(lambda: lat.init("random"))
    assert not any(c.startswith("launch") for c in calls())
    fake.fake_limits(ANY, ANY)
    lat.init("random")
    lat.halfstep(1, 0, "hb")
""")


def test_image_with_wilson_extents_of_none(fake):
    """A state image whose Wilson loop has no extent, which no lattice can have set, is
    refused: the loop kernel's lines start from a link and step by the extents."""
    _run(fake, """
with Q.Lattice(sun=2, dims=(4, 4, 4, 4), max_measurements=2) as lat:
    lat.set_wilson(21, 34)
    img = lat.save_state()
    at = [i for i in range(0, 512, 4) if img[i:i + 8].tobytes() == np.array([21, 34], "<u4").tobytes()]
    assert len(at) == 1, at
    lat.load_state(img)
    for field in (0, 4):
        for value in (0, -3):
            bad = img.copy()
            bad[at[0] + field:at[0] + field + 4] = np.frombuffer(np.array([value], "<i4").tobytes(), np.uint8)
            try:
                lat.load_state(bad)
            except Q.QCDError as e:
                assert "Wilson" in str(e)
            else:
                raise SystemExit("accepted")
    lat.load_state(img)
""")


def test_batch_has_one_set_of_ranlux_tables(fake):
    """The chains of a batch share the luxury level's tables instead of each allocating
    and filling its own; they are freed once."""
    _run(fake, """
tables = "copy kind 1 bytes 253440"
chains = [((4, 4, 4, 4), 5.7, k + 1) for k in range(5)]
calls()
for _ in range(2):
    with Q.Batch(chains, sun=3, prng="RANLUX", max_measurements=2) as b:
        assert calls().count(tables) == 1
        b.init("cold")
        b.sweep("hb")
        b.sync()
calls()
with Q.Lattice(sun=3, dims=(4, 4, 4, 4), prng="RANLUX", max_measurements=2):
    assert calls().count(tables) == 1
with Q.Batch(chains, sun=3, prng="XOR128", max_measurements=2):
    assert calls().count(tables) == 0
""")


def test_autotune_times_what_will_run(fake):
    """The buckets of a batch run merged, so the tuner times merged half-steps too, and the
    choice is made on one production of the RANLUX quads; the maps it made are given back."""
    _run(fake, """
chains = [((8, 8, 8, 4), 5.7, 1), ((8, 8, 8, 6), 5.7, 2), ((6, 6, 6, 8), 5.7, 3)]
grid = lambda c: int(c.split()[1])
with Q.Batch(chains, sun=3, prng="RANLUX", max_measurements=2) as b:
    b.init("cold")
    b.sync()
    calls()
    b.sweep("or")
    merged = {grid(c) for c in calls() if c.startswith("launch")}
    assert len(merged) == 1
    b.sweep("hb")
    produce = {grid(c) for c in calls() if c.startswith("launch")} - merged
    b.autotune(repeats=2)
    seen = [grid(c) for c in calls() if c.startswith("launch")]
    assert seen.count(next(iter(merged))) >= 2 * 3, seen
    assert sum(seen.count(g) for g in produce) <= 1, (produce, seen)
    b.sweep("or")
    assert {grid(c) for c in calls() if c.startswith("launch")} == merged   # every time is equal here: the first choice
""")


def test_flow_parameters_are_uploaded_by_a_plain_copy(fake):
    """Parameters come from a caller's array that is often new; a plain copy stages it,
    and is waited for before the flow's stream packs it."""
    _run(fake, """
from qcdgpu_amd import flow as QF
f = QF.Flow(dims=(4, 4, 4, 4), layers=2, max_batch=2)
p = np.zeros(f.param_count(), np.float32)
calls()
f.set_params(p)
seen = calls()
at = seen.index("copy kind 1 bytes %d" % p.nbytes)
assert seen[at + 1].startswith("wait on 0") or seen[at + 1] == "wait on ", seen
assert seen[at + 2].startswith("launch"), seen
""")
