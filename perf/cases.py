"""The workloads this framework's speed is measured on.

Each case is one unit of work a user's program has the framework do, through
the package's public classes (qcdgpu_amd.Lattice, Batch, flow.Flow):

  run      a Monte Carlo run: `steps` measurement cycles of heatbath and
           overrelaxation sweeps replayed from the captured graph, then the
           plaquette and Polyakov records and the links are read
  loop     the host program's loop with everything a parameter file can turn
           on: eager heatbath sweeps, after each the plaquette, Polyakov loop
           and its slices, F_munu and the Wilson loop, with or without the
           twisted boundary
  observe  a stored configuration is loaded and every observable measured
  batch    an ensemble of chains of several sizes and couplings, all updated
           by each launch; every chain's records are read
  sample   independent configurations drawn from the learned flow, with their
           log density and action
  evaluate log density and action of given configurations (the inverse flow)
  learned  chains that alternate a heatbath sweep and a learned Metropolis
           sweep, measured every step
  train    the flow's training objective and its gradient on given batches

A lattice's links stay on the card between calls; a pass that ends a run
reads them back, as a user who stores the configuration does.  Ensembles and
the largest lattice return their records alone: their links are gigabytes
that such a program leaves where they are.
"""
import math

import numpy as np
import torch

import qcdgpu_amd as Q
from qcdgpu_amd import flow as QF


def listed():
    return [
        # Small lattice, where launches and their latency are the cost: SU(2)
        # 8^4 in FP64, beta 2.3, RANLUX, 1 heatbath + 3 overrelaxation sweeps
        # per measured step.
        dict(name="su2_8x8x8x8_fp64", kind="run", sun=2, n1=8, n2=8, n3=8, n4=8, precision="fp64", storage=4,
             prng="RANLUX", lux=3, beta=2.3, n_hb=1, n_or=3, steps=200, links=True),
        # The finite-temperature lattice of the headline figure: 500 steps of
        # 1 heatbath + 4 overrelaxation sweeps.
        dict(name="su3_32x32x32x8_fp32", kind="run", sun=3, n1=32, n2=32, n3=32, n4=8, precision="fp32", storage=18,
             prng="XOR128", lux=3, beta=5.9, n_hb=1, n_or=4, steps=500, links=True),
        # The same observables with FP64 links on a lattice whose extents are
        # no powers of two.
        dict(name="su3_24x24x24x12_fp64", kind="run", sun=3, n1=24, n2=24, n3=24, n4=12, precision="fp64", storage=18,
             prng="XOR128", lux=3, beta=6.0, n_hb=1, n_or=4, steps=100, links=True),
        # Heatbath only, as the reference runs it, with its generator and its
        # two-row link storage on ragged extents.
        dict(name="su3_20x12x28x10_rows2", kind="run", sun=3, n1=20, n2=12, n3=28, n4=10, precision="fp32", storage=12,
             prng="RANLUX", lux=3, beta=5.7, n_hb=1, n_or=0, steps=100, links=True),
        # The largest single lattice: 64^4, 1.2e9 stored reals.
        dict(name="su3_64x64x64x64_fp32", kind="run", sun=3, n1=64, n2=64, n3=64, n4=64, precision="fp32", storage=18,
             prng="XOR128", lux=3, beta=6.0, n_hb=1, n_or=4, steps=5, links=False),
        # The reference's parameter file: SU(2) 16^4, beta 3.5, twisted in Y
        # by PHI = 3, F_munu, Wilson loop 10 x 3, RANLUX; ten measured sweeps.
        dict(name="su2_16x16x16x16_twisted", kind="loop", sun=2, n1=16, n2=16, n3=16, n4=16, precision="fp32",
             storage=4, prng="RANLUX", lux=3, beta=3.5, phi=3.0, R=10, T=3, steps=10),
        # Every observable of a stored SU(3) configuration, the Wilson loop
        # at the host program's default 7 x 2.
        dict(name="su3_16x16x16x16_observe", kind="observe", sun=3, n1=16, n2=16, n3=16, n4=16, precision="fp32",
             storage=18, R=7, T=2),
        # Finite-temperature scan: 96 chains, N_s in {12,16,20,24}, N_t in
        # {4,6,8}, beta 5.5 to 6.2, RANLUX streams.
        dict(name="su3_batch_96", kind="batch", sun=3, chains=96, ns_min=12, ns_max=24, ns_step=4, precision="fp32",
             storage=18, prng="RANLUX", lux=3, beta0=5.5, beta1=6.2, n_hb=1, n_or=4, steps=20),
        # Independent proposals from the flow in batches of 64 configurations.
        dict(name="flow_sample_8x8x8x4", kind="sample", n1=8, n2=8, n3=8, n4=4, layers=8, bins=4, batch=64, beta=2.2),
        # The density of one chain state (the other direction, batch of 1).
        dict(name="flow_evaluate_1", kind="evaluate", n1=8, n2=8, n3=8, n4=4, layers=8, bins=4, batch=1, beta=2.2),
        # Heatbath + learned sweep chain at 8^3 x 4, beta 2.2.
        dict(name="flow_chain_8x8x8x4", kind="learned", n1=8, n2=8, n3=8, n4=4, layers=8, bins=4, beta=2.2, steps=50),
        # Loss and gradient of two batches of 16 configurations (forward and
        # backward through every layer; the optimiser's element-wise step is
        # left to the caller, since it scales vanishing components up).
        dict(name="flow_train_16", kind="train", n1=8, n2=8, n3=8, n4=4, layers=8, bins=4, batch=16, steps=2),
    ]


# ------------------------------------------------------------------ drawing
def _even(rng, lo, hi):
    return 2 * int(round(math.exp(rng.uniform(math.log(lo / 2), math.log(hi / 2)))))


def _dims(rng, lo, hi, cap):
    while True:
        d = [_even(rng, lo, hi) for _ in range(4)]
        if d[0] * d[1] * d[2] * d[3] <= cap:
            return dict(n1=d[0], n2=d[1], n3=d[2], n4=d[3])


def draw(rng):
    kind = rng.choice(["run", "run", "run", "loop", "observe", "batch", "sample", "evaluate", "learned", "train"])
    if kind in ("run", "loop", "observe"):
        sun = rng.choice([2, 3, 3])
        c = dict(kind=kind, sun=sun, precision=rng.choice(["fp32", "fp32", "fp64"]),
                 storage=4 if sun == 2 else rng.choice([18, 18, 12]))
        c.update(_dims(rng, 4, 40, 1 << 19 if kind == "run" else 1 << 17))
        V = c["n1"] * c["n2"] * c["n3"] * c["n4"]
        if kind != "observe":
            c.update(prng=rng.choice(["XOR128", "XOR128", "RANLUX", "PM"]), lux=rng.randrange(5),
                     beta=round(rng.uniform(2.0, 3.5) if sun == 2 else rng.uniform(5.5, 6.2), 3))
        if kind == "run":
            steps = max(4, min(100, (1 << 22) // V))
            c.update(n_hb=1, n_or=rng.choice([0, 1, 3, 4]), steps=rng.randint(max(2, steps // 2), steps), links=True)
        else:
            m = min(c["n1"], c["n2"], c["n3"], c["n4"])
            c.update(R=rng.randint(1, max(1, min(10, m))), T=rng.randint(1, max(1, min(4, m))))
        if kind == "loop":
            c.update(phi=rng.choice([0.0, round(rng.uniform(0.1, 3.1), 3)]), steps=rng.randint(2, 10))
        return c
    if kind == "batch":
        sun = rng.choice([2, 3, 3])
        lo = _even(rng, 4, 12)
        return dict(kind=kind, sun=sun, chains=rng.randint(2, 64), ns_min=lo, ns_max=lo + 2 * rng.randint(0, 4), ns_step=2,
                    precision=rng.choice(["fp32", "fp32", "fp64"]), storage=4 if sun == 2 else 18,
                    prng=rng.choice(["RANLUX", "RANLUX", "XOR128", "PM"]), lux=rng.randrange(5),
                    beta0=2.0 if sun == 2 else 5.5, beta1=2.8 if sun == 2 else 6.2, n_hb=1, n_or=rng.choice([0, 1, 4]),
                    steps=rng.randint(4, 12))
    c = dict(kind=kind, layers=rng.choice([4, 8, 8, 12]), bins=rng.randint(2, 5))
    c.update(_dims(rng, 4, 12, 1 << 12))
    V = c["n1"] * c["n2"] * c["n3"] * c["n4"]
    if kind == "learned":
        c.update(beta=round(rng.uniform(1.8, 2.5), 2), steps=rng.randint(5, 40))
    elif kind == "train":
        c.update(batch=rng.randint(1, max(1, min(32, (1 << 15) // V))), steps=rng.randint(1, 3))
    else:
        c.update(beta=round(rng.uniform(1.8, 2.5), 2), batch=rng.randint(1, max(1, min(96, (1 << 17) // V))))
    return c


# ------------------------------------------------------------------ inputs
def _dims_of(case):
    return (case["n1"], case["n2"], case["n3"], case["n4"])


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _series(seed):
    return 1 + int(np.random.default_rng(seed).integers(1, 1 << 30))


def _lattice(case, seed, records):
    return Q.Lattice(sun=case["sun"], dims=_dims_of(case), beta=case["beta"], precision=case["precision"],
                     storage_reals=case["storage"], prng=case["prng"], ranlux_luxury=case["lux"],
                     randseries=_series(seed), max_measurements=records)


def _stored_links(case, seed):
    """A configuration as read from disk: random SU(N) links exp(i H) of
    moderate roughness, rounded to the lattice's precision; canonical layout
    (V, 4, N, N, 2) in float64."""
    N, V = case["sun"], int(np.prod(_dims_of(case)))
    a = torch.randn((V, 4, N, N, 2), generator=_rng(seed), device="cuda", dtype=torch.float64)
    h = torch.view_as_complex(a) * 0.35
    u = torch.linalg.matrix_exp(h - h.mH)
    u = u / torch.linalg.det(u)[..., None, None] ** (1.0 / N)
    u = torch.view_as_real(u)
    if case["precision"] == "fp32":
        u = u.float().double()
    if N == 2:   # a quaternion: the second row is fixed by the first
        u[..., 1, 0, 0], u[..., 1, 0, 1] = -u[..., 0, 1, 0], u[..., 0, 1, 1]
        u[..., 1, 1, 0], u[..., 1, 1, 1] = u[..., 0, 0, 0], -u[..., 0, 0, 1]
    elif case["storage"] == 12:   # two stored rows: the third is their cross product
        c = torch.view_as_complex(u)
        c[..., 2, :] = torch.linalg.cross(c[..., 0, :], c[..., 1, :]).conj()
    return u


def _chains(case, seed):
    r = np.random.default_rng(54)   # the sizes; the streams are the seed's
    ns = r.choice(np.arange(case["ns_min"], case["ns_max"] + 1, case["ns_step"]), size=case["chains"])
    nt = r.choice([4, 6, 8], size=case["chains"])
    k = max(1, case["chains"] - 1)
    return [((int(s),) * 3 + (int(t),), case["beta0"] + (case["beta1"] - case["beta0"]) * i / k, 1000 + seed % 100000 + i)
            for i, (s, t) in enumerate(zip(ns, nt))]


def _flow_params(case, seed):
    """Parameters of the size a trained flow has, float32, the flat layout of
    Flow.set_params: per layer W1 (32 x 81*8), b1, W2 (16 x 81*32), b2."""
    g = _rng(seed)
    out = []
    for _ in range(case["layers"]):
        for n, s in ((QF.W1N, 1 / math.sqrt(QF.STENCIL * 5)), (QF.HIDDEN, 0.1), (QF.W2N, 0.006), (QF.COUT, 0.1)):
            out.append(torch.randn(n, generator=g, device="cuda") * s)
    return torch.cat(out)


def _quaternions(case, seed, count):
    """`count` SU(2) configurations (count, 4, V, 4), unit quaternions about
    as ordered as the heatbath's at these couplings, float32."""
    V = int(np.prod(_dims_of(case)))
    q = torch.randn((count, 4, V, 4), generator=_rng(seed), device="cuda") * 0.45
    q[..., 0] += 1.0
    return q / q.norm(dim=-1, keepdim=True)


def _flow(case, seed, batch):
    f = QF.Flow(dims=_dims_of(case), layers=case["layers"], bins=case["bins"], max_batch=batch)
    f.set_params(_flow_params(case, seed).cpu().numpy())
    return f


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "loop"):
        lat = _lattice(case, seed, case["steps"] + 4)
        lat.prng_init()
        lat.init("cold")
        for _ in range(3):   # off the cold start
            lat.sweep("hb")
        if kind == "run":
            lat.capture_cycle(n_hb=case["n_hb"], n_or=case["n_or"])
        else:
            lat.set_wilson(case["R"], case["T"])
            if case["phi"]:
                lat.set_twist(case["phi"])
        lat.sync()
        return dict(case=case, lat=lat)
    if kind == "observe":
        links = _stored_links(case, seed).cpu().numpy()
        lat = Q.Lattice(sun=case["sun"], dims=_dims_of(case), precision=case["precision"], storage_reals=case["storage"],
                        max_measurements=4)
        lat.set_wilson(case["R"], case["T"])
        return dict(case=case, lat=lat, links=links)
    if kind == "batch":
        b = Q.Batch(_chains(case, seed), sun=case["sun"], precision=case["precision"], storage_reals=case["storage"],
                    prng=case["prng"], ranlux_luxury=case["lux"], max_measurements=case["steps"] + 4)
        b.init("cold")
        for _ in range(3):
            b.sweep("hb")
        b.autotune(repeats=2)
        b.capture_cycle(n_hb=case["n_hb"], n_or=case["n_or"])
        b.sync()
        return dict(case=case, batch=b)
    if kind == "sample":
        return dict(case=case, flow=_flow(case, seed, case["batch"]), seed=_series(seed))
    if kind == "evaluate":
        return dict(case=case, flow=_flow(case, seed, case["batch"]),
                    links=_quaternions(case, seed + 1, case["batch"]).cpu().numpy())
    if kind == "learned":
        lat = Q.Lattice(sun=2, dims=_dims_of(case), beta=case["beta"], precision="fp32", prng="XOR128",
                        randseries=_series(seed), max_measurements=case["steps"] + 4)
        flow = _flow(case, seed, 1)
        lat.set_wilson(2, 2)
        lat.prng_init()
        lat.init("hot")
        for _ in range(10):
            lat.sweep("hb")
        flow.imh_seed(_series(seed) << 32)
        lat.graph_begin()   # one step, recorded and replayed
        lat.sweep("hb")
        flow.imh_sweep_next(lat, case["beta"])
        lat.measure(wilson=True)
        lat.graph_end()
        lat.sync()
        return dict(case=case, lat=lat, flow=flow)
    data = _quaternions(case, seed + 1, case["batch"] * case["steps"]).cpu().numpy()
    return dict(case=case, flow=_flow(case, seed, case["batch"]), data=data)


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        lat = state["lat"]
        lat.reset_measurements()
        lat.launch_cycle(case["steps"])
        plq, poly = lat.raw_measurements()
        return dict(plaquette=plq, polyakov=poly, links=lat.export_links()) if case["links"] else \
            dict(plaquette=plq, polyakov=poly)
    if kind == "loop":
        lat = state["lat"]
        lat.reset_measurements()
        for _ in range(case["steps"]):
            lat.sweep("hb")
            lat.measure(wilson=True, polyakov_slices=True, fmunu="H")
        plq, poly = lat.raw_measurements()
        return dict(plaquette=plq, polyakov=poly, wilson=lat.wilson_measurements(raw=True), fmunu=lat.fmunu(raw=True),
                    slices=lat.polyakov_slices(raw=True), links=lat.export_links())
    if kind == "observe":
        lat = state["lat"]
        lat.import_links(state["links"])
        lat.reset_measurements()
        lat.measure(wilson=True, polyakov_slices=True, fmunu="H", action_slices=True)
        plq, poly = lat.raw_measurements()
        return dict(plaquette=plq, polyakov=poly, wilson=lat.wilson_measurements(raw=True), fmunu=lat.fmunu(raw=True),
                    slices=lat.polyakov_slices(raw=True), action=lat.action_slices(raw=True))
    if kind == "batch":
        b = state["batch"]
        chains = [b.chain(i) for i in range(case["chains"])]
        for c in chains:
            c.reset_measurements()
        b.launch_cycle(case["steps"])
        b.sync()
        m = [c.raw_measurements() for c in chains]
        return dict(plaquette=np.stack([x[0] for x in m]), polyakov=np.stack([x[1] for x in m]))
    if kind == "sample":
        links, logq, action = state["flow"].sample(state["seed"], case["batch"], case["beta"])
        return dict(links=links, logq=logq, action=action)
    if kind == "evaluate":
        logq, action = state["flow"].evaluate(state["links"], case["beta"])
        return dict(logq=logq, action=action)
    if kind == "learned":
        lat = state["lat"]
        lat.reset_measurements()
        lat.launch_cycle(case["steps"])
        plq, poly = lat.raw_measurements()
        accepted, proposed = state["flow"].imh_counts()
        return dict(plaquette=plq, polyakov=poly, wilson=lat.wilson_measurements(raw=True), links=lat.export_links(),
                    accepted=accepted, proposed=proposed)
    flow, B = state["flow"], case["batch"]
    out = [flow.train_grad(state["data"][k * B:(k + 1) * B]) for k in range(case["steps"])]
    return dict(losses=np.array([o[0] for o in out]), grads=[o[1] for o in out])


# ------------------------------------------------------------------ work
def work(case):
    """Bytes: a half-step reads the eight links each updated link's staples
    and update need once per updated link and writes the link (the updates of
    a half-step depend on the whole one before it), generator states are read
    and written once per heatbath half-step; measurements read the links
    once.  Flops: SU(3) staple 2000, update 900, plaquette 6 x 220 per site;
    an eighth of that for SU(2)."""
    kind = case["kind"]
    if kind in ("run", "loop", "observe", "batch"):
        s = case["storage"] * (4 if case["precision"] == "fp32" else 8)
        f = 1.0 if case["sun"] == 3 else 0.125
        if kind == "batch":
            V = float(sum(int(np.prod(d)) for d, _, _ in _chains(case, 1)))
        else:
            V = float(np.prod(_dims_of(case)))
        if kind == "observe":
            return dict(bytes=4 * V * s * 2, flops=V * f * (6 * 220 + 3 * 420 + (6 * case["R"] + 4 * case["T"]) * 200))
        r = 112 if case["prng"] == "RANLUX" else 16
        if kind == "loop":
            step = 4 * V * (9 * s + 2 * r) + 4 * V * s
            fl = V * f * (4 * 2900 + 6 * 220 + 3 * 420 + (6 * case["R"] + 4 * case["T"]) * 200)
            return dict(bytes=case["steps"] * step, flops=case["steps"] * fl)
        step = 4 * V * (case["n_hb"] * (9 * s + 2 * r) + case["n_or"] * 9 * s) + V * s
        fl = V * f * (4 * 2900 * (case["n_hb"] + case["n_or"]) + 6 * 72)
        return dict(bytes=case["steps"] * step, flops=case["steps"] * fl)
    V = float(np.prod(_dims_of(case)))
    conv = 2 * V * (648 * 32 + 2592 * 16) * case["layers"]
    par = 2.0 * QF.LAYER_PARAMS * case["layers"]
    cfg = V * 4 * 16
    if kind == "learned":
        return dict(bytes=case["steps"] * (par + 2 * cfg + 4 * V * (9 * 16 + 32)), flops=case["steps"] * conv)
    if kind == "train":
        return dict(bytes=case["steps"] * (case["batch"] * cfg + 3 * par), flops=case["steps"] * 3 * case["batch"] * conv)
    return dict(bytes=case["batch"] * cfg + par, flops=case["batch"] * conv)


# ------------------------------------------------------------------ 64-bit values
def exact(case, seed):
    """Monte Carlo chains (run, loop, batch, learned) have no 64-bit value to
    compare with: their accept decisions amplify any rounding to another,
    equally valid, trajectory."""
    with torch.no_grad():
        if case["kind"] == "observe":
            return _exact_observe(case, _stored_links(case, seed))
        if case["kind"] == "sample":
            return _exact_sample(case, seed)
        if case["kind"] == "evaluate":
            return _exact_evaluate(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None


_AXIS = {0: 0, 1: 3, 2: 2, 3: 1}   # direction -> axis of a (x, t, z, y) array


def _exact_observe(case, u):
    n1, n2, n3, n4 = _dims_of(case)
    N = case["sun"]
    U = torch.view_as_complex(u).reshape(n1, n4, n3, n2, 4, N, N)
    L = [U[..., d, :, :] for d in range(4)]

    def sh(a, d, k=1):
        return torch.roll(a, -k, _AXIS[d])

    def tr(a):
        return a.diagonal(dim1=-2, dim2=-1).sum(-1)

    def line(d, k):
        p = L[d]
        for j in range(1, k):
            p = p @ sh(L[d], d, j)
        return p

    P, spat, temp = {}, 0, 0
    for a in range(3):
        for b in range(a + 1, 4):
            P[a, b] = L[a] @ sh(L[b], a) @ sh(L[a], b).mH @ L[b].mH
            if b == 3:
                temp = temp + tr(P[a, b]).real
            else:
                spat = spat + tr(P[a, b]).real
    pol = tr(line(3, n4)[:, 0])   # (x, z, y)
    a2 = pol.abs() ** 2
    R, T = case["R"], case["T"]
    B, w = line(3, T), 0
    for d in range(3):
        E = line(d, R)
        w = w + tr(B @ sh(E, 3, T) @ sh(B, d, R).mH @ E.mH).real.sum()
    f = []
    for gen in range(2):
        for pl in ((0, 1), (0, 2), (1, 2)):
            p = P[pl]
            if gen == 0:
                z = p[..., 0, 0] - p[..., 1, 1]
            elif N == 3:
                z = (p[..., 0, 0] + p[..., 1, 1] - 2 * p[..., 2, 2]) / math.sqrt(3.0)
            else:
                z = 1j * (p[..., 0, 1] - p[..., 1, 0])
            z = z.sum()
            f.append(0.5 * z.imag + (0 if N == 2 else -0.5j * z.real))
    act = torch.stack([spat, temp], -1)   # (x, t, z, y, 2)

    def host(a):
        return a.cpu().numpy()[None]

    return dict(plaquette=host(torch.stack([spat.sum(), temp.sum()])),
                polyakov=host(torch.stack([pol.real.sum(), pol.imag.sum(), a2.sum(), (a2 ** 2).sum()])),
                wilson=host(w), fmunu=host(torch.stack([torch.as_tensor(v, dtype=torch.complex128, device=u.device)
                                                        for v in f]).reshape(2, 3)),
                slices=dict(x=host(pol.sum((1, 2))), y=host(pol.sum((0, 1))), z=host(pol.sum((0, 2)))),
                action=dict(x=host(act.sum((1, 2, 3))), y=host(act.sum((0, 1, 2))), z=host(act.sum((0, 1, 3)))))


def _qmul(a, b):
    a0, av = a[..., :1], a[..., 1:]
    b0, bv = b[..., :1], b[..., 1:]
    return torch.cat([a0 * b0 - (av * bv).sum(-1, keepdim=True), a0 * bv + b0 * av - torch.linalg.cross(av, bv)], -1)


def _qdag(a):
    return torch.cat([a[..., :1], -a[..., 1:]], -1)


class _Flow64:
    """The flow of flow.py's documentation, in plain 64-bit torch."""

    def __init__(self, case):
        self.n = _dims_of(case)
        self.K = case["bins"]
        n1, n2, n3, n4 = self.n
        self.V = n1 * n2 * n3 * n4
        x, t, z, y = torch.meshgrid(*[torch.arange(k, device="cuda") for k in (n1, n4, n3, n2)], indexing="ij")
        self.c = [x.reshape(-1), y.reshape(-1), z.reshape(-1), t.reshape(-1)]

    def at(self, off):
        """Site index of x + off for every x."""
        e = [(c + o) % n for c, o, n in zip(self.c, off, self.n)]
        return e[1] + self.n[1] * (e[2] + self.n[2] * (e[3] + self.n[3] * e[0]))

    def step(self, d, k=1):
        return self.at([k if j == d else 0 for j in range(4)])

    def plaq(self, L, a, b):
        return _qmul(_qmul(L[:, a], L[:, b][:, self.step(a)]), _qdag(_qmul(L[:, b], L[:, a][:, self.step(b)])))[..., 0]

    def staple(self, L, mu):
        A = 0
        for nu in range(4):
            if nu == mu:
                continue
            f = _qmul(_qmul(L[:, nu][:, self.step(mu)], _qdag(L[:, mu][:, self.step(nu)])), _qdag(L[:, nu]))
            m = self.step(nu, -1)
            b = _qmul(_qdag(_qmul(L[:, mu], L[:, nu][:, self.step(mu)])), L[:, nu])[:, m]
            A = A + f + b
        return A

    def conv(self, x, w, b):
        out = b
        k = 0
        for ox in (-1, 0, 1):
            for oy in (-1, 0, 1):
                for oz in (-1, 0, 1):
                    for ot in (-1, 0, 1):
                        out = out + x[:, self.at((ox, oy, oz, ot))] @ w[:, k].T
                        k += 1
        return out

    def spline(self, r, v, inverse):
        K, eps = self.K, 1e-3
        w = math.pi * (eps + (1 - K * eps) * torch.softmax(r[..., :K], -1))
        h = math.pi * (eps + (1 - K * eps) * torch.softmax(r[..., K:2 * K], -1))
        d = eps + (1 - eps) * torch.nn.functional.softplus(r[..., 2 * K:3 * K + 1]) / math.log(2.0)
        xk, yk = torch.cumsum(w, -1) - w, torch.cumsum(h, -1) - h
        k = ((yk if inverse else xk)[..., 1:] <= v[..., None]).sum(-1, keepdim=True)
        g = lambda a, j: torch.gather(a, -1, j)[..., 0]  # noqa: E731
        x0, y0, w, h, d0, d1 = g(xk, k), g(yk, k), g(w, k), g(h, k), g(d, k), g(d, k + 1)
        s = h / w
        if inverse:
            dy, dd = v - y0, d1 + d0 - 2 * s
            a, b, c = h * (s - d0) + dy * dd, h * d0 - dy * dd, -s * dy
            xi = 2 * c / (-b - torch.sqrt((b * b - 4 * a * c).clamp(min=0)))
        else:
            xi = (v - x0) / w
        xi = xi.clamp(0, 1)
        den = s + (d1 + d0 - 2 * s) * xi * (1 - xi)
        num = s * s * (d1 * xi * xi + 2 * s * xi * (1 - xi) + d0 * (1 - xi) ** 2)
        out = x0 + w * xi if inverse else y0 + h * (s * xi * xi + d0 * xi * (1 - xi)) / den
        return out, torch.log(num) - 2 * torch.log(den)

    def layer(self, L, l, params, inverse):
        """(links, log J per configuration) of layer l."""
        mu, par = l % 4, (l // 4) % 2
        o = params[l * QF.LAYER_PARAMS:(l + 1) * QF.LAYER_PARAMS]
        w1, b1, w2, b2 = torch.split(o, [QF.W1N, QF.HIDDEN, QF.W2N, QF.COUT])
        on = (sum(self.c[d] for d in range(4) if d != mu) + par) % 2 == 0
        A = self.staple(L, mu)
        k = A.norm(dim=-1)
        z = torch.zeros_like(k)
        pl = [self.plaq(L, a, b) for a in range(4) for b in range(a + 1, 4) if mu not in (a, b)]
        x = torch.stack([k / 6 * on] + pl + [z + on, z, z, z], -1)
        hid = torch.tanh(self.conv(x, w1.reshape(QF.HIDDEN, QF.STENCIL, -1), b1))
        r = self.conv(hid, w2.reshape(QF.COUT, QF.STENCIL, -1), b2)
        Vq = A / k[..., None]
        W = _qmul(L[:, mu], Vq)
        sn = W[..., 1:].norm(dim=-1)
        th = torch.atan2(sn, W[..., 0])
        th2, dlog = self.spline(r, th, inverse)
        lj = dlog + 2 * (torch.log(torch.sin(th)) - torch.log(torch.sin(th2))) * (1 if inverse else -1)
        Wn = torch.cat([torch.cos(th2)[..., None], W[..., 1:] * (torch.sin(th2) / sn)[..., None]], -1)
        new = torch.where(on[:, None], _qmul(Wn, _qdag(Vq)), L[:, mu])
        return torch.cat([L[:, :mu], new[:, None], L[:, mu + 1:]], 1), torch.where(on, lj, z).sum(-1)

    def action(self, L, beta):
        return beta * sum((1 - self.plaq(L, a, b)).sum(-1) for a in range(4) for b in range(a + 1, 4))


def _mix64(x):
    """splitmix64's output function on uint64 arrays."""
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _haar64(seed, n):
    """The flow's prior: link j's quaternion from the counter-based uniforms
    of (seed, j) by Box and Muller, normalised."""
    with np.errstate(over="ignore"):
        key = _mix64(np.array([seed], dtype=np.uint64))
        z = _mix64(key ^ _mix64(np.arange(n, dtype=np.uint64) + np.uint64(0x632BE59BD9B4E019)))
        u = []
        for _ in range(2):
            z = z + np.uint64(0x9E3779B97F4A7C15)
            x = _mix64(z)
            for bits in (x >> np.uint64(40), (x >> np.uint64(8)) & np.uint64(0xFFFFFF)):
                u.append((bits.astype(np.float64) + 0.5) * 2.0 ** -24)
    r1, r2 = np.sqrt(-2 * np.log(u[0])), np.sqrt(-2 * np.log(u[2]))
    q = np.stack([r1 * np.cos(2 * np.pi * u[1]), r1 * np.sin(2 * np.pi * u[1]), r2 * np.cos(2 * np.pi * u[3]),
                  r2 * np.sin(2 * np.pi * u[3])], -1)
    return q / np.linalg.norm(q, axis=-1, keepdims=True)


def _exact_sample(case, seed):
    f, p = _Flow64(case), _flow_params(case, seed).double()
    out = []
    q = torch.from_numpy(_haar64(_series(seed), case["batch"] * 4 * f.V)).cuda().reshape(-1, 4, f.V, 4)
    for L in q.split(16):
        lq = 0
        for l in range(case["layers"]):
            L, lj = f.layer(L, l, p, False)
            lq = lq - lj
        out.append((L, lq, f.action(L, case["beta"])))
    links, logq, action = (torch.cat(v).cpu().numpy() for v in zip(*out))
    return dict(links=links, logq=logq, action=action)


def _exact_evaluate(case, seed):
    f, p = _Flow64(case), _flow_params(case, seed).double()
    out = []
    for L in _quaternions(case, seed + 1, case["batch"]).double().split(16):
        S, lq = f.action(L, case["beta"]), 0
        for l in reversed(range(case["layers"])):
            L, lj = f.layer(L, l, p, True)
            lq = lq - lj
        out.append((lq, S))
    logq, action = (torch.cat(v).cpu().numpy() for v in zip(*out))
    return dict(logq=logq, action=action)


def _exact_train(case, seed):
    f, p = _Flow64(case), _flow_params(case, seed).double()
    data = _quaternions(case, seed + 1, case["batch"] * case["steps"]).double()
    losses, grads = [], []
    for L in data.split(case["batch"]):
        grad, loss = torch.zeros_like(p), 0.0
        for l in range(case["layers"]):   # a layer's loss depends on its own parameters only
            for part in L.split(8):
                q = p.detach().clone().requires_grad_(True)
                lj = f.layer(part, l, q, True)[1].sum()
                grad += torch.autograd.grad(lj, q)[0]
                loss += float(lj.detach())
        losses.append(loss / case["batch"])
        grads.append(grad.cpu().numpy())
    return dict(losses=np.array(losses), grads=grads)
