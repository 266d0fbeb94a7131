"""Performance cases: what a program does with a resident lattice, through glac_amd's public calls.

Each case is one `op` on one lattice:

  flow      copy the chain to the flow field and flow it, measuring before the first and after every step
            (System::copyToFlowLattice + System::flowConfiguration); observables "clover" or "super" (with Weinberg)
  sweeps    Metropolis sweeps of the chain with the plaquette after each (System::update); "save" also brings the
            chain to the host, as a program does that keeps the configuration
  ensemble  run_ensemble: sweeps, copy, unmeasured flow, plaquette and clover measurement per configuration
  measure   one measurement of a resident field: "clover", "super" or per-site "density"
  config    a configuration from the host, flowed with measurement and taken back (flowing stored configurations)
  train     standardise the held (staple, link) samples and train the learned proposal

Lattice sizes are those of the tests and the benchmark (8^3 x 16, 16^4, 24^3 x 48, 32^4, 48^3 x 96), plus ragged
ones whose extents are no multiples of the layout's blocks.  `precision` is the lattice's link storage: "fp64",
"fp32" (three rows) or "fp32c" (two rows, the third rebuilt).  What comes back from FP32 lattices (and from the FP32
training) is float32, the precision that their links carry; FP64 lattices give float64.

The fields themselves stay on the device between calls, as in a program's run: a case returns the observables that the
calls return, and the field where the program takes it to the host ("config", and "sweeps" with "save").
"""
import math

import numpy as np
import torch

import glac_amd as G
from glac_amd.proposal import init_params
from glac_amd.system import EnsembleConfig, run_ensemble

PREC = {"fp64": G.FP64, "fp32": G.FP32_LINKS, "fp32c": G.FP32_COMPRESSED}
REAL = {"fp64": 8, "fp32": 4, "fp32c": 4}
LINK_REALS = {"fp64": 18, "fp32": 18, "fp32c": 12}
NOISE = 0.44  # spread of a link around a pure gauge: plaquette about 0.6, as at beta = 6
BETA, EPS = 6.1, 0.24
THERM = 30  # sweeps from the hot start before a chain is used
# the learned proposal's standardisation: mean and deviation of the six staple features of such a chain
MEAN = np.array([41.0, 710.0, 2500.0, 45.0, 0.0, BETA], np.float32)
STD = np.array([10.0, 290.0, 2200.0, 21.0, 5.5, 1.0], np.float32)


def listed():
    return [
        # a small lattice's flow, the run of the GLAC example sizes: launches and latency count
        {"name": "flow_8x8x8x16_fp64", "op": "flow", "nx": 8, "ny": 8, "nz": 8, "nt": 16, "precision": "fp64",
         "steps": 40, "eps": 0.02, "observables": "clover"},
        # the benchmark's flow
        {"name": "flow_32x32x32x32_fp32c", "op": "flow", "nx": 32, "ny": 32, "nz": 32, "nt": 32, "precision": "fp32c",
         "steps": 10, "eps": 0.01, "observables": "clover"},
        # the plain FP64 flow at the size where it is compared with FP32
        {"name": "flow_24x24x24x48_fp64", "op": "flow", "nx": 24, "ny": 24, "nz": 24, "nt": 48, "precision": "fp64",
         "steps": 10, "eps": 0.01, "observables": "clover"},
        # extents that are no multiples of the blocks (z of 14), three stored rows, GLAC's observables with Weinberg
        {"name": "flow_super_12x10x14x18_fp32", "op": "flow", "nx": 12, "ny": 10, "nz": 14, "nt": 18,
         "precision": "fp32", "steps": 20, "eps": 0.015, "observables": "super"},
        # the largest lattice of the pipeline test
        {"name": "flow_48x48x48x96_fp32c", "op": "flow", "nx": 48, "ny": 48, "nz": 48, "nt": 96, "precision": "fp32c",
         "steps": 3, "eps": 0.02, "observables": "clover"},
        # the smallest call: one measurement of a small lattice, all launch and latency
        {"name": "measure_8x8x8x16_fp64", "op": "measure", "nx": 8, "ny": 8, "nz": 8, "nt": 16, "precision": "fp64",
         "mode": "clover"},
        # the benchmark's Metropolis chain
        {"name": "sweeps_32x32x32x32_fp32c", "op": "sweeps", "nx": 32, "ny": 32, "nz": 32, "nt": 32,
         "precision": "fp32c", "proposal": "rst", "sweeps": 10, "hits": 10, "reunit": 1, "save": False},
        # GLAC's plain FP64 chain between two stored configurations
        {"name": "sweeps_16x16x16x16_fp64", "op": "sweeps", "nx": 16, "ny": 16, "nz": 16, "nt": 16,
         "precision": "fp64", "proposal": "rst", "sweeps": 20, "hits": 10, "reunit": 1, "save": True},
        # the learned chain at the size where it is compared with the plain one
        {"name": "learned_24x24x24x48_fp32c", "op": "sweeps", "nx": 24, "ny": 24, "nz": 24, "nt": 48,
         "precision": "fp32c", "proposal": "learned", "sweeps": 10, "hits": 10, "reunit": 1, "save": False},
        # the production loop on a small lattice: every kernel under-fills the chip
        {"name": "ensemble_8x8x8x16_fp32c", "op": "ensemble", "nx": 8, "ny": 8, "nz": 8, "nt": 16,
         "precision": "fp32c", "configs": 2, "sweeps": 20, "steps": 50},
        # stored configurations flowed one after the other: host transfers count as the flow does
        {"name": "config_24x24x24x48_fp32c", "op": "config", "nx": 24, "ny": 24, "nz": 24, "nt": 48,
         "precision": "fp32c", "steps": 10, "eps": 0.02},
        # the learned proposal's training at its default batch and draws
        {"name": "train_16x16x16x16_fp32c", "op": "train", "nx": 16, "ny": 16, "nz": 16, "nt": 16,
         "precision": "fp32c", "stride": 2, "steps": 200, "batch": 4096, "draws": 4},
    ]


def _extents(rng, vmax):
    """Four even extents, the volume spread over its logarithm from 256 to vmax."""
    v = math.exp(rng.uniform(math.log(256), math.log(vmax)))
    while True:
        n = [2 * rng.randint(1, 24) for _ in range(4)]
        if 0.6 * v <= math.prod(n) <= min(1.2 * v, vmax):
            return dict(zip(("nx", "ny", "nz", "nt"), n))


def draw(rng):
    op = rng.choice(["flow", "flow", "flow", "sweeps", "sweeps", "ensemble", "measure", "config", "train"])
    c = {"op": op}
    c.update(_extents(rng, {"flow": 1 << 20, "sweeps": 1 << 20, "ensemble": 1 << 16, "measure": 1 << 20,
                            "config": 1 << 19, "train": 1 << 17}[op]))
    c["precision"] = rng.choice(["fp64", "fp32c", "fp32c", "fp32"])
    v = _volume(c)
    if op == "flow":
        most = max(1, min(40, int(2e7 / (v * (3 if c["precision"] == "fp64" else 1.5)))))
        c.update(steps=rng.randint(1, most), eps=round(rng.uniform(0.005, 0.02), 4),
                 observables=rng.choice(["clover", "clover", "super"]))
    elif op == "sweeps":
        most = max(1, min(20, int(4e6 / v)))
        learned = rng.random() < 0.35
        c.update(proposal="learned" if learned else "rst", sweeps=rng.randint(1, most), hits=rng.choice([5, 10, 10]),
                 reunit=rng.choice([1, 1, 4]), save=v <= 1 << 17 and rng.random() < 0.5)
    elif op == "ensemble":
        c.update(configs=rng.randint(1, 2), sweeps=rng.randint(5, 20), steps=rng.randint(5, 50))
    elif op == "measure":
        c.update(mode=rng.choice(["clover", "super", "density"]))
    elif op == "config":
        c.update(steps=rng.randint(1, 5), eps=round(rng.uniform(0.005, 0.02), 4))
    else:
        c.update(stride=rng.randint(1, 4), steps=rng.randint(10, 100), batch=rng.choice([1000, 2048, 4096, 5000]),
                 draws=rng.choice([2, 4, 4, 8]))
    return c


def _dims(c):
    return (c["nx"], c["ny"], c["nz"], c["nt"])


def _volume(c):
    return c["nx"] * c["ny"] * c["nz"] * c["nt"]


def _out(c, v):
    """Results in the precision of the lattice's links."""
    if isinstance(v, tuple):
        return tuple(_out(c, x) for x in v)
    return v if c["precision"] == "fp64" else np.asarray(v, dtype=np.float32)


# ---- gauge fields in plain torch: U[mu][i, j] over the (Nt, Nz, Ny, Nx) grid ------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _mul(a, b):
    return torch.stack([torch.stack([a[i, 0] * b[0, j] + a[i, 1] * b[1, j] + a[i, 2] * b[2, j] for j in range(3)])
                        for i in range(3)])


def _dag(a):
    return a.transpose(0, 1).conj()


def _unit(like):
    u = torch.zeros_like(like)
    for i in range(3):
        u[i, i] = 1
    return u


def _shift(a, mu, s):
    """a(x + s mu)"""
    return torch.roll(a, -s, dims=5 - mu)


def _exp(y, halvings=6, terms=12):
    """exp of small 3 x 3 matrices: Taylor series of y / 2^halvings, squared back."""
    y = y / 2 ** halvings
    x = _unit(y)
    for k in range(terms, 0, -1):
        x = _unit(y) + _mul(y, x) / k
    for _ in range(halvings):
        x = _mul(x, x)
    return x


def _gauge_field(c, seed):
    """Links spread around a random pure gauge: Haar-distributed links, plaquette about 0.6."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    grid = (c["nt"], c["nz"], c["ny"], c["nx"])
    m = torch.randn((3, 3) + grid, generator=gen, device=dev, dtype=torch.complex128)
    rows = []
    for i in range(2):
        r = m[i]
        for q in rows:
            r = r - q * (q.conj() * r).sum(0)
        rows.append(r / r.abs().square().sum(0).sqrt())
    rows.append(torch.stack([(rows[0][(j + 1) % 3] * rows[1][(j + 2) % 3]
                              - rows[0][(j + 2) % 3] * rows[1][(j + 1) % 3]).conj() for j in range(3)]))
    g = torch.stack(rows)
    field = []
    for mu in range(4):
        a = torch.randn((3, 3) + grid, generator=gen, device=dev, dtype=torch.complex128) * NOISE
        h = (a + _dag(a)) / 2
        h = h - _unit(h) * ((h[0, 0] + h[1, 1] + h[2, 2]) / 3)
        field.append(_mul(_mul(g, _exp(1j * h)), _dag(_shift(g, mu, 1))))
    return field


def _to_host(field):
    """The field in GLAC's host layout: (4, V, 18) doubles."""
    return np.stack([torch.view_as_real(u.permute(2, 3, 4, 5, 0, 1).contiguous()).reshape(-1, 18).cpu().numpy()
                     for u in field])


# ---- the calls -------------------------------------------------------------------------------
def prepare(case, seed):
    op, n = case["op"], _dims(case)
    lat = G.Lattice(n, PREC[case["precision"]])
    state = {"case": case, "lattice": lat}
    if op in ("flow", "measure") and _volume(case) <= 1 << 21:
        lat.upload(_to_host(_gauge_field(case, seed)))
    elif op == "config":
        state["links"] = _to_host(_gauge_field(case, seed))
    else:
        lat.hot_start(seed)
        lat.metropolis(THERM, BETA, EPS, 10, seed=seed + 1)
    if op == "sweeps" and case["proposal"] == "learned":
        # a network whose steps are about as long as a trained one's
        lat.proposal_set(init_params(seed, step=0.3), MEAN, STD)
    if op == "train":
        half = _volume(case) // 2
        lat.samples_reset(8 * -(-half // case["stride"]) * 2)
        for i in range(2):
            lat.metropolis(1, BETA, EPS, 10, seed=seed + 1, sweep_offset=THERM + i)
            lat.samples_collect(case["stride"])
        state["params"] = init_params(seed)
    state["seed"] = seed
    lat.synchronize()
    return state


def run(state):
    c, lat = state["case"], state["lattice"]
    op = c["op"]
    if op == "flow":
        lat.copy(G.FLOW, G.MAIN)
        flow = lat.flow if c["observables"] == "clover" else lat.flow_super
        return _out(c, flow(c["steps"], c["eps"]))
    if op == "sweeps":
        update = lat.metropolis_learned if c["proposal"] == "learned" else lat.metropolis
        got = update(c["sweeps"], BETA, EPS, c["hits"], reunit_every=c["reunit"], seed=state["seed"],
                     sweep_offset=1000, plaquette=True)
        return _out(c, got + (lat.download(),) if c["save"] else got)
    if op == "ensemble":
        r = run_ensemble(lat, EnsembleConfig(dims=_dims(c), beta=BETA, NTherm=0, NCf=c["configs"], NCor=c["sweeps"],
                                             NFlows=c["steps"], flowEpsilon=0.02, seed=state["seed"]),
                         thermalise=False, sweep_offset=1000)
        return _out(c, (r.plaq, r.q, r.e, r.sweep_acc))
    if op == "measure":
        measure = {"clover": lat.measure, "super": lat.measure_super, "density": lat.measure_density}[c["mode"]]
        return _out(c, measure(G.MAIN))
    if op == "config":
        lat.upload(state["links"], G.FLOW)
        got = lat.flow(c["steps"], c["eps"])
        return _out(c, got + (lat.download(G.FLOW),))
    mean, std = lat.samples_stats(BETA)
    lat.proposal_set(state["params"], mean, std)
    loss = lat.train(c["steps"], batch=c["batch"], draws=c["draws"], lr=2e-3, beta=BETA, seed=state["seed"])
    return (np.asarray(loss, dtype=np.float32),) + lat.proposal_get()


def work(case):
    """Bytes that have to move through HBM and operations in the products, per pass (a 3 x 3 complex product: 198)."""
    op, v = case["op"], _volume(case)
    real, link = REAL[case["precision"]], LINK_REALS[case["precision"]] * REAL[case["precision"]]
    stage_flops = 4 * v * (14 * 198 + 150)         # 12 staple products, U A, exp(Z) U and the exponential
    step = {"bytes": v * (24 * link + 16 * 8 * real), "flops": 3 * stage_flops}
    clover = {"bytes": 4 * v * link, "flops": 6 * v * (12 * 198 + 100)}
    if op in ("flow", "config"):
        s = case["steps"]
        w = {"bytes": s * step["bytes"] + clover["bytes"], "flops": s * step["flops"] + (s + 1) * clover["flops"]}
        if op == "config":
            w["bytes"] += 2 * 4 * v * (144 + link)
        return w
    if op == "sweeps" or op == "ensemble":
        n, hits = case["sweeps"], case.get("hits", 10)
        w = {"bytes": n * 8 * 4.5 * v * link, "flops": n * 4 * v * (12 * 198 + hits * (2 * 198 + 60))}
        if op == "ensemble":
            k = case["configs"]
            return {"bytes": k * (w["bytes"] + case["steps"] * step["bytes"] + 2 * clover["bytes"]),
                    "flops": k * (w["flops"] + case["steps"] * step["flops"] + clover["flops"])}
        w["bytes"] += n * clover["bytes"] + (4 * v * (144 + link) if case["save"] else 0)
        return w
    if op == "measure":
        return {"bytes": clover["bytes"] + (16 * v if case["mode"] == "density" else 0), "flops": clover["flops"]}
    per = 2 * 3 * 2400 + case["draws"] * 1200      # forward and backward of the network, and the draws
    return {"bytes": 8 * -(-(v // 2) // case["stride"]) * 2 * 72 + case["steps"] * case["batch"] * 144,
            "flops": case["steps"] * case["batch"] * per}


# ---- the same in 64 bits, in plain torch ---------------------------------------------------------
PLANES = [(0, 1, 2, 3), (0, 2, 3, 1), (0, 3, 1, 2)]  # (0, nu) with its dual (rho, sigma)


def _staple(u, mu):
    a = 0
    for nu in range(4):
        if nu != mu:
            a = a + _mul(_mul(_shift(u[nu], mu, 1), _dag(_shift(u[mu], nu, 1))), _dag(u[nu]))
            back = _shift(u[nu], nu, -1)
            a = a + _mul(_mul(_dag(_shift(back, mu, 1)), _dag(_shift(u[mu], nu, -1))), back)
    return a


def _traceless(m):
    """M - M^dag without its trace"""
    f = m - _dag(m)
    return f - _unit(f) * ((f[0, 0] + f[1, 1] + f[2, 2]) / 3)


def _flow_step(u, eps):
    acc = None
    for cz, ca in ((0.25, 0.0), (8 / 9, 17 / 36), (0.75, 1.0)):
        new, kept = [], []
        for mu in range(4):
            z = _traceless(_mul(u[mu], _staple(u, mu))) * -0.5
            y = cz * eps * z
            if acc is not None:
                y = y - (ca * eps if cz == 8 / 9 else 1.0) * acc[mu]
            new.append(_mul(_exp(y), u[mu]))
            kept.append(z if acc is None else y)
        u, acc = new, kept
    return u


def _clover(u, mu, nu):
    um, un = _shift(u[mu], mu, -1), _shift(u[nu], nu, -1)
    l1 = _mul(_mul(u[mu], _shift(u[nu], mu, 1)), _dag(_mul(u[nu], _shift(u[mu], nu, 1))))
    l2 = _mul(_mul(u[mu], _dag(_shift(un, mu, 1))), _mul(_dag(_shift(u[mu], nu, -1)), un))
    corner_mu, corner_nu = _shift(um, nu, -1), _shift(un, mu, -1)
    l3 = _mul(_dag(_mul(corner_nu, um)), _mul(corner_mu, un))
    l4 = _mul(_mul(_dag(um), _shift(u[nu], mu, -1)), _mul(_shift(um, nu, 1), _dag(u[nu])))
    return l1, _traceless(l1 - l2 + l3 - l4)


def _retr(a, b):
    return sum((a[i, k] * b[k, i]).real for i in range(3) for k in range(3))


def _measure(u, mode):
    """(plaq, E_raw, Q, [W,] Q(t), [W(t)]) or, for "density", (q(x), e(x), plaq, E_raw, Q)"""
    v = u[0][0, 0].numel()
    plaq, e, q, f = 0.0, 0, 0, {}
    for m0, n0, m1, n1 in PLANES:
        (p1, f1), (p2, f2) = _clover(u, m0, n0), _clover(u, m1, n1)
        plaq += float(sum((p[i, i].real).sum() for p in (p1, p2) for i in range(3)))
        e = e + _retr(f1, f1) + _retr(f2, f2)
        q = q - _retr(f1, f2)
        f[m0, n0], f[m1, n1] = f1, f2
    q = q / (256 * math.pi ** 2)
    plaq, e_raw, total = plaq / (18 * v), float(e.sum()) / v, float(q.sum())
    if mode == "density":
        return q.reshape(-1).cpu().numpy(), e.reshape(-1).cpu().numpy(), plaq, e_raw, total
    q_t = q.sum((1, 2, 3)).cpu().numpy()
    if mode == "clover":
        return plaq, e_raw, total, q_t
    tensor = lambda a, b: f[a, b] if (a, b) in f else -f[b, a]  # noqa: E731
    w = 0
    for _, nu, rho, sigma in PLANES:
        for lam in range(1, 4):
            if lam != nu:
                w = w - _retr(_mul(tensor(0, lam), tensor(nu, lam)), f[rho, sigma])
    w_t = (w.sum((1, 2, 3)) * (128 / (3 * 16 ** 3))).cpu().numpy()
    return plaq, e_raw, total, float(w_t.sum()), q_t, w_t


def exact(case, seed):
    """What run() returns for fields made in torch.  Markov chains and the training follow random streams and
    accept/reject decisions in the lattice's own precision: they have no such value."""
    op = case["op"]
    if op not in ("flow", "measure", "config") or _volume(case) * case.get("steps", 1) > 12 << 20:
        return None
    u = _gauge_field(case, seed)
    if op == "measure":
        return _measure(u, case["mode"])
    mode = case.get("observables", "clover")
    rows = [_measure(u, mode)]
    for _ in range(case["steps"]):
        u = _flow_step(u, case["eps"])
        rows.append(_measure(u, mode))
    got = tuple(np.array(col) for col in zip(*rows))
    return got + (_to_host(u),) if op == "config" else got
