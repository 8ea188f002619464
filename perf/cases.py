"""Workloads of the spring-block dynamics, with their exact counterparts.

A case is a dict of plain values; `prepare(case, seed)` builds what a user's
program holds before a call (systems on the GPU, a stored configuration),
`run(state)` is one pass through the public entry points, and
`exact(case, seed)` is what the first pass returns, evaluated with torch in
float64 without this package (its own pcg32, landscape, forces, Verlet steps,
stop rule and protocol, and autograd for the gradients).

Kinds of cases:

* steps        a single system stepped by a script that reads it between calls
* protocol     a single system through the quasistatic loop of the examples
               (quench, elastic step, kick + minimise) as Python calls,
               restarted from a stored configuration
* quasistatic  the same protocol for a batch of replicas on the device
* flow         a batch of replicas in flowSteps / timeSteps
* longrange    a batch of long-range chains with random forcing
* ragged       a set of systems of mixed classes and sizes, same protocol
* adjoint      differentiable runs of a batch, forward and backward
"""

import math

import numpy as np
import torch

import frictionqpotspringblock_amd as fq
from frictionqpotspringblock_amd import adjoint
from frictionqpotspringblock_amd.batch import Batch
from frictionqpotspringblock_amd.ragged import Ragged

EPS = 1e-3
DT = 0.1
ETA = 2.0 * math.sqrt(3.0) / 10.0
OFFSET = -100.0

# interaction -> constructor arguments
INTERACTIONS = {
    "Laplace1d": dict(k_interactions=1.0),
    "Quartic1d": dict(a1=1.0, a2=5.0),
    "QuarticGradient1d": dict(k2=1.0, k4=0.5),
    "LongRange1d": dict(k_interactions=1.0, alpha=1.0),
    "Laplace2d": dict(k_interactions=1.0),
}
# (potential, interaction) -> class of a single system
SINGLE = {
    ("Cuspy", "Laplace1d"): fq.Line1d.System_Cuspy_Laplace,
    ("SemiSmooth", "Laplace1d"): fq.Line1d.System_SemiSmooth_Laplace,
    ("Smooth", "Laplace1d"): fq.Line1d.System_Smooth_Laplace,
    ("Cuspy", "Quartic1d"): fq.Line1d.System_Cuspy_Quartic,
    ("Cuspy", "LongRange1d"): fq.Line1d.System_Cuspy_LongRange,
    ("Cuspy", "Laplace2d"): fq.Line2d.System_Cuspy_Laplace,
}
CLASSES = [("Cuspy", "Laplace1d"), ("SemiSmooth", "Laplace1d"), ("Smooth", "Laplace1d"), ("Cuspy", "Quartic1d"),
           ("SemiSmooth", "Quartic1d"), ("Smooth", "Quartic1d"), ("Cuspy", "QuarticGradient1d")]


def listed():
    return [
        # a script that advances one chain a few steps at a time and looks at
        # it in between (the examples' chain of 1000)
        dict(name="steps-1000", kind="steps", potential="Cuspy", interactions="Laplace1d", rows=1000, cols=1, n=20),
        # the examples' quasistatic loop on one chain of 1024
        dict(name="protocol-1024", kind="protocol", potential="Cuspy", interactions="Laplace1d", rows=1024, cols=1,
             events=5),
        # the same with long-range interactions (the examples' chain)
        dict(name="protocol-longrange-1000", kind="protocol", potential="Cuspy", interactions="LongRange1d", rows=1000,
             cols=1, events=3),
        # the examples' 50 x 50 lattice as an ensemble
        dict(name="quasistatic-50x50", kind="quasistatic", potential="Cuspy", interactions="Laplace2d", rows=50,
             cols=50, replicas=100, events=3),
        # an ensemble of 1024 chains of 1024
        dict(name="quasistatic-1024x1024", kind="quasistatic", potential="Cuspy", interactions="Laplace1d", rows=1024,
             cols=1, replicas=1024, events=5),
        # an ensemble of another class, odd sizes
        dict(name="quasistatic-semismooth", kind="quasistatic", potential="SemiSmooth", interactions="Quartic1d",
             rows=1537, cols=1, replicas=200, events=3),
        # the batched flow: 1024 chains of 4096 in blocks of 1000 slow steps
        dict(name="flow-1024x4096", kind="flow", potential="Cuspy", interactions="Laplace1d", rows=4096, cols=1,
             replicas=1024, n=1000, v_frame=1e-3, load=0.0),
        # steady sliding: wells change all the time and the windows (of 100
        # yield positions) move along
        dict(name="flow-sliding", kind="flow", potential="Cuspy", interactions="Laplace1d", rows=1999, cols=1,
             replicas=256, n=1000, v_frame=0.5, load=0.45),
        # one chain far beyond a workgroup
        dict(name="flow-long-chain", kind="flow", potential="Cuspy", interactions="Laplace1d", rows=250007, cols=1,
             replicas=1, n=512, v_frame=1e-3, load=0.1),
        # a set of systems of every class, 512 to 65536 particles
        dict(name="ragged-96", kind="ragged", systems=96, log2min=9.0, log2max=16.0, sizes=1, events=3),
        # long-range ensemble with random forcing
        dict(name="longrange-256x8192", kind="longrange", rows=8192, replicas=256, n=20, alpha=1.5, dinc=10),
        # gradients of a run of 2000 steps
        dict(name="adjoint-64x4096", kind="adjoint", rows=4096, replicas=64, n=2000, window=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "protocol", "quasistatic", "quasistatic", "flow", "flow", "ragged", "longrange",
                       "adjoint"])
    if kind in ("steps", "protocol"):
        pot, inter = rng.choice([c for c in SINGLE if c[0] != "Smooth" or kind == "steps"])
        rows = _log(rng, 64, 1500 if inter == "LongRange1d" else 3000)
        cols = 1
        if inter == "Laplace2d":
            rows, cols = _log(rng, 8, 70), _log(rng, 8, 70)
        c = dict(kind=kind, potential=pot, interactions=inter, rows=rows, cols=cols)
        c.update(dict(n=_log(rng, 1, 200)) if kind == "steps" else dict(events=3))
        return c
    if kind == "quasistatic":
        pot, inter = rng.choice(CLASSES + [("Cuspy", "Laplace2d")])
        if inter == "Laplace2d":
            rows, cols = _log(rng, 20, 80), _log(rng, 20, 80)
        else:
            rows, cols = _log(rng, 256, 4096), 1
        replicas = max(1, min(1024, _log(rng, 3e4, 5e5) // (rows * cols)))
        return dict(kind=kind, potential=pot, interactions=inter, rows=rows, cols=cols, replicas=replicas, events=3)
    if kind == "flow":
        pot, inter = rng.choice([("Cuspy", "Laplace1d")] + CLASSES)
        sliding = rng.random() < 0.4
        rows = _log(rng, 256, 4000 if sliding else 20000)
        replicas = max(1, min(1024, _log(rng, 1e4, 5e5 if sliding else 2e6) // rows))
        return dict(kind=kind, potential=pot, interactions=inter, rows=rows, cols=1, replicas=replicas,
                    n=1000 if sliding else _log(rng, 100, 1000), v_frame=0.5 if sliding else 1e-3,
                    load=0.45 if sliding else 0.1)
    if kind == "ragged":
        return dict(kind=kind, systems=_log(rng, 8, 64), log2min=9.0, log2max=rng.choice([13.0, 14.0, 15.0, 16.0]),
                    sizes=rng.randrange(1, 1000), events=3)
    if kind == "longrange":
        return dict(kind=kind, rows=_log(rng, 500, 8192), replicas=_log(rng, 16, 256), n=_log(rng, 5, 20), alpha=1.5,
                    dinc=10)
    return dict(kind=kind, rows=_log(rng, 512, 6000), replicas=_log(rng, 4, 48), n=_log(rng, 200, 1500),
                window=rng.choice([50, 100]))


# what a user's program has in hand ------------------------------------------


def _nchunk(case):
    if case["kind"] == "adjoint":
        return 400
    return 100 if case.get("v_frame", 0.0) > 0.1 else 200


def _arguments(case, seed):
    """Constructor arguments shared by every class; replica r / system i of a
    case draws its landscape from seeds of its own."""
    rows, cols = case["rows"], case.get("cols", 1)
    kw = dict(m=1.0, eta=ETA, mu=1.0, k_frame=1.0 / (rows * cols), dt=DT, shape=[rows] if cols == 1 else [rows, cols],
              seed=(seed % 100003) * 10**7, distribution="weibull", parameters=[2.0, 1.0, 0.0], offset=OFFSET,
              nchunk=_nchunk(case))
    inter = case.get("interactions", "LongRange1d" if case["kind"] == "longrange" else "Laplace1d")
    kw.update(INTERACTIONS[inter])
    if case.get("potential") == "SemiSmooth":
        kw["kappa"] = 1.0
    if case["kind"] == "longrange":
        kw["alpha"] = case["alpha"]
    return kw


def _noise(case, seed, scale=0.5):
    """A stored configuration: slips [replicas, N] scattered over the wells."""
    n = case["rows"] * case.get("cols", 1)
    return np.random.default_rng(seed).uniform(-scale, scale, size=(case.get("replicas", 1), n))


def _batch(case, seed, **more):
    inter = case.get("interactions", "LongRange1d" if case["kind"] == "longrange" else "Laplace1d")
    return Batch(case["replicas"], seed_stride=case["rows"] * case.get("cols", 1),
                 potential=case.get("potential", "Cuspy"), interactions=inter, **_arguments(case, seed), **more)


def _ragged_classes(case):
    """(class, rows, cols) of every system of a ragged set: chains of all
    classes (a third of them with quartic interactions), a few lattices and a
    few chains with the no-passing minimiser."""
    rng = np.random.default_rng(case["sizes"])
    out = []
    for i in range(case["systems"]):
        rows = int(2.0 ** rng.uniform(case["log2min"], case["log2max"]))
        if i % 24 == 11:
            side = max(20, int(math.sqrt(rows)))
            out.append(("Line2d.System_Cuspy_Laplace", side, side + 3))
        elif i % 8 == 5:
            out.append(("System_Cuspy_Laplace_Nopassing", rows, 1))
        else:
            pot = ("Cuspy", "SemiSmooth", "Smooth")[i % 3]
            out.append((f"System_{pot}_{'Quartic' if rng.uniform() < 0.3 else 'Laplace'}", rows, 1))
    return out


def _ragged(case, seed):
    systems, u0, first = [], [], (seed % 100003) * 10**7
    rng = np.random.default_rng(seed)
    for name, rows, cols in _ragged_classes(case):
        kw = _arguments(dict(case, rows=rows, cols=cols), seed)
        kw["seed"] = first
        first += rows * cols
        if "Quartic" in name:
            kw.pop("k_interactions")
            kw.update(INTERACTIONS["Quartic1d"])
        if "SemiSmooth" in name:
            kw["kappa"] = 1.0
        if "Nopassing" in name:
            # (its sweeps need not converge from slips scattered both ways)
            kw.update(eta=0.0, dt=0.0)
            u0.append(np.zeros(kw["shape"]))
        else:
            u0.append(rng.uniform(-0.5, 0.5, size=kw["shape"]))
        systems.append((name, kw))
    return Ragged(systems), u0, np.array(["Smooth_" in n and "Semi" not in n for n, _ in systems])


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("steps", "protocol"):
        cls = SINGLE[(case["potential"], case["interactions"])]
        s["system"] = cls(**_arguments(case, seed))
        s["u0"] = _noise(case, seed)[0].reshape(s["system"].u.shape)
        if kind == "steps":
            s["system"].u = s["u0"]
    elif kind == "quasistatic":
        s["batch"] = _batch(case, seed)
        s["u0"] = _noise(case, seed).reshape([case["replicas"]] + s["batch"].shape)
    elif kind == "flow":
        b = s["batch"] = _batch(case, seed)
        b.u = _noise(case, seed, 0.3)
        if case["load"]:
            b.advanceToFixedForce(case["load"], allow_plastic=True)
    elif kind == "longrange":
        b = s["batch"] = _batch(case, seed, external="RandomNormalForcing", mean=0.0, stddev=0.1,
                                seed_forcing=seed % 100003, dinc_init=case["dinc"], dinc=case["dinc"])
        b.u = _noise(case, seed)
    elif kind == "ragged":
        s["set"], s["u0"], s["smooth"] = _ragged(case, seed)
    else:
        b = s["batch"] = _batch(case, seed)
        s.update(_adjoint_inputs(case, seed))
        s["params"] = adjoint.parameters(b)
        s["y"] = adjoint.chunk_data(b)
    return s


def _adjoint_inputs(case, seed):
    """Start state and the target of the loss of a differentiable run."""
    rng = np.random.default_rng(seed)
    shape = (case["replicas"], case["rows"])
    dev = torch.device("cuda")
    return dict(
        u0=torch.from_numpy(rng.uniform(-0.5, 0.5, size=shape)).to(dev),
        v0=torch.from_numpy(0.3 * rng.standard_normal(shape)).to(dev),
        a0=torch.zeros(shape, dtype=torch.float64, device=dev),
        target=torch.from_numpy(rng.uniform(-0.5, 0.5, size=shape)).to(dev),
    )


# one pass ---------------------------------------------------------------------


def run(state):
    case = state["case"]
    return {"steps": _run_steps, "protocol": _run_protocol, "quasistatic": _run_quasistatic, "flow": _run_flow,
            "longrange": _run_longrange, "ragged": _run_ragged, "adjoint": _run_adjoint}[case["kind"]](state, case)


def _run_steps(state, case):
    s = state["system"]
    s.flowSteps(case["n"], 1e-2)
    return dict(u=s.u, v=s.v, f_potential=s.f_potential)


def _run_protocol(state, case):
    s = state["system"]
    s.u = state["u0"]
    u_frame, f_frame, S = [], [], []
    for k in range(case["events"]):
        i_n = s.chunk.index_at_align
        if k == 0:
            s.u_frame = 0.0
        else:
            s.eventDrivenStep(EPS, k % 2 == 0)
        if k % 2 == 0:
            s.minimise()
        u_frame.append(s.u_frame)
        f_frame.append(float(np.mean(s.f_frame)))
        S.append(int(np.sum(s.chunk.index_at_align - i_n)))
    return dict(u=s.u, u_frame=np.array(u_frame), f_frame=np.array(f_frame), S=np.array(S))


def _run_quasistatic(state, case):
    b = state["batch"]
    b.u = state["u0"]
    q = b.quasistatic(EPS, case["events"], kicks_only=case["potential"] == "Smooth")
    return dict(u=adjoint.get_field(b, "u"), u_frame=q["u_frame"], f_frame=q["f_frame"], S=q["S"])


def _run_flow(state, case):
    b = state["batch"]
    b.flowSteps(case["n"], case["v_frame"])
    return dict(u=adjoint.get_field(b, "u"), v=adjoint.get_field(b, "v"))


def _run_longrange(state, case):
    b = state["batch"]
    b.timeSteps(case["n"])
    return dict(u=adjoint.get_field(b, "u"), v=adjoint.get_field(b, "v"), f=adjoint.get_field(b, "f"))


def _run_ragged(state, case):
    rg, smooth = state["set"], state["smooth"]
    rg.u = state["u0"]
    a = rg.quasistatic(EPS, case["events"], active=~smooth)
    b = rg.quasistatic(EPS, 2, kicks_only=True, active=smooth)
    u = np.concatenate([x.ravel() for x in rg.u])
    return dict(u=u, u_frame=a["u_frame"], f_frame=a["f_frame"], S=a["S"], u_frame_smooth=b["u_frame"],
                f_frame_smooth=b["f_frame"], S_smooth=b["S"])


def _run_adjoint(state, case):
    leaves = [state[k].clone().requires_grad_(True) for k in ("u0", "v0", "a0", "params", "y")]
    u, v, a = adjoint.run(state["batch"], case["n"], case["window"], *leaves)
    ((u - state["target"]) ** 2).sum(dim=1).mean().backward()
    # (v and a have decayed to rounding after a run of this length)
    out = dict(u=u.detach())
    out.update({"d" + k: x.grad for k, x in zip(("u0", "v0", "a0", "params", "y"), leaves)})
    return out


# what a pass cannot do without, and how far correct results may be apart --------

# operations of a particle's step (Verlet with two correctors, forces)
STEP_FLOP = 40.0
# steps of a quench from a stored configuration and of a kick's minimisation
QUENCH, KICK = 1200.0, 600.0


def work(case):
    kind = case["kind"]
    if kind == "ragged":
        sizes = [r * c for _, r, c in _ragged_classes(case)]
        n = float(sum(sizes))
        # slips in and out, the current wells
        return dict(bytes=32.0 * n, flops=STEP_FLOP * (QUENCH + KICK) * n)
    n = float(case["rows"] * case.get("cols", 1) * case.get("replicas", 1))
    if kind in ("protocol", "quasistatic"):
        steps = QUENCH + KICK * ((case["events"] - 1) // 2)
        pair = 0.0
        if case["interactions"] == "LongRange1d":
            pair = 3.0 * case["rows"]
        return dict(bytes=32.0 * n, flops=(STEP_FLOP + pair) * steps * n)
    if kind == "longrange":
        return dict(bytes=64.0 * n, flops=(2.0 * case["rows"] + STEP_FLOP) * case["n"] * n)
    if kind == "adjoint":
        y = 8.0 * n * _nchunk(case)
        # landscape in, its gradient out, states; forward, recomputation and
        # reverse
        return dict(bytes=2.0 * y + 80.0 * n, flops=3.0 * STEP_FLOP * case["n"] * n)
    # state and well in, state out
    return dict(bytes=64.0 * n, flops=STEP_FLOP * case["n"] * n)


def tolerance(case):
    """float64 throughout. A difference in the last bit of a yield position or
    of a sum travels along with the dynamics; against `exact` (whose logarithm
    and sums are torch's) it ends between 1e-15 and 1e-13 of the result."""
    if case["kind"] == "flow":
        # velocities of a pinned chain are about 1e-7, next to slips of 0.3
        return dict(rel=2e-9, max=1e-7)
    return dict(rel=1e-12, max=1e-9)


# the same in float64, by torch --------------------------------------------------

_MULT = 6364136223846793005


def _wrap64(x):
    """A Python integer as a signed 64-bit one (torch multiplies modulo 2^64)."""
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _shift(x, k):
    """Logical right shift of int64."""
    return (x >> k) & ((1 << (64 - k)) - 1)


def _pcg_uniform(state):
    """The uniform number in [0, 1) that pcg32 gives from each state."""
    x = _shift(_shift(state, 18) ^ state, 27) & 0xFFFFFFFF
    rot = _shift(state, 59)
    out = ((x >> rot) | (x << ((32 - rot) & 31))) & 0xFFFFFFFF
    return out.to(torch.float64) / 4294967296.0


def _landscape(first, shape, wells):
    """Yield positions [R, N, wells] of particles whose generators are seeded
    first, first + 1, ... : cumulative sums of Weibull (k = 2) increments."""
    n = int(np.prod(shape))
    seeds = torch.arange(n, dtype=torch.int64, device="cuda") + first
    mult = _wrap64(_MULT)
    state = (seeds + 1) * mult + 1
    y = torch.empty((n, wells), dtype=torch.float64, device="cuda")
    run = torch.zeros(n, dtype=torch.float64, device="cuda")
    for k in range(wells):
        run = run + torch.sqrt(-torch.log(1.0 - _pcg_uniform(state)))
        y[:, k] = run + OFFSET
        state = state * mult + 1
    return y.reshape(*shape, wells)


class _Exact:
    """[R, N] replicas stepped in float64."""

    def __init__(self, case, seed, u, wells):
        self.pot, self.inter = case.get("potential", "Cuspy"), case.get("interactions", "LongRange1d")
        self.rows, self.cols = case["rows"], case.get("cols", 1)
        kw = _arguments(case, seed)
        self.kw, self.kf = kw, kw["k_frame"]
        self.y = _landscape(kw["seed"], u.shape, wells)
        self.u = torch.as_tensor(u, device="cuda").clone()
        self.v = torch.zeros_like(self.u)
        self.a = torch.zeros_like(self.u)
        self.uf = torch.zeros((u.shape[0], 1), dtype=torch.float64, device="cuda")
        self.noise = None
        self.j = torch.searchsorted(self.y, self.u.unsqueeze(-1), right=True).squeeze(-1) - 1
        self.bounds()
        if self.inter == "LongRange1d":
            d = torch.arange(self.rows, dtype=torch.float64, device="cuda")
            d = torch.minimum(d, self.rows - d)
            d[0] = 1.0
            pref = kw["k_interactions"] / d ** (kw["alpha"] + 1.0)
            pref[0] = 0.0
            self.pref, self.kernel = pref, torch.fft.rfft(pref)

    def bounds(self):
        if bool(((self.j < 0) | (self.j + 2 > self.y.shape[-1])).any()):
            raise RuntimeError("a slip left the generated wells")
        self.yl = torch.gather(self.y, -1, self.j.unsqueeze(-1)).squeeze(-1)
        self.yr = torch.gather(self.y, -1, self.j.unsqueeze(-1) + 1).squeeze(-1)
        self.ym = 0.5 * (self.yl + self.yr)

    def walk(self):
        while True:
            up, down = self.u >= self.yr, self.u < self.yl
            if not bool((up | down).any()):
                return
            self.j = self.j + up.to(torch.int64) - down.to(torch.int64)
            self.bounds()

    def potential(self, u):
        yl, yr, ym = self.yl, self.yr, self.ym
        if self.pot == "Cuspy":
            return ym - u
        if self.pot == "SemiSmooth":
            ul, ur = (ym + yl) / 2.0, (ym + yr) / 2.0
            return torch.where(u < ul, u - yl, torch.where(u <= ur, ym - u, u - yr))
        h = 0.5 * (yr - yl)
        return -h / math.pi * torch.sin(math.pi * (u - ym) / h)

    def interaction(self, u):
        kw = self.kw
        if self.inter == "LongRange1d":
            w = u - u[:, :1]
            f = torch.fft.irfft(torch.fft.rfft(w) * self.kernel, n=self.rows) if self.rows > 2048 else w @ self.matrix()
            return f - self.pref.sum() * w
        if self.inter == "Laplace2d":
            x = u.reshape(-1, self.rows, self.cols)
            f = x.roll(1, 1) + x.roll(-1, 1) + x.roll(1, 2) + x.roll(-1, 2) - 4 * x
            return (f * kw["k_interactions"]).reshape(u.shape)
        um, up = u.roll(1, -1), u.roll(-1, -1)
        lap = um - 2 * u + up
        if self.inter == "Laplace1d":
            return lap * kw["k_interactions"]
        if self.inter == "Quartic1d":
            p, n = up - u, um - u
            return kw["a1"] * lap + kw["a2"] * (p * p * p + n * n * n)
        d = up - um
        return lap * (kw["k2"] + 0.25 * kw["k4"] * d * d)

    def matrix(self):
        if not hasattr(self, "_matrix"):
            i = torch.arange(self.rows, device="cuda")
            self._matrix = self.pref[(i[:, None] - i[None, :]) % self.rows]
        return self._matrix

    def step(self):
        dt = DT
        u = self.u + dt * self.v + 0.5 * dt * dt * self.a
        self.u = u
        self.walk()
        ff = self.kf * (self.uf - u)
        f0 = ff + self.potential(u) + self.interaction(u)
        if self.noise is not None:
            f0 = f0 + self.noise
        v, a = self.v + dt * self.a, None
        for _ in range(2):
            a = f0 - ETA * v
            v = self.v + 0.5 * dt * (self.a + a)
        self.v, self.a = v, f0 - ETA * v
        self.ff = ff

    def minimise(self):
        """Until ten descending residuals below 1e-5 (or below 1e-10), per
        replica; replicas that have stopped stay at rest."""
        R = self.u.shape[0]
        ring = torch.full((R, 10), math.inf, dtype=torch.float64, device="cuda")
        running = torch.ones((R, 1), dtype=torch.bool, device="cuda")
        zero = torch.zeros_like(self.u)
        while bool(running.any()):
            keep = self.u, self.v, self.a, self.j, self.yl, self.yr, self.ym
            self.step()
            rf, re = self.a.norm(dim=1), self.ff.norm(dim=1)
            r = torch.where(re != 0, rf / re, rf)
            ring = torch.cat([ring[:, 1:], r[:, None]], dim=1)
            stop = (((ring[:, 1:] < ring[:, :-1]).all(1)) & (ring < 1e-5).all(1)) | (ring < 1e-10).all(1)
            new = self.u, self.v, self.a, self.j, self.yl, self.yr, self.ym
            self.u, self.v, self.a, self.j, self.yl, self.yr, self.ym = (
                torch.where(running, n, k) for n, k in zip(new, keep))
            running = running & ~stop[:, None]
            self.v, self.a = torch.where(running, self.v, zero), torch.where(running, self.a, zero)

    def advance(self, du):
        """Shift all particles by du [R, 1], the frame with them."""
        self.u = self.u + du
        self.uf = self.uf + du * (self.kf + 1.0) / self.kf
        self.walk()

    def event(self, kick):
        if kick:
            return self.advance(torch.full_like(self.uf, EPS))
        if self.pot == "SemiSmooth":
            ul, ur = (self.ym + self.yl) / 2.0, (self.ym + self.yr) / 2.0
            room = torch.where((self.u < ul) | (self.u > ur), torch.full_like(self.u, -math.inf), ur - self.u)
        else:
            room = self.yr - self.u
        m = room.amin(dim=1, keepdim=True)
        self.advance(torch.where(m < 0.5 * EPS, torch.zeros_like(m), m - 0.5 * EPS))

    def protocol(self, events, kicks_only):
        uf, ff, S = [], [], []
        for k in range(events):
            j0 = self.j
            if k > 0:
                self.event(kicks_only or k % 2 == 0)
            if kicks_only or k % 2 == 0:
                self.minimise()
            uf.append(self.uf[:, 0])
            ff.append((self.kf * (self.uf - self.u)).mean(dim=1))
            S.append((self.j - j0).sum(dim=1))
        return tuple(torch.stack(x, dim=1) for x in (uf, ff, S))


def _normals(case, seed, count):
    """The first `count` random forces of every particle, [R, count, N]:
    Box-Muller from the generator of each replica, in particle order."""
    R, N = case["replicas"], case["rows"]
    mask = (1 << 64) - 1
    inc = ((0xDA3E39CB94B95BDB << 1) | 1) & mask
    total = 2 * N * count
    # state after k draws: A[k] s + C[k]; both by doubling
    A = torch.ones(1, dtype=torch.int64, device="cuda")
    C = torch.zeros(1, dtype=torch.int64, device="cuda")
    m, c = _MULT, inc
    while A.numel() < total:
        A, C = torch.cat([A, A * _wrap64(m)]), torch.cat([C, C * _wrap64(m) + _wrap64(c)])
        m, c = (m * m) & mask, (m * c + c) & mask
    first = seed % 100003
    s = [((inc + first + r * N) * _MULT + inc) & mask for r in range(R)]
    s = torch.tensor([_wrap64(x) for x in s], dtype=torch.int64, device="cuda")
    x = _pcg_uniform(A[None, :total] * s[:, None] + C[None, :total]).reshape(R, count, N, 2)
    return 0.1 * torch.sqrt(-2.0 * torch.log(1.0 - x[..., 0])) * torch.cos(2.0 * math.pi * x[..., 1])


def exact(case, seed):
    kind = case["kind"]
    if kind == "ragged":  # dozens of systems of different sizes, one after the other: minutes
        return None
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "flow":
        reach = 2.0 * case["v_frame"] * case["n"] * DT + 25.0
        e = _Exact(case, seed, _noise(case, seed, 0.3), int((100.0 + reach) / 0.8) + 10)
        if case["load"]:
            e.advance(case["load"] - (e.kf * (e.uf - e.u)).mean(dim=1, keepdim=True))
    else:
        e = _Exact(case, seed, _noise(case, seed), 200)
    if kind in ("steps", "flow"):
        for _ in range(case["n"]):
            e.uf = e.uf + case.get("v_frame", 1e-2) * DT
            e.step()
        if kind == "flow":
            return dict(u=e.u, v=e.v)
        shape = _arguments(case, seed)["shape"]
        return dict(u=e.u[0].reshape(shape), v=e.v[0].reshape(shape), f_potential=e.potential(e.u)[0].reshape(shape))
    if kind == "longrange":
        count = case["n"] // case["dinc"]
        draws = _normals(case, seed, max(1, count))
        for k in range(1, case["n"] + 1):
            if k % case["dinc"] == 0:
                e.noise = draws[:, k // case["dinc"] - 1]
            e.step()
        return dict(u=e.u, v=e.v, f=e.a)
    uf, ff, S = e.protocol(case["events"], case["potential"] == "Smooth")
    if kind == "protocol":
        return dict(u=e.u[0].reshape(_arguments(case, seed)["shape"]), u_frame=uf[0], f_frame=ff[0], S=S[0])
    return dict(u=e.u, u_frame=uf, f_frame=ff, S=S)


def _exact_adjoint(case, seed):
    """The loss's gradients by autograd over the same steps, recomputed in
    windows; wells are held at those of the trajectory."""
    from torch.utils.checkpoint import checkpoint

    x = _adjoint_inputs(case, seed)
    R, N = case["replicas"], case["rows"]
    kw = _arguments(case, seed)
    wells = _nchunk(case)
    y = _landscape(kw["seed"], (R, N), wells + 100)
    # the window that a new system holds: 30 wells before the one at u = 0,
    # where the first window does not hold that one with two to spare
    j0 = torch.searchsorted(y, torch.zeros((R, N, 1), dtype=torch.float64, device="cuda"), right=True) - 1
    if bool((j0 > wells - 4).any()):
        return None
    y = y[:, :, :wells].contiguous().requires_grad_(True)
    par = torch.tensor([1.0, kw["k_interactions"], kw["k_frame"], ETA], dtype=torch.float64, device="cuda")
    par = par.repeat(R, 1).requires_grad_(True)
    u0, v0, a0 = (x[k].clone().requires_grad_(True) for k in ("u0", "v0", "a0"))

    def steps(n, u, v, a, yl, yr, where, par, y):
        mu, k, kf, eta = (par[:, i:i + 1] for i in range(4))
        for _ in range(n):
            un = u + DT * v + 0.5 * DT * DT * a
            with torch.no_grad():
                j = where[0]
                while True:
                    lo = torch.gather(y, -1, j.unsqueeze(-1)).squeeze(-1)
                    hi = torch.gather(y, -1, j.unsqueeze(-1) + 1).squeeze(-1)
                    up, down = un >= hi, un < lo
                    if not bool((up | down).any()):
                        break
                    j = j + up.to(torch.int64) - down.to(torch.int64)
                where[0] = j
            ym = 0.5 * (torch.gather(y, -1, j.unsqueeze(-1)).squeeze(-1)
                        + torch.gather(y, -1, j.unsqueeze(-1) + 1).squeeze(-1))
            f0 = kf * (0.0 - un) + (ym - un) * mu + (un.roll(1, -1) - 2 * un + un.roll(-1, -1)) * k
            vn = v + DT * a
            for _ in range(2):
                vn = v + 0.5 * DT * (a + (f0 - eta * vn))
            u, v, a = un, vn, f0 - eta * vn
        return u, v, a

    with torch.no_grad():
        j = torch.searchsorted(y, u0.unsqueeze(-1), right=True).squeeze(-1) - 1
    u, v, a = u0, v0, a0
    for done in range(0, case["n"], case["window"]):
        n = min(case["window"], case["n"] - done)
        start = j.clone()
        after = [j]

        def block(u, v, a, par, y, n=n, start=start, after=after):
            where = [start.clone()]
            out = steps(n, u, v, a, None, None, where, par, y)
            after[0] = where[0]
            return out

        u, v, a = checkpoint(block, u, v, a, par, y, use_reentrant=False)
        j = after[0].clone()
    ((u - x["target"]) ** 2).sum(dim=1).mean().backward()
    return dict(u=u.detach(), du0=u0.grad, dv0=v0.grad, da0=a0.grad,
                dparams=par.grad, dy=y.grad)
