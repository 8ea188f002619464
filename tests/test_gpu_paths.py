"""Kernel paths chosen by size, class or state, against the CPU oracle bit for
bit: the windows that move inside a launch, and the rules that route a call."""

import numpy as np
import pytest

from oracle import pyoracle
from tests import protocols as P

pytestmark = pytest.mark.gpu


def _kw(N, **extra):
    kw = dict(m=1.0, eta=2.0 * np.sqrt(3.0) / 10.0, mu=1.0, k_interactions=1.0, k_frame=1.0 / N, dt=0.1, shape=[N],
              seed=5, distribution="weibull", parameters=[2.0, 1.0, 0.0], offset=-20.0, nchunk=60)
    kw.update(extra)
    return kw


def _sliding(v_frame, N, **extra):
    """A batch of two chains and the oracle's, loaded so that they slide."""
    from frictionqpotspringblock_amd.batch import Batch

    kw = _kw(N, **extra)
    b = Batch(2, seed_stride=N, potential="Cuspy", interactions="Laplace1d", **kw)
    ref = [pyoracle.Line1d.System_Cuspy_Laplace(**dict(kw, seed=kw["seed"] + r * N)) for r in range(2)]
    load = 0.5 if v_frame > 0 else -0.5
    b.advanceToFixedForce(load, allow_plastic=True)
    for s in ref:
        s.advanceToFixedForce(load, allow_plastic=True)
    return b, ref


def _same(b, ref):
    for r, s in enumerate(ref):
        assert np.array_equal(b.u[r], s.u)
        assert np.array_equal(b.v[r], s.v)
        assert np.array_equal(b.f[r], s.f)
        assert np.array_equal(b.index_at_align[r], s.chunk.index_at_align)
        assert np.array_equal(b._get_state("start").reshape(2, -1)[r], s.chunk.start)
        assert np.array_equal(b._get_state("y").reshape(2, b.size, -1)[r], s.chunk.data)


@pytest.mark.parametrize("v_frame", [0.5, -0.5])
@pytest.mark.parametrize("ppt,threads,N", [(1, 64, 3), (1, 128, 65), (2, 64, 127), (4, 64, 256), (8, 64, 509), (4, 1024, 4096)])
def test_windows_move_inside_flow(ppt, threads, N, v_frame):
    """flowSteps of sliding chains: every window moves several times inside
    the launch (forward and backward), at each launch shape, with launches
    that end between any two steps."""
    b, ref = _sliding(v_frame, N)
    b.set_launch(ppt, threads)
    n = 300 if N < 4096 else 120
    i0 = b.index_at_align
    b.flowSteps(n, v_frame, block=37)
    for s in ref:
        s.flowSteps(n, v_frame)
    assert np.abs(b.index_at_align - i0).max() > (15 if N < 4096 else 5)
    _same(b, ref)


def test_windows_move_in_many_replicas():
    """More replicas of one particle per thread than fit the compute units with
    the refill's registers: the launch ends at the first window that moves
    and the run goes on with the form that moves them itself."""
    from frictionqpotspringblock_amd.batch import Batch

    N, R = 65, 2050
    kw = _kw(N)
    b = Batch(R, seed_stride=N, potential="Cuspy", interactions="Laplace1d", **kw)
    b.set_launch(1, 128)
    b.advanceToFixedForce(0.5, allow_plastic=True)
    i0 = b.index_at_align
    b.flowSteps(200, 0.5)
    assert np.abs(b.index_at_align - i0).max() > 15
    start = b._get_state("start").reshape(R, -1)
    for r in (0, 1027, R - 1):
        s = pyoracle.Line1d.System_Cuspy_Laplace(**dict(kw, seed=kw["seed"] + r * N))
        s.advanceToFixedForce(0.5, allow_plastic=True)
        s.flowSteps(200, 0.5)
        assert np.array_equal(b.u[r], s.u) and np.array_equal(b.f[r], s.f)
        assert np.array_equal(start[r], s.chunk.start)


@pytest.mark.parametrize("ppt,threads,N", [(1, 128, 65), (2, 64, 127), (4, 128, 257), (8, 64, 509)])
@pytest.mark.parametrize("cls", ["SemiSmooth_Laplace", "Smooth_Laplace", "Cuspy_Quartic", "Cuspy_Laplace_RandomForcing"])
def test_windows_move_in_every_class(cls, ppt, threads, N):
    """The same for other potentials and interactions and with random forcing
    (chains thrown forwards, whose windows move while they come to rest)."""
    from frictionqpotspringblock_amd.batch import Batch

    pot, inter = cls.split("_")[:2]
    kw = _kw(N, **(dict(kappa=1.0) if pot == "SemiSmooth" else {}))
    if inter == "Quartic":
        del kw["k_interactions"]
        kw.update(a1=1.0, a2=5.0)
    more = {}
    if "Forcing" in cls:
        kw.update(mean=0.0, stddev=0.1, seed_forcing=7, dinc_init=5, dinc=10)
        more["external"] = "RandomNormalForcing"
    b = Batch(2, seed_stride=N, potential=pot, interactions=inter + "1d", **kw, **more)
    ref = []
    for r in range(2):
        k = dict(kw, seed=kw["seed"] + r * N)
        if more:
            k.update(seed_forcing=kw["seed_forcing"] + r * N, dinc_init=[5] * N, dinc=[10] * N)
        ref.append(getattr(pyoracle.Line1d, f"System_{cls}")(**k))
    b.set_launch(ppt, threads)
    v = np.full(N, 20.0)
    b.v = np.broadcast_to(v, [2, N])
    i0 = b.index_at_align
    b.flowSteps(100, 0.1, block=37)
    for s in ref:
        s.v = v
        s.flowSteps(100, 0.1)
    assert np.abs(b.index_at_align - i0).min() > 30 and b._get_state("start").max() > 0
    _same(b, ref)


def test_window_jumps_inside_flow():
    """Slips that leave the window altogether (fast particles) and slips that
    stay where they are (a particle at rest next to them)."""
    b, ref = _sliding(0.5, 64, nchunk=12)
    v = np.zeros(64)
    v[3], v[40], v[41] = 400.0, -350.0, 90.0
    b.v = np.broadcast_to(v, [2, 64])
    for s in ref:
        s.v = v
    b.flowSteps(40, 0.5)
    for s in ref:
        s.flowSteps(40, 0.5)
    _same(b, ref)


def test_adjoint_refuses_moved_windows():
    """A window moved inside a launch is noticed by the adjoint forward pass."""
    import torch

    from frictionqpotspringblock_amd import adjoint as A

    b, _ = _sliding(0.5, 64)
    z = torch.zeros((2, 64), dtype=torch.float64, device="cuda")
    with pytest.raises(RuntimeError, match="left the landscape window"):
        A.run(b, 300, 50, z, z + 20.0, z, A.parameters(b), flow=True, v_frame=0.5)


def _longrange_kw(N, **extra):
    return _kw(N, alpha=1.0, offset=-100.0, nchunk=200, **extra)


@pytest.mark.parametrize("N", [3, 64, 511, 512, 513, 577, 1000])
def test_longrange_exact_sum(N):
    """A long-range chain on both sides of the size at which its steps and
    minimisations spread over tiles; the operations that stay resident in
    between (until event, activity, truncation) continue from the same state."""
    import frictionqpotspringblock_amd as fq

    kw = _longrange_kw(N)
    g, o = fq.Line1d.System_Cuspy_LongRange(**kw), pyoracle.Line1d.System_Cuspy_LongRange(**kw)
    v = np.random.default_rng(N).normal(size=N)
    for s in (g, o):
        s.v = v
        s.flowSteps(30, 0.2)
        s.timeSteps(17)
    assert np.array_equal(g.u, o.u) and np.array_equal(g.v, o.v) and np.array_equal(g.f, o.f)
    ret = []
    for s in (g, o):
        r = [s.minimise(), s.eventDrivenStep(1e-3, False), s.eventDrivenStep(1e-3, True)]
        r += [s.timeStepsUntilEvent(), s.minimise(time_activity=True), s.quasistaticActivityLast]
        s.eventDrivenStep(1e-3, True)
        r += [s.minimise(), s.inc, s.u_frame]
        ret.append(r)
    assert ret[0] == ret[1]
    assert np.array_equal(g.u, o.u) and np.array_equal(g.f_interactions, o.f_interactions)
    assert np.array_equal(g.chunk.index_at_align, o.chunk.index_at_align)


@pytest.mark.parametrize("N", [255, 256, 257, 511, 512, 513, 1024, 1025, 2047, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 16384])
def test_longrange_product(N):
    """The batched long-range forces at the sizes where the transforms change
    (powers of two, one more, one less; the matrix product below 257 and above
    8192), against the sum in extended precision. The transforms' error is
    at most a small multiple of eps log2(M) |g| |w| (2-norms of the kernel and
    of the shifted slips; forward, product and inverse, 8 for the constants);
    the matrix product's at most gamma_N times the sum of the terms."""
    from frictionqpotspringblock_amd.batch import Batch

    R = 2
    b = Batch(R, seed_stride=N, potential="Cuspy", interactions="LongRange1d", **_longrange_kw(N))
    u = np.random.default_rng(N).normal(size=(R, N))
    b.u = u
    b.timeSteps(1)
    u = b.u.astype(np.longdouble)
    d = np.minimum(np.arange(N), N - np.arange(N)).astype(float)
    g = np.zeros(N)
    g[1:] = 1.0 / d[1:] ** 2.0
    gl, uu = g.astype(np.longdouble), np.concatenate([u, u], axis=1)
    f = np.zeros((R, N), dtype=np.longdouble)
    for k in range(1, N):
        f += gl[k] * (uu[:, k:k + N] - u)
    w = np.linalg.norm((u - u[:, :1]).astype(float), axis=1)
    eps = np.finfo(float).eps
    bound = 8.0 * eps * np.log2(4 * N) * np.linalg.norm(g) * w[:, None]
    bound = np.maximum(bound, 2.0 * N * eps * g.sum() * np.abs(u - u[:, :1]).max()) if N < 257 or N == 8193 else bound
    assert np.all(np.abs(b.f_interactions - f) <= bound)


CLASSES = [("Line1d", "System_Cuspy_Laplace", dict(k_interactions=1.0)),
           ("Line1d", "System_SemiSmooth_Laplace", dict(k_interactions=1.0, kappa=1.0)),
           ("Line1d", "System_Smooth_Laplace", dict(k_interactions=1.0)),
           ("Line1d", "System_Cuspy_Quartic", dict(a1=1.0, a2=5.0)),
           ("Particles", "System_Cuspy", {})]


def _pair(sub, cls, shape, extra, **more):
    import frictionqpotspringblock_amd as fq

    kw = _kw(int(np.prod(shape)), **more)
    del kw["k_interactions"]
    kw.update(extra, shape=list(shape))
    return getattr(getattr(fq, sub), cls)(**kw), getattr(getattr(pyoracle, sub), cls)(**kw)


def _minimise(g, o):
    """Minimisations that end by their step limit, by convergence from a
    moving state, and after a uniform displacement."""
    v = np.random.default_rng(g.u.size).normal(size=g.u.shape)
    for s in (g, o):
        s.v = v
    assert g.minimise(max_iter=7, max_iter_is_error=False) == o.minimise(max_iter=7, max_iter_is_error=False)
    for k in ("u", "v", "a", "f"):
        assert np.array_equal(getattr(g, k), getattr(o, k)), k
    assert g.minimise() == o.minimise()
    assert g.inc == o.inc
    for s in (g, o):
        s.eventDrivenStep(1e-3, True)
    assert g.minimise(tol=1e-3, niter_tol=3) == o.minimise(tol=1e-3, niter_tol=3)
    assert g.inc == o.inc
    for k in ("u", "v", "f", "f_potential", "f_interactions"):
        assert np.array_equal(getattr(g, k), getattr(o, k)), k
    assert np.array_equal(g.chunk.index_at_align, o.chunk.index_at_align)
    assert np.array_equal(g.chunk.start, o.chunk.start)


@pytest.mark.parametrize("N", [3, 65, 511, 513, 2047, 2049, 4096, 4097])
@pytest.mark.parametrize("sub,cls,extra", CLASSES, ids=[c[1] for c in CLASSES])
def test_minimise_chains(sub, cls, extra, N):
    """minimise of single chains on both sides of the sizes at which the launch
    shape changes; masses other than 1 with the odd sizes."""
    _minimise(*_pair(sub, cls, [N], extra, m=2.0 if N in (65, 2049) else 1.0))


@pytest.mark.parametrize("shape", [(3, 4), (5, 103), (19, 27), (45, 45), (41, 50), (64, 64), (65, 64)])
@pytest.mark.parametrize("cls,extra", [("System_Cuspy_Laplace", dict(k_interactions=1.0)),
                                       ("System_Cuspy_QuarticGradient", dict(k2=1.0, k4=1.0))])
def test_minimise_lattices(cls, extra, shape):
    _minimise(*_pair("Line2d", cls, shape, extra, m=2.0 if shape[0] == 41 else 1.0))


@pytest.mark.parametrize("shape,N", [((0, 0), 4097), ((0, 0), 8192), ((4, 1024), 4096), ((16, 256), 4093), ((16, 512), 8191)])
@pytest.mark.parametrize("pot,inter", [("Cuspy", "Laplace1d"), ("SemiSmooth", "Laplace1d"), ("Smooth", "Laplace1d"), ("Cuspy", "Quartic1d")])
def test_quasistatic_of_large_variants(pot, inter, shape, N):
    """The protocol and minimise at the launch shapes whose driver is chosen
    by class (the pipelined one or the general kernels), the sizes above 4096
    among them, where no other variant holds a chain."""
    from frictionqpotspringblock_amd.batch import Batch

    extra = {"Laplace1d": dict(k_interactions=1.0), "Quartic1d": dict(a1=1.0, a2=5.0)}[inter]
    kw = _kw(N)
    del kw["k_interactions"]
    kw.update(extra, offset=-100.0, nchunk=200)
    if pot == "SemiSmooth":
        kw["kappa"] = 1.0
    b = Batch(2, seed_stride=N, potential=pot, interactions=inter, **kw)
    if shape[0]:
        b.set_launch(*shape)
    u = np.random.default_rng(N).uniform(-0.5, 0.5, size=(2, N))
    b.u = u
    kicks = pot == "Smooth"
    q = b.quasistatic(1e-3, 2 if kicks else 3, kicks_only=kicks)
    o = getattr(pyoracle.Line1d, f"System_{pot}_{inter[:-2]}")(**dict(kw, seed=kw["seed"] + N))
    o.u = u[1]
    for k in range(q["S"].shape[1]):
        if k == 0:
            o.u_frame = 0.0
        else:
            o.eventDrivenStep(1e-3, kicks or k % 2 == 0)
        if kicks or k % 2 == 0:
            o.minimise()
        assert q["u_frame"][1, k] == o.u_frame and q["inc"][1, k] == o.inc
    assert np.array_equal(b.u[1], o.u)
    b.u = u
    b.minimise()
    o.u = u[1]
    o.minimise()
    assert np.array_equal(b.u[1], o.u) and b.inc[1] == o.inc


@pytest.mark.parametrize("pot,inter,shape,ppt", [
    ("Cuspy", "Laplace1d", [513], 4), ("SemiSmooth", "Laplace1d", [513], 1), ("Smooth", "Laplace1d", [2500], 4),
    ("Cuspy", "Quartic1d", [1537], 2), ("Cuspy", "Laplace2d", [19, 28], 1), ("Cuspy", "Laplace2d", [33, 33], 2)])
def test_automatic_shapes(pot, inter, shape, ppt):
    """Steps, runs that decide after every step and the driver each have a
    launch shape of their own, which depends on the number of replicas as
    well: two replicas have the results of the first two of 300."""
    from frictionqpotspringblock_amd.batch import Batch

    N = int(np.prod(shape))
    kw = _kw(N, offset=-100.0, nchunk=200)
    kw["shape"] = shape
    if inter == "Quartic1d":
        del kw["k_interactions"]
        kw.update(a1=1.0, a2=5.0)
    if pot == "SemiSmooth":
        kw["kappa"] = 1.0
    u = np.random.default_rng(N).uniform(-0.5, 0.5, size=[300] + shape)
    got = []
    for R in (2, 300):
        b = Batch(R, seed_stride=N, potential=pot, interactions=inter, **kw)
        if R == 2:
            assert b.launch[0] == ppt
        b.u = u[:R]
        i_n = b.index_at_align
        b.flowSteps(40, 0.01)
        got.append([b.u[:2], b.v[:2]])
        ret = b.minimise_truncate(i_n, S_truncate=N // 8, max_iter=300, max_iter_is_error=False)
        got[-1] += [ret[:2], b.u[:2]]
        b.minimise()
        got[-1] += [b.inc[:2], b.u[:2], b.f[:2], b.index_at_align[:2]]
    for k, (x, y) in enumerate(zip(*got)):
        assert np.array_equal(x, y), k


@pytest.mark.parametrize("sub,cls,extra", CLASSES[:4], ids=[c[1] for c in CLASSES[:4]])
def test_tiles_windows_and_forces(sub, cls, extra):
    """A chain over tiles whose windows move between blocks of steps, and the
    operations over many workgroups around it (uniform displacement, largest
    elastic displacement, forces)."""
    g, o = _pair(sub, cls, [9001], extra, m=2.0 if cls == "System_SemiSmooth_Laplace" else 1.0)
    for s in (g, o):
        s.advanceToFixedForce(0.6, allow_plastic=True)
        s.flowSteps(300, 0.5)
    assert np.array_equal(g.u, o.u) and np.array_equal(g.f, o.f)
    assert np.array_equal(g.chunk.start, o.chunk.start) and g.chunk.start.max() > 0
    assert np.array_equal(g.chunk.data, o.chunk.data)
    if "_Smooth_" not in cls:
        for s in (g, o):
            s.minimise()
        assert g.maxUniformDisplacement() == o.maxUniformDisplacement()
        assert g.eventDrivenStep(1e-3, False) == o.eventDrivenStep(1e-3, False)
        assert np.array_equal(g.u, o.u) and np.array_equal(g.f, o.f)


@pytest.mark.parametrize("N", [8191, 8192, 8193])
def test_transfers(N):
    """Fields on both sides of the size that passes through pinned memory
    (64 KiB), read by several threads at once."""
    from concurrent.futures import ThreadPoolExecutor

    import frictionqpotspringblock_amd as fq

    s = fq.Line1d.System_Cuspy_Laplace(**_kw(N))
    rng = np.random.default_rng(N)
    x, v = 1e-3 * rng.normal(size=N), rng.normal(size=N)
    s.u, s.v = x, v
    assert np.array_equal(s.u, x) and np.array_equal(s.v, v)
    with ThreadPoolExecutor(4) as ex:
        got = list(ex.map(lambda k: getattr(s, k).copy(), ["u", "v"] * 16))
    assert all(np.array_equal(q, (x, v)[i % 2]) for i, q in enumerate(got))


def test_many_run_states():
    """More replicas than the run states' pinned memory holds."""
    from frictionqpotspringblock_amd.batch import Batch

    R = 8000
    kw = _kw(3)
    b = Batch(R, potential="Cuspy", interactions="Laplace1d", seed_stride=3, **kw)
    b.flowSteps(50, 0.1)
    u = b.u
    for r in (0, 4321, R - 1):
        o = pyoracle.Line1d.System_Cuspy_Laplace(**dict(kw, seed=kw["seed"] + 3 * r))
        o.flowSteps(50, 0.1)
        assert np.array_equal(u[r], o.u)


@pytest.mark.parametrize("N,m", [(256 * 1024, 1.0), (256 * 1024 + 1, 1.0), (256 * 1024 + 1, 2.0)])
def test_tiles_share_units(N, m):
    """Chains of as many tiles as compute units, and one more."""
    g, o = _pair("Line1d", "System_Cuspy_Laplace", [N], dict(k_interactions=1.0), m=m)
    v = np.random.default_rng(N).normal(size=N)
    for s in (g, o):
        s.v = v
        s.flowSteps(150, 0.5)
    assert np.array_equal(g.u, o.u) and np.array_equal(g.f, o.f)
    assert np.array_equal(g.chunk.index_at_align, o.chunk.index_at_align)
