"""Batching on the GPU: GEMM tile shapes and the autotuner, HIP-graph capture of the CP step,
and one graph for several independent lattices.  Every replay of a graph is checked against
the same calls run eagerly on an identical propagator (same seed), with eager work and
synchronisation between the replays; results must be identical."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from afqmclab_amd._lib import check, lib  # noqa: E402
from afqmclab_amd.cp import Context, CPGroup, CPMethod, CPPropagator  # noqa: E402
from afqmclab_amd.model import HubbardModel, free_electron_trial, spin_block_trial  # noqa: E402
from tests.gpu_util import ctx, gauged  # noqa: E402
from tests.test_zz_no_alloc import DevArray, comb_host  # noqa: E402


# the Green GEMM's epilogue needs the 64-column tiles
GREEN_TILES = tuple(t for t, name in enumerate(CPPropagator.TILES)
                    if name.split("x")[1].startswith("64") or name == "128x128")


def make(c, nx, ny, nup, U, precision=0, nw=16, seed=5, t2=0.0, blocks=True, phases=False):
    model = HubbardModel.square(nx, ny, 2 * nup, U, 1.0, t2)
    if phases:
        model = gauged(model)
    phi = spin_block_trial(model, nup, nup) if blocks else free_electron_trial(model)
    m = CPMethod(dt=0.01, walkerSizePerThread=nw, ET=-1.0)
    kw = dict(nup=nup, spin_blocks=True) if blocks else dict(spin_blocks=False)
    prop = CPPropagator(c, model, m, phi, precision=precision, max_walkers=nw, **kw)
    prop.set_seed(seed, 0)
    prop.set_ET(-1.0)
    ws = prop.walkers(nw)
    ws.set_from_trial(phi)
    prop.stabilize(ws)
    return prop, ws


def state(prop, ws):
    wf, lw, al = ws.download()
    e = prop.energy()
    return wf, lw, al, prop.counter(), e["HNum"], e["den"]


def same(a, b):
    for x, y in zip(a, b):
        if isinstance(x, np.ndarray):
            assert np.array_equal(x, y)
        else:
            assert x == y, (x, y)


def block_of_work(prop, ws):
    """The enqueue-only sequence a driver repeats: steps, QR, comb, measurement."""
    for _ in range(3):
        prop.step(ws)
    prop.stabilize(ws)
    prop.pop_control(ws)
    prop.measure(ws)


@pytest.mark.parametrize("phases", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
def test_every_tile_shape_gives_the_same_step(precision, phases):
    """(Complex operators take the shapes; real ones, whose kernels have one shape, ignore them.)"""
    ref = None
    for t in range(len(CPPropagator.TILES)):
        prop, ws = make(ctx(), 4, 4, 5, 4.0, precision=precision, phases=phases)
        prop.set_tiles(propagate=t, overlap=t, green=t if t in GREEN_TILES else 0)
        for _ in range(2):
            prop.step(ws)
        prop.measure(ws)
        st = state(prop, ws)
        if ref is None:
            ref = st
        else:
            same(st, ref)
        ws.close()
        prop.close()


@pytest.mark.parametrize("phases", [False, True])
def test_autotune_keeps_state_and_results(phases):
    prop_a, ws_a = make(ctx(), 6, 6, 13, 4.0, precision=1, nw=64, phases=phases)
    prop_b, ws_b = make(ctx(), 6, 6, 13, 4.0, precision=1, nw=64, phases=phases)
    before = ws_a.download()
    tiles, ms = prop_a.autotune(ws_a, reps=3)
    after = ws_a.download()
    for x, y in zip(before, after):
        assert np.array_equal(x, y)
    nt = len(CPPropagator.TILES)
    assert tiles.shape == (3,) and all(0 <= t < nt for t in tiles) and tiles[2] in GREEN_TILES
    assert ms.shape == (3, nt) and np.all(ms[:, 0] > 0)
    assert all(ms[2, t] == -1.0 for t in range(nt) if t not in GREEN_TILES)
    if phases:
        assert np.all(ms[:2] > 0) and all(ms[2, t] > 0 for t in GREEN_TILES)
        assert all(ms[r, t] == np.min(ms[r][ms[r] > 0]) for r, t in enumerate(tiles))
    for _ in range(3):
        prop_a.step(ws_a)
        prop_b.step(ws_b)
    same(state(prop_a, ws_a), state(prop_b, ws_b))


@pytest.mark.parametrize("precision", [0, 1])
def test_autotune_leaves_the_shapes_that_no_kernel_takes(precision):
    """Real walkers: three kernels of one shape, timed once, and the shapes set for complex walkers stay.
    Complex walkers on real operators: the Green GEMM alone is tuned."""
    prop, ws = make(ctx(), 6, 6, 13, 4.0, precision=precision, nw=64)
    nt = len(CPPropagator.TILES)
    own = (6, 3, 7)
    prop.set_tiles(*own)
    tiles, ms = prop.autotune(ws, reps=2)
    assert tuple(tiles) == own
    assert np.all(ms[:, 0] > 0) and np.all(ms[:, 1:] == -1.0)
    wf, lw, _ = ws.download()
    wf[:, :, 0] *= np.exp(0.6j)
    ws.upload(wf, lw)
    tiles, ms = prop.autotune(ws, reps=2)
    assert tuple(tiles[:2]) == own[:2] and np.all(ms[:2, 0] > 0) and np.all(ms[:2, 1:] == -1.0)
    assert all((ms[2, t] > 0) == (t in GREEN_TILES) for t in range(nt)) and ms[2, tiles[2]] == np.min(ms[2][ms[2] > 0])


@pytest.mark.parametrize("phases", [False, True])
@pytest.mark.parametrize("blocks", [True, False])
def test_graph_replays_match_eager_calls(blocks, phases):
    c_graph, c_eager = Context(0), Context(0)
    pg, wg = make(c_graph, 4, 4, 5, 4.0, blocks=blocks, phases=phases)
    pe, we = make(c_eager, 4, 4, 5, 4.0, blocks=blocks, phases=phases)
    c_graph.capture_begin()
    block_of_work(pg, wg)
    g = c_graph.capture_end()
    assert g.nodes() > 10
    # nothing ran during the capture
    same(state(pg, wg)[:4], state(pe, we)[:4])
    for rep in range(3):
        g.launch()
        block_of_work(pe, we)
        c_graph.synchronize()
        same(state(pg, wg), state(pe, we))
        # eager work on the graph's own walkers between replays
        pg.step(wg)
        pe.step(we)
    g.close()


@pytest.mark.parametrize("phases", [False, True])
def test_group_graph_of_independent_lattices_matches_per_instance_calls(phases):
    shapes = [(4, 4, 5, 4.0), (6, 6, 13, 3.0), (6, 4, 9, 6.0)]
    origin = Context(0)
    gctx = [Context(0) for _ in shapes]
    ectx = Context(0)
    graph_sets = [make(c, *s, precision=1, seed=11 + i, phases=phases) for i, (c, s) in enumerate(zip(gctx, shapes))]
    eager_sets = [make(ectx, *s, precision=1, seed=11 + i, phases=phases) for i, s in enumerate(shapes)]
    for p, w in graph_sets:
        p.autotune(w, reps=2)
    origin.capture_begin(members=gctx)
    for p, w in graph_sets:
        block_of_work(p, w)
    g = origin.capture_end()
    for rep in range(2):
        g.launch()
        for p, w in eager_sets:
            block_of_work(p, w)
        origin.synchronize()
        for (p1, w1), (p2, w2) in zip(graph_sets, eager_sets):
            same(state(p1, w1), state(p2, w2))
    g.close()


def test_calls_that_return_data_fail_inside_a_capture():
    c = Context(0)
    p, w = make(c, 4, 4, 5, 4.0)
    c.capture_begin()
    with pytest.raises(Exception, match="cannot be recorded"):
        p.log_overlap(w)
    g = c.capture_end()
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("phases", [False, True])
def test_grouped_qr_of_ill_conditioned_walkers_equals_own_calls(precision, phases):
    """Restabilisation of a group whose members hold walkers that need further passes in one spin block
    only (a column 1e-16 from parallel to another: condition 1e16, after the shifted pass Q^H Q is 1e-3
    or more from I, beyond the 1e-4 at which a mixed-precision walker is redone): the blocks share the
    list of walkers to redo, the alive flags and the log-weights.  Identical to the members' own
    calls, and orthonormal: to 1e-12 in FP64; in mixed precision to the check's 1e-4 and the rounding
    of its FP32 Gram matrix (2 L 2^-24 <= 1e-5), a lost pass leaving 1e-3."""
    nw = 24
    shapes = [(8, 8, 28, 4.0), (6, 8, 20, 3.0)]
    c = Context(0)
    rng = np.random.default_rng(3)
    sets = [[make(c, *s, precision=precision, nw=nw, phases=phases) for s in shapes] for _ in range(2)]
    for j, (nx, ny, nup, _) in enumerate(shapes):
        L = nx * ny
        wfs = []
        for k in range(nw):
            w = np.zeros((2 * L, 2 * nup), dtype=np.complex128)
            for b in (0, 1):
                x = rng.uniform(-1, 1, (L, nup)) + (1j * rng.uniform(-1, 1, (L, nup)) if phases else 0.0)
                if (k + b) % 3 == 0:  # walker k's up block, walker k + 2's down block
                    x[L // 2:, -2] = 0.0
                    x[:L // 2, -1] = 2 * x[:L // 2, -2]
                    x[L // 2:, -1] *= 1e-16
                w[b * L:(b + 1) * L, b * nup:(b + 1) * nup] = x
            wfs.append(w)
        for s in sets:
            s[j][1].upload(wfs, np.zeros(nw))
    grp = CPGroup(sets[0])
    grp.stabilize()
    for p, w in sets[1]:
        p.stabilize(w)
    c.synchronize()
    for (p1, w1), (p2, w2), (nx, ny, nup, _) in zip(*sets, shapes):
        a, b = w1.download(), w2.download()
        same(a, b)
        assert p1.qr_stats() == p2.qr_stats() and p1.qr_stats()[0] >= nw // 2
        assert np.sum(a[2] != 0) >= nw // 3  # the well-conditioned third at least
        for k in np.flatnonzero(a[2]):
            q = a[0][k]
            assert np.max(np.abs(q.conj().T @ q - np.eye(2 * nup))) < (1e-12 if precision == 0 else 1.1e-4), k
    grp.close()


class Comb:
    """afqmc_comb_noalloc on device arrays: call() enqueues it, check() compares with afqmc_comb."""

    def __init__(self, c, nw, seed):
        rng = np.random.default_rng(seed)
        self.c, self.w, self.u = c, rng.uniform(0, 5, nw), rng.uniform(0, 1, nw)
        self.dev = [DevArray(a) for a in (self.w, self.u, np.full(nw, -7, dtype=np.int32), np.zeros(3))]
        self.ref = comb_host(self.w, self.u)

    def call(self):
        dw, du, dt, ds = self.dev
        check(lib().afqmc_comb_noalloc(self.c.h, len(self.w), dw.p, du.p, dt.p, ds.p))

    def check(self):
        """The results so far, which are then wiped."""
        dt, ds = self.dev[2:]
        assert np.array_equal(dt.get(), self.ref[0]) and np.array_equal(ds.get(), self.ref[1])
        for d in (dt, ds):
            d.put(np.full_like(d.host, -7))


@pytest.mark.parametrize("form", ["context", "members", "group", pytest.param("group on a member", marks=pytest.mark.skip(
    reason="a capture whose member stream forks a group's side streams has crashed the process in capture_end; "
           "group calls on a member context are refused"))])
@pytest.mark.parametrize("precision", [0, 1])
def test_graph_of_real_walkers_makes_all_its_calls_for_complex_ones(form, precision):
    """A graph captured while its sets are real, launched after one of them became complex: every
    recorded call is made again, those on other sets and those without walkers (the comb on device
    buffers) included, from one context, from member contexts and for a group's calls.  Identical to
    eager calls, real and complex walkers in turn (one restabilisation a block, so the walkers' buffers
    change parity between the launches)."""
    shapes = [(4, 4, 5, 4.0), (6, 4, 9, 3.0)]
    origin = Context(0)
    member = Context(0)
    gctx = {"members": [member, Context(0)], "group on a member": [member, member]}.get(form, [origin, origin])
    gsets = [make(c, *s, precision=precision, seed=21 + i) for i, (c, s) in enumerate(zip(gctx, shapes))]
    esets = [make(ctx(), *s, precision=precision, seed=21 + i) for i, s in enumerate(shapes)]
    grp = CPGroup(gsets) if form.startswith("group") else None
    comb = Comb(gctx[1], 500, 8)
    start = [w.download()[0] for _, w in gsets]

    def block(sets, grp=None):
        if grp is None:
            for p, w in sets:
                block_of_work(p, w)
            return
        for _ in range(3):
            grp.step()
        grp.stabilize()
        grp.pop_control()
        for p, w in sets:
            p.measure(w)

    origin.capture_begin(members=[c for c in dict.fromkeys(gctx) if c is not origin])
    block(gsets, grp)
    comb.call()
    g = origin.capture_end()
    for theta in (0.0, 0.6, 0.0, 0.0, 0.6, 0.6):
        up = [w.copy() for w in start]
        up[0][:, :, 0] *= np.exp(1j * theta)  # the second set stays real
        for sets in (gsets, esets):
            for (p, w), x in zip(sets, up):
                w.upload(x, np.full(w.nw, -1j * theta if x is up[0] else 0.0))
                p.reset_measure()
        for _ in range(2):
            g.launch()
            block(esets)
            for c in [origin] + gctx:
                c.synchronize()
            comb.check()
            for (p1, w1), (p2, w2) in zip(gsets, esets):
                same(state(p1, w1), state(p2, w2))
    g.close()
    if grp:
        grp.close()


def test_group_calls_are_captured_on_the_origin_only():
    """A group whose context is a member of the capture: refused before anything is recorded, and the capture
    stays whole."""
    origin, member = Context(0), Context(0)
    p, w = make(member, 4, 4, 5, 4.0)
    grp = CPGroup([(p, w)])
    before = state(p, w)
    origin.capture_begin(members=[member])
    for call in (grp.step, grp.stabilize, grp.pop_control):
        with pytest.raises(Exception, match="captured on the capture's origin"):
            call()
    p.onebody(w, 0)
    g = origin.capture_end()
    same(state(p, w), before)
    g.launch()
    origin.synchronize()
    member.synchronize()
    assert not np.array_equal(w.download()[0], before[0])
    g.close()
    grp.step()
    member.synchronize()
    assert p.counter() > before[3]
    grp.close()


def test_graph_with_phaseless_calls_makes_them_for_complex_walkers_too():
    """The phaseless measurement, comb and resets recorded beside a real constraint-path set: made by
    the graph and, after that set became complex, by the repeated calls, as eagerly."""
    from tests.test_gpu_ph import make_case
    c = Context(0)
    cp, cw = make(c, 4, 4, 5, 4.0)
    got = []
    for _ in range(2):  # on the shared context
        _, dm, _, prop, ws, *_ = make_case(seed=4)
        B, lw = dm.exp_minus_alpha_k(-0.025)
        prop.set_onebody(2, B, lw, False)
        got.append((prop, ws))
    shared = ctx()
    real = cw.download()[0]

    def work(prop, ws, k):
        if k:
            prop.adjust_ET()
        else:
            prop.reset_measure()
        prop.measure(ws)
        prop.pop_control(ws)
        prop.measure(ws)

    graphs = []
    for k in range(2):
        c.capture_begin(members=[shared])
        cp.step(cw)
        work(*got[0], k)
        graphs.append(c.capture_end())
    for theta in (0.0, 0.6, 0.0):
        up = real.copy()
        up[:, :, 0] *= np.exp(1j * theta)
        cw.upload(up, np.full(cw.nw, -1j * theta))
        for k in (0, 1, 1):
            graphs[k].launch()
            work(*got[1], k)
            c.synchronize()
            shared.synchronize()
            (p1, w1), (p2, w2) = got
            same(w1.download(), w2.download())
            e1, e2 = p1.energy(), p2.energy()
            assert all(np.array_equal(e1[n], e2[n]) for n in e1)
            assert p1.get_ET() == p2.get_ET() and p1.counter() == p2.counter()
    for g in graphs:
        g.close()


def test_graph_launch_returns_before_the_work_is_done():
    """Launches are asynchronous, also where the recorded calls are made again for complex walkers: 40
    propagations of 1024 walkers of 256 x 56 + 56 are enqueued in a fraction of their time."""
    c = Context(0)
    p, w = make(c, 16, 16, 56, 4.0, nw=1024)
    c.capture_begin()
    for _ in range(20):
        p.onebody(w, 0)
        p.onebody(w, 1)
    g = c.capture_end()
    up = np.zeros((1024, 512, 112), dtype=np.complex128)
    up[:, :256, :56] = up[:, 256:, 56:] = np.eye(256)[:, :56]
    for theta in (0.0, 0.6):
        up[:, :, 0] *= np.exp(1j * theta)
        w.upload(up)
        g.launch()
        c.synchronize()
        w.upload(up)
        t0 = time.perf_counter()
        g.launch()
        t1 = time.perf_counter()
        c.synchronize()
        t2 = time.perf_counter()
        assert t1 - t0 < 0.5 * (t2 - t0), (theta, t1 - t0, t2 - t0)
    g.close()


def test_phaseless_calls_that_synchronise_leave_a_capture_whole():
    """Phaseless calls that synchronise are refused before they record anything: the capture goes on, the
    walkers stay as they were, and contexts outside the capture run as ever."""
    from tests.test_gpu_ph import make_case
    c = Context(0)
    cp, cw = make(c, 4, 4, 5, 4.0)
    _, dm, _, prop, ws, *_ = make_case(seed=4)  # on the shared context
    for which, alpha in ((0, 0.05), (2, -0.025)):
        prop.set_onebody(which, *dm.log_exp_minus_alpha_k(alpha), True)
    before, counter = ws.download(), prop.counter()
    c.capture_begin(members=[ctx()])
    for call in (lambda: prop.step(ws), lambda: prop.stabilize(ws), lambda: prop.onebody(ws, 0), lambda: prop.measure(ws),
                 lambda: prop.log_overlap(ws), lambda: prop.energy(), lambda: prop.pop_control(ws, record=True),
                 lambda: prop.set_seed(3), lambda: ws.download()):
        with pytest.raises(Exception, match="captured|recorded into a graph"):
            call()
    cp.step(cw)
    g = c.capture_end()
    n = g.nodes()
    g.launch()
    c.synchronize()
    same(before, ws.download())
    assert prop.counter() == counter
    g.close()
    c.capture_begin()  # without the shared context
    cp.step(cw)
    prop.step(ws)
    g = c.capture_end()
    assert prop.counter() > counter and g.nodes() in (n - 1, n, n + 1)
    g.close()
