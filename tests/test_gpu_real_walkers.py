"""Kernels for real operators and real walkers: the products against numpy, and whole calls on real
walkers against the same walkers with a phase on one column (complex data, so the general kernels),
whose overlaps, Green's functions, fields and energies are the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from afqmclab_amd._lib import check, dptr, iptr, lib  # noqa: E402
from afqmclab_amd.cp import CPMethod, CPPropagator  # noqa: E402
from afqmclab_amd.model import HubbardModel, free_electron_trial, spin_block_trial  # noqa: E402
from tests.gpu_util import crand, ctx, gj_inverse_masked  # noqa: E402

EPS = {0: 2.0 ** -53, 1: 2.0 ** -24}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("op_t", [0, 1])
@pytest.mark.parametrize("b_real", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 64, 16), (17, 65, 15), (37, 1200, 29), (112, 2100, 256),
                                   (130, 1100, 33), (256, 9000, 48)])
def test_real_gemm_matches_numpy(precision, op_t, b_real, shape):
    """Every rounding of a K-term sum of products bounded by 1 is below K eps (two products per
    complex element, so no cross terms)."""
    M, N, K = shape
    rng = np.random.default_rng(M + N + K + op_t)
    A = rng.uniform(-1, 1, (M, K))
    B = crand(rng, K, N)
    group = 7
    scale = None if op_t else crand(rng, (N + group - 1) // group, K)
    C = np.zeros((N, M), dtype=np.complex128)
    Abuf = np.ascontiguousarray(A if op_t else A.T)  # op T: K x M column-major
    Bbuf = np.ascontiguousarray(B.T)
    sbuf = None if scale is None else np.ascontiguousarray(scale)
    check(lib().afqmc_test_real_gemm(ctx().h, precision, op_t, M, N, K, dptr(Abuf), dptr(Bbuf), dptr(sbuf), group,
                                     b_real, dptr(C)))
    S = 1.0 if scale is None else scale[np.arange(N) // group].T
    if b_real:
        B, S = B.real, np.real(S)
    ref = A @ (S * B)
    assert np.max(np.abs(C.T - ref)) <= 4 * (K + 4) * EPS[precision]
    if b_real:
        assert np.all(C.imag == 0)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("M,N", [(1, 1), (9, 3), (16, 16), (33, 17), (40, 31), (64, 48), (100, 63), (144, 65), (256, 112),
                                 (300, 128)])
def test_walker_products_match_numpy(precision, M, N):
    """W B (general and upper triangular B, in place) and W^T W; FP32 walkers take FP64 products, so
    only the stored result is rounded to FP32.  Dead walkers are left alone."""
    rng = np.random.default_rng(M + N)
    nw = 5
    W = rng.uniform(-1, 1, (nw, M, N))
    if precision:
        W = W.astype(np.float32).astype(np.float64)
    alive = np.array([1, 0, 1, 1, 1], dtype=np.int32)
    Wbuf = np.ascontiguousarray(W.transpose(0, 2, 1)).astype(np.complex128)
    for upper in (0, 1):
        B = rng.uniform(-1, 1, (nw, N, N))
        B = np.triu(B) if upper else B
        Bbuf = np.ascontiguousarray(B.transpose(0, 2, 1)).astype(np.complex128)
        out = np.zeros_like(Wbuf)
        check(lib().afqmc_test_walker_panel(ctx().h, precision, 1, M, N, nw, dptr(Wbuf), dptr(Bbuf), upper, iptr(alive),
                                            dptr(out)))
        ref = np.where(alive[:, None, None] != 0, W @ B, W).transpose(0, 2, 1)
        bound = 2 * (N + 2) * EPS[0] + (2 * N * EPS[1] if precision else 0.0)
        assert np.max(np.abs(out - ref)) <= bound
    out = np.zeros((nw, N, N), dtype=np.complex128)
    check(lib().afqmc_test_walker_panel(ctx().h, precision, 2, M, N, nw, dptr(Wbuf), None, 0, iptr(alive), dptr(out)))
    ref = np.where(alive[:, None, None] != 0, W.transpose(0, 2, 1) @ W, 0.0)
    assert np.max(np.abs(out - ref)) <= 2 * (M + 2) * EPS[0]
    assert np.array_equal(out, out.transpose(0, 2, 1))


def pair(nx, ny, nup, ndn, dense, precision, nw=4, decomp="densitySpin", U=6.0, seed=3):
    """Two propagators with real walkers and the same walkers with a phase on their first column."""
    model = HubbardModel.square(nx, ny, nup + ndn, U)
    L = model.L
    phi = free_electron_trial(model) if dense else spin_block_trial(model, nup, ndn)
    m = CPMethod(dt=0.02, decompType=decomp, walkerSizePerThread=nw)
    rng = np.random.default_rng(seed)
    wfs = []
    for _ in range(nw):
        w = np.zeros_like(phi)
        noise = 0.3 / np.sqrt(L) * rng.uniform(-1, 1, phi.shape)
        w[:] = phi + (noise if dense else np.where(phi_mask(L, nup, phi.shape), noise, 0.0))
        wfs.append(w)
    logw = 0.1 * rng.uniform(-1, 1, nw) + 0j
    theta = 0.6
    out = []
    for phase in (0.0, theta):
        prop = CPPropagator(ctx(), model, m, phi, nup=nup, spin_blocks=not dense, precision=precision, max_walkers=nw)
        prop.set_seed(11)
        prop.set_ET(-3.0)
        ws = prop.walkers(nw)
        up = [w.copy() for w in wfs]
        for w in up:
            w[:, 0] *= np.exp(1j * phase)
        ws.upload(up, logw - 1j * phase)
        out.append((prop, ws))
    return out


def phi_mask(L, nup, shape):
    mask = np.zeros(shape, dtype=bool)
    mask[:L, :nup] = mask[L:, nup:] = True
    return mask


def same(a, b, rtol):
    a, b = np.asarray(a), np.asarray(b)
    assert np.max(np.abs(a - b)) <= rtol * max(1e-300, np.max(np.abs(b))), np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,nup,ndn,dense", [(3, 3, 1, 2, False), (4, 4, 5, 7, False), (6, 6, 16, 15, False),
                                                 (6, 6, 17, 18, False), (9, 7, 31, 28, False), (12, 12, 64, 65, False),
                                                 (16, 16, 112, 97, False), (17, 16, 129, 128, False),
                                                 (3, 3, 2, 2, True), (4, 4, 5, 5, True), (8, 8, 28, 29, True)])
def test_real_walkers_equal_the_general_path(precision, nx, ny, nup, ndn, dense):
    # 30 roundings' worth of FP64; FP32 overlaps of up to 129 electrons lose about 1e-5 in log det
    rtol = 1e-10 if precision == 0 else 2e-3
    (pr, wr), (pc, wc) = pair(nx, ny, nup, ndn, dense, precision)
    same(np.exp(pr.log_overlap(wr)), np.exp(pc.log_overlap(wc)), rtol)
    for a, b in zip(pr.green_diagonal(wr), pc.green_diagonal(wc)):
        same(a + 1.0, b + 1.0, rtol)  # off-diagonal parts may be zero
    for i in range(2):
        (fr, xr), (fc, xc) = pr.step(wr, record=True), pc.step(wc, record=True)
        on = wr.alive() != 0
        assert np.array_equal(on, wc.alive() != 0) and on.any()
        assert np.array_equal(xr[on], xc[on])
        assert np.max(np.abs(fr[on] - fc[on])) <= rtol
        pr.stabilize(wr)
        pc.stabilize(wc)
    for p, w in ((pr, wr), (pc, wc)):
        p.onebody(w, 1)
        p.measure(w)
    er, ec = pr.energy(), pc.energy()
    same([er[k] for k in ("den", "HNum", "KNum", "VNum")], [ec[k] for k in ("den", "HNum", "KNum", "VNum")], rtol)
    same(pr.site_measure(), pc.site_measure(), rtol)
    wt, tb, _ = pr.pop_control(wr, record=True)
    wt2, tb2, _ = pc.pop_control(wc, record=True)
    same(wt, wt2, rtol)
    wf, _, _ = wr.download()
    assert np.all(wf.imag == 0)


def test_graph_of_real_walkers_serves_complex_ones():
    """A graph captured while the walkers are real, launched after complex walkers were uploaded,
    gives what the calls themselves give, and real walkers uploaded later take the graph again."""
    (pr, wr), (pc, wc) = pair(4, 4, 5, 5, False, 0)
    real, _, _ = wr.download()
    c, _, _ = wc.download()
    ctx().capture_begin()
    pr.step(wr)
    pr.stabilize(wr)
    pr.measure(wr)
    g = ctx().capture_end()
    for k, w in enumerate((real, c, real, c)):
        wr.upload(w)
        wc.upload(w)
        for p in (pr, pc):
            p.reset_measure()
            p.set_seed(5 + k)
        for _ in range(3):
            g.launch()
            pc.step(wc)
            pc.stabilize(wc)
            pc.measure(wc)
            ctx().synchronize()
        a, b = wr.download(), wc.download()
        same(a[0], b[0], 1e-12)
        same(a[1] + 1.0, b[1] + 1.0, 1e-12)
        same(list(pr.energy().values()), list(pc.energy().values()), 1e-11)
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [1, 2, 4, 5, 15, 16, 17, 32, 33, 48, 49, 63, 64, 65, 80, 81, 97, 112, 113, 128, 129, 160])
def test_gj_real_matches_lapack(precision, N):
    """Inverse and log-determinant of real matrices in every size class, with a permutation, a
    singular matrix and a badly scaled one among them.  A backward-stable inverse is within cond * N eps of the exact one; FP32 storage rounds the input-independent result once."""
    rng = np.random.default_rng(N)
    A = rng.standard_normal((6, N, N))
    A[1] = np.eye(N)[rng.permutation(N)]
    A[2] *= 1e-30 if precision else 1e-140
    A[3] = A[3] @ np.diag(np.logspace(0, -6, N))
    if precision:
        A = A.astype(np.float32).astype(np.float64)
    A[4][:, -1] = 0.0
    alive = np.array([1, 1, 1, 1, 1, 0], dtype=np.int32)
    Ainv, ld, info = gj_inverse_masked(A, alive, 16, precision, fill=7.0)
    assert list(info[:5]) == [0, 0, 0, 0, 1]
    assert np.array_equal(Ainv[5], A[5]) and ld[5] == 7.0
    for b in range(4):
        ref = np.linalg.inv(A[b])
        cond = np.linalg.cond(A[b], 2)
        bound = 8 * N * cond * EPS[0] + (2 * EPS[1] if precision else 0.0)
        assert np.max(np.abs(Ainv[b] - ref)) <= bound * np.max(np.abs(ref))
        assert np.all(Ainv[b].imag == 0)
        sign, logabs = np.linalg.slogdet(A[b])
        assert abs(ld[b].real - logabs) <= 8 * N * cond * EPS[0] * max(1.0, abs(logabs))
        assert abs(np.exp(1j * ld[b].imag) - sign) < 1e-12


@pytest.mark.parametrize("N", [1, 3, 16, 17, 33, 64, 65, 97, 112, 113, 128, 129, 160])
def test_chol_real_matches_lapack(N):
    rng = np.random.default_rng(N)
    W = rng.standard_normal((4, N + 20, N))
    S = np.ascontiguousarray(W.transpose(0, 2, 1) @ W).astype(np.complex128)
    out, ld, info = np.zeros_like(S), np.zeros(4, dtype=np.complex128), np.zeros(4, dtype=np.int32)
    S[3] -= 1.01 * np.linalg.eigvalsh(S[3])[-1] * np.eye(N)  # not positive definite
    check(lib().afqmc_test_chol_inverse_real(ctx().h, N, 4, dptr(S), dptr(out), dptr(ld), iptr(info)))
    assert list(info) == [0, 0, 0, 1]
    for b in range(3):
        R = np.linalg.cholesky(S[b].real).T
        ref = np.linalg.inv(R)
        cond = np.linalg.cond(S[b].real)
        got = out[b].T  # column-major
        assert np.max(np.abs(got - ref)) <= 8 * N * cond * EPS[0] * np.max(np.abs(ref))
        assert np.all(np.tril(got, -1) == 0) and np.all(got.imag == 0)
        assert abs(ld[b].real - np.sum(np.log(np.diag(R)))) <= 8 * N * cond * EPS[0]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,nup,ndn", [(4, 4, 1, 5), (6, 6, 16, 17), (8, 8, 33, 31), (12, 12, 64, 65), (16, 16, 112, 128)])
def test_qr_of_ill_conditioned_real_walkers(precision, nx, ny, nup, ndn):
    """Orthonormal result, log det R and the span for well- and ill-conditioned walkers (nearly
    parallel columns, which take the shifted pass); a walker with two equal columns dies."""
    model = HubbardModel.square(nx, ny, nup + ndn, 4.0)
    L, nw = model.L, 6
    phi = spin_block_trial(model, nup, ndn)
    m = CPMethod(dt=0.02, walkerSizePerThread=nw)
    prop = CPPropagator(ctx(), model, m, phi, nup=nup, spin_blocks=True, precision=precision, max_walkers=nw)
    rng = np.random.default_rng(nup)
    wfs = []
    for k in range(nw):
        w = np.where(phi_mask(L, nup, phi.shape), rng.uniform(-1, 1, phi.shape), 0.0) + 0j
        if k == 2:  # condition about 1e6
            w[L:, -1] = w[L:, -2] + 1e-6 * w[L:, -1]
        if k == 3:
            w[L:, -1] = w[L:, -2]
        if k == 4:
            w *= 1e4
        wfs.append(w if precision == 0 else w.astype(np.complex64).astype(np.complex128))
    ws = prop.walkers(nw)
    ws.upload(wfs, np.zeros(nw))
    prop.stabilize(ws)
    q, lw, alive = ws.download()
    eps = 1e-12 if precision == 0 else 4e-6
    assert list(alive[[0, 1, 2, 4, 5]]) == [1, 1, 1, 1, 1]
    # equal columns: dead, or (a last rounding apart) a log-weight that weighs nothing
    assert alive[3] == 0 or lw[3].real < lw[0].real - 20
    shifted, killed = prop.qr_stats()
    assert shifted >= 1 and killed == 1 - alive[3]
    for k in (0, 1, 2, 4, 5):
        Q = q[k]
        assert np.max(np.abs(Q.conj().T @ Q - np.eye(nup + ndn))) < eps
        R = np.linalg.qr(wfs[k])[1]
        # log det R: u kappa^2 of an unshifted Cholesky (kappa <= 1e3 here), and u kappa c with the
        # shift's c = 11 (M N + N^2) <= 1e6 for the walker with kappa = 1e6
        ref = np.sum(np.log(np.abs(np.diag(R))))
        assert abs(lw[k].real - ref) < (1e-4 if k == 2 else 1e-9) * max(1.0, abs(ref))
        R = Q.conj().T @ wfs[k]  # upper triangular with a positive diagonal: Q spans W
        size = np.max(np.abs(R))
        assert np.max(np.abs(np.tril(R, -1))) < 20 * eps * size
        assert np.all(np.diag(R).real > 0)
        assert np.max(np.abs(Q @ R - wfs[k])) < 20 * eps * size


@pytest.mark.parametrize("nw", [1, 63, 1023, 1024, 1025, 2049])
def test_step_head_numbers_the_alive_walkers(nw):
    """The uniforms of a step: walker w draws its own from (alive walkers before it) L on, whatever
    the population's size and with dead walkers in between; the counter moves by (alive) L."""
    model = HubbardModel.square(3, 3, 4, 4.0)
    L = model.L
    phi = spin_block_trial(model, 2, 2)
    rng = np.random.default_rng(nw)
    dead = rng.uniform(size=nw) < 0.3
    dead[0] = False
    wfs = [phi + np.where(phi != 0, 0.05 * rng.uniform(-1, 1, phi.shape), 0.0) for _ in range(nw)]
    got = []
    for n in (nw, max(1, nw // 2)):  # the first half alone draws the same fields
        prop = CPPropagator(ctx(), model, CPMethod(dt=0.02, walkerSizePerThread=n), phi, nup=2, spin_blocks=True,
                            precision=0, max_walkers=n)
        prop.set_seed(11, 5)
        ws = prop.walkers(n)
        ws.upload(wfs[:n], np.zeros(n), (~dead[:n]).astype(np.int32))
        _, aux = prop.step(ws, record=True)
        al = ws.alive()
        assert not np.any(al[dead[:n]])
        assert prop.counter() == 5 + int(np.sum(al != 0)) * L
        got.append(np.where(al[:, None] != 0, aux, 0))
    assert np.array_equal(got[0][:len(got[1])], got[1])


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nup,col", [(1, 0), (5, 0), (5, 4), (20, 19)])
def test_walkers_whose_overlap_overflows_weigh_nothing(precision, nup, col):
    """A walker whose overlap with the trial is beyond the largest number has no usable weight: it counts as
    one of overlap zero (log-overlap -1e300, weight 0, killed by the comb) and leaves the others alone,
    with real walkers and with complex ones."""
    nx = 4 if nup < 10 else 7
    (pr, wr), (pc, wc) = pair(nx, nx, nup, nup, False, precision, nw=4)
    big = 3e38 if precision else 1.7e308
    model = HubbardModel.square(nx, nx, 2 * nup, 6.0)
    phi = spin_block_trial(model, nup, nup)
    L = model.L
    assert np.sum(np.abs(phi[:L, col])) > 1.2 * (3.41 / 3 if precision else 1.8 / 1.7)
    for p, w, phase in ((pr, wr, 1.0), (pc, wc, np.exp(0.6j))):
        wf, lw, _ = w.download()
        good = p.log_overlap(w)
        x = big * np.sign(phi[:L, col].real)
        wf[2, :L, col] = x * (phase if col == 0 else 1.0)
        w.upload(wf, lw)
        lo = p.log_overlap(w)
        assert lo[2].real < -1e299 and np.array_equal(lo[[0, 1, 3]], good[[0, 1, 3]])
        weight, table, _ = p.pop_control(w, record=True)
        assert weight[2] == 0 and np.all(weight[[0, 1, 3]] > 0) and np.all(np.isfinite(weight))
        assert 2 not in table and np.all(w.alive() != 0)
