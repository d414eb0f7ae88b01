"""The blocked history sums (far sums once per block of steps, the newest slots
in the sweep) at the edges of a block and at grids of every launch variant.

Tolerances: FP64, 1e-12 norm-wise relative error against the oracle, as the
plain path's; FP32 increments, 1e-6 (each rounds at 2^-24 of itself, the sums
are FP64); the SOE form, 1e-6 (the bar its fit is held to at creation)."""
import numpy as np
import pytest

from oracle import oracle as O
from theses_code_amd import _native as N
from theses_code_amd import solvers as S

pytestmark = pytest.mark.gpu
B = 16  # steps per block


@pytest.fixture(scope="module")
def ctx():
    c = N.Context(0)
    yield c
    c.close()


def relerr(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def _case(sN, M):
    rng = np.random.default_rng(sN + 1000 * M)
    nn = (sN + 2) * (M + 2)
    vx, vy = rng.uniform(-0.1, 0.1, (2, nn))
    return S.coefs_advection(vx, vy, 1e-3, 1.0 / (sN + 1)), rng.uniform(0, 1, nn)


# the one-workgroup path at the edges of its lanes, nodes per thread and LDS;
# then fewer nodes than 2^15, than 2^18, and more (one launch variant each)
@pytest.mark.parametrize("precision,tol", [(N.PREC_F64, 1e-12), (N.PREC_F32C, 1e-6),
                                           (N.PREC_SOE, 1e-6), (N.PREC_MFMA_BF16, 1e-6)])
@pytest.mark.parametrize("sN,M", [(2, 2), (3, 2), (33, 32), (33, 34), (40, 33), (65, 20), (20, 65),
                                  (66, 20), (41, 33), (201, 188), (530, 511)])
def test_lod2d_blocks_match_oracle(ctx, sN, M, precision, tol):
    coefs, C0 = _case(sN, M)
    steps = 2 * B + 5
    o = O.TGSolver(sN, M, 0.7, 1e-3, 1.0, 0.0, 0.05, *coefs, C0)
    g = S.TGSolver(ctx, sN, M, 0.7, 1e-3, 1.0, coefs, C0, capacity=steps, C1=0.0, S=0.05,
                   precision=precision)
    t = 0
    for k in (1, B // 2 - 1, B // 2, B // 2 + 1, B - 1, B, B + 1, 2 * B, steps):  # calls that end on, before and after a block
        o.step(k - t)
        g.calc_step(k - t)
        t = k
        assert relerr(g.b_C, o.state().reshape(M + 2, sN + 2)) <= tol, k
    whole = g.b_C
    g.set_state(C0)
    g.calc_step(steps)  # one call: the same blocks, bit for bit
    assert np.array_equal(g.b_C, whole)
    g.close()


# chunks of 6, 12 and 24 unknowns per lane: lines that fill their last lane, and
# one unknown more than the shape before holds
@pytest.mark.parametrize("precision,tol", [(N.PREC_F64, 1e-12), (N.PREC_MFMA_BF16, 1e-6)])
@pytest.mark.parametrize("W,n", [(1, 257), (1, 384), (1, 513), (1, 768), (1, 1025), (1, 1536),
                                 (2, 768), (2, 1025), (2, 3072), (4, 1536), (4, 3072), (4, 4097),
                                 (4, 6144)])
def test_lod2d_chunks_of_six_twelve_and_24(ctx, W, n, precision, tol):
    for sN, M in ((n + 1, 11), (11, n + 1)):
        coefs, C0 = _case(sN, M)
        steps = 3
        o = O.TGSolver(sN, M, 0.7, 1e-3, 1.0, 0.0, 0.05, *coefs, C0)
        g = S.TGSolver(ctx, sN, M, 0.7, 1e-3, 1.0, coefs, C0, capacity=steps, C1=0.0, S=0.05,
                       precision=precision, sweep_w=W)
        cm = g.sweep_shape[0 if sN > M else 1][0]
        assert cm in (6, 12, 24) and 64 * W * cm >= n
        o.step(steps)
        g.calc_step(steps)
        assert relerr(g.b_C, o.state().reshape(M + 2, sN + 2)) <= tol
        g.close()


# coefficients that all rows, all columns, both or all but one line share (the
# sweeps then read one line's); 1e-12 as above, 1e-9 for g(t) = t^p, whose
# weights' series stop at int_err = 1e-10 on both sides
@pytest.mark.parametrize("g", [dict(), dict(g_func=3, g_pow=0.8, int_err=1e-10)])
@pytest.mark.parametrize("alike", ["rows", "cols", "both", "all but the last row's last"])
def test_lod2d_lines_with_the_same_coefficients(ctx, alike, g):
    sN, M, steps = 70, 67, 5
    rng = np.random.default_rng(5)
    vx = np.full((M + 2, sN + 2), 0.03)
    vy = np.full((M + 2, sN + 2), -0.02)
    if alike == "rows":
        vx[:], vy[:] = rng.uniform(-0.1, 0.1, (2, sN + 2))
    elif alike == "cols":
        vx[:], vy[:] = rng.uniform(-0.1, 0.1, (2, M + 2))[:, :, None]
    elif alike != "both":
        vx[M - 1, sN - 1] = 0.1
    coefs = S.coefs_advection(vx.reshape(-1), vy.reshape(-1), 1e-3, 1.0 / (sN + 1))
    C0 = rng.uniform(0, 1, (sN + 2) * (M + 2))
    orc = dict(func=3, fpow=g["g_pow"], int_err=g["int_err"]) if g else {}
    o = O.TGSolver(sN, M, 0.7, 1e-3, 1.0, 0.0, 0.05, *coefs, C0, **orc)
    s = S.TGSolver(ctx, sN, M, 0.7, 1e-3, 1.0, coefs, C0, capacity=steps, C1=0.0, S=0.05, **g)
    o.step(steps)
    s.calc_step(steps)
    assert relerr(s.b_C, o.state().reshape(M + 2, sN + 2)) <= (1e-9 if g else 1e-12)
    s.close()


@pytest.mark.parametrize("keep", [1, B - 1, B, B + 5, 2 * B])
def test_lod2d_restricted_sums_across_blocks(ctx, keep):
    sN, M, steps = 41, 33, 3 * B + 2
    coefs, C0 = _case(sN, M)
    _, _, _, wr, wc = N.host_caputo_lod_weights(0.7, 1e-3, steps)
    eps = 0.5 * (wc[keep - 1] + wc[keep])  # columns keep `keep` lags
    o = O.TGSolver(sN, M, 0.7, 1e-3, 1.0, 0.0, 0.0, *coefs, C0, dt2=eps)
    g = S.TGSolver(ctx, sN, M, 0.7, 1e-3, 1.0, coefs, C0, capacity=steps, C1=0.0, trunc_eps=eps)
    o.step(steps)
    g.calc_step(steps)
    assert relerr(g.b_C, o.state().reshape(M + 2, sN + 2)) <= 1e-12
    g.close()


def _mt_prob(n, rng, kind):
    p = dict(N=n, L=1.0, alpha=float(rng.uniform(0.5, 0.9)))
    if kind == N.MT_AB:
        p.update(src=int(rng.integers(0, 3)), ab_maxl=50, ab_maxkiter=1000, ab_eps=1e-10)
        return p, np.zeros(n + 2)
    p.update(beta=float(rng.uniform(0.6, 1.4)), form=N.FORM_KEXP, k0=2e-3, b=1.0,
             top=N.TOP_DIRICHLET, top_val=0.4, bottom_cond=1, Hbottom=0.2)
    u = rng.uniform(0.1, 0.4, n + 2)
    u[0], u[n], u[n + 1] = 0.4, 0.2, 0.2
    return p, u


# A batch large enough that every wavefront of the far sums takes four nodes
# of one problem and its whole history, against its problems one by one (a
# node's history split among wavefronts).  The sums are the same products in
# FP64 in two orders; FP32 increments may round differently where the states
# differ in the last bit.  Calls that end on and around a block's edges.
@pytest.mark.parametrize("kind", [N.MT_L1, N.MT_PSI, N.MT_AB])
@pytest.mark.parametrize("precision,tol", [(N.PREC_F64, 1e-12), (N.PREC_F32C, 1e-6)])
def test_mt1d_large_batch_matches_single_problems(ctx, kind, precision, tol):
    if kind == N.MT_AB and precision == N.PREC_F32C:
        pytest.skip("the Atangana-Baleanu batch is FP64")
    rng = np.random.default_rng(7)
    sizes = [2, 3, 65, 66, 129, 256, 257, 258, 513, 770, 1025] + [128] * 1024
    pairs = [_mt_prob(n, rng, kind) for n in sizes]
    tau, steps = (1.0 / 400 if kind == N.MT_AB else 1e-3), 3 * B + 4
    probs, U0 = [p for p, _ in pairs], [u for _, u in pairs]
    b = S.MT1DBatch(ctx, probs, tau, steps, U0, kind=kind, precision=precision)
    t = 0
    for k in (1, 2, 3, B - 1, B + 1, B + 2, B + 3, 2 * B, steps):
        b.calc_step(k - t)
        t = k
    got = b.state()
    b.set_state(U0)
    b.calc_step(steps)
    assert all(np.array_equal(x, y) for x, y in zip(got, b.state()))
    b.close()
    for q in list(range(12)) + [500, len(sizes) - 1]:
        s = S.MT1DBatch(ctx, [probs[q]], tau, steps, [U0[q]], kind=kind, precision=precision)
        s.calc_step(steps)
        assert relerr(got[q], s.state()[0]) <= tol, sizes[q]
        s.close()


# The series history of several steps per launch, at the edges of its launch
# variants (nodes per wavefront, accumulators that just fit LDS and that do
# not), beside a full-history problem, in calls that end inside and across its
# runs; the last case's accumulators overflow, so that sums restart from the
# sorted pyramid.  Bar: 1e-12 against the oracle, as the series path's.
@pytest.mark.parametrize("N_,maxl,alpha,tau,steps", [
    (2, 3, 0.5, 0.01, 20), (64, 50, 0.6, 0.01, 40), (65, 50, 0.2, 0.01, 40), (66, 50, 0.9, 0.02, 60),
    (129, 50, 0.7, 0.01, 40), (130, 17, 0.4, 0.02, 60), (190, 50, 0.6, 0.01, 20),
    (200, 50, 0.6, 0.01, 20), (330, 20, 0.6, 0.01, 20), (8, 600, 0.3, 0.05, 80)])
def test_ab_series_fused_steps_match_oracle(ctx, N_, maxl, alpha, tau, steps):
    series = dict(N=N_, alpha=alpha, src=2, ab_maxl=maxl, ab_maxkiter=1000, ab_eps=1e-10, ab_series=1)
    full = dict(N=40, alpha=0.6, src=1, ab_maxl=50, ab_maxkiter=1000, ab_eps=1e-10)
    _, ref = O.ab_solve_series(alpha, steps * tau, steps, N_, maxl, 1000, 1e-10, 2)
    _, ref_full = O.ab_solve(0.6, steps * tau, steps, 40, 50, 1000, 1e-10, 1)
    for probs in ([series], [series, full, series]):
        b = S.MT1DBatch(ctx, probs, tau, steps, [np.zeros(p["N"] + 2) for p in probs], kind=N.MT_AB)
        for k in (1, 2, B - 2, steps - B - 1):
            b.calc_step(k)
        got = b.state()
        b.close()
        for q, p in enumerate(probs):
            r = ref if "ab_series" in p else ref_full
            assert relerr(got[q][:p["N"] + 1], r) <= 1e-12, (q, len(probs))
