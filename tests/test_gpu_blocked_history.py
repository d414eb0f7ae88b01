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


# fewer nodes than 2^15, than 2^18, and more (one launch variant each)
@pytest.mark.parametrize("precision,tol", [(N.PREC_F64, 1e-12), (N.PREC_F32C, 1e-6),
                                           (N.PREC_SOE, 1e-6), (N.PREC_MFMA_BF16, 1e-6)])
@pytest.mark.parametrize("sN,M", [(3, 2), (41, 33), (201, 188), (530, 511)])
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
