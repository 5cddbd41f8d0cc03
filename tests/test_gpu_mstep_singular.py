"""The M-step where a factorisation meets a non-positive pivot: the retries with a
jitter (1e-13 tr(A) / n, growing tenfold, at most eight), and what follows a
failure, for both solvers (M + 1 <= 126 and above) against numpy.

A zero column of FI makes its pivot exactly 0, wherever it stands, and W's row of
it exactly 0.  The rest of A has a condition below 1e4 (K at least four times M + 1,
Gaussian FI), so the jitter moves W by 1e-9 of its largest entry at most and the
solution is good to 1e-10."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


def _problem(M1, D=5):
    rng = np.random.default_rng(M1)
    K, N = 4 * M1 + 3, 1200
    T = rng.normal(size=(N, D)) / np.sqrt(D)
    Y = rng.normal(size=(K, D)) / np.sqrt(D)
    return T, Y, rng.normal(size=(K, M1)), 0.5


def _solution(FI, G, RT, jitter):
    A = FI.T @ (FI * G[:, None])
    return np.linalg.solve(A + jitter * np.eye(len(A)), FI.T @ RT)


def _check(e, FI, T, N, D):
    G, RT = e.stats()
    beta = e.mstep()
    W, Y, _ = e.download()
    assert np.abs(Y - FI @ W).max() <= 1e-10 * np.abs(Y).max()
    s = (T * T).sum() - 2 * (Y * RT).sum() + (G * (Y * Y).sum(1)).sum()
    assert beta == pytest.approx(N * D / s, rel=1e-9)
    return G, RT, W, Y


@pytest.mark.parametrize("prec", [dg.FP64, dg.MIXED])
@pytest.mark.parametrize("M1", [26, 126, 127, 191, 260])
def test_zero_column_takes_a_jitter(M1, prec):
    T, Y0, FI, beta = _problem(M1)
    N, D = T.shape
    for col in sorted({0, 1, M1 // 2, 63 % M1, 64 % M1, M1 - 1}):
        print(f"case: M1={M1} precision={prec} zero column {col}", flush=True)
        F = FI.copy()
        F[:, col] = 0.0
        with dg.Engine(precision=prec, lam=0.0) as e:
            e.upload(T, F, Y0, beta)
            e.estep(True, 1.3)
            G, RT, W, _ = _check(e, F, T, N, D)
            jit = 1e-13 * np.trace(F.T @ (F * G[:, None])) / M1
            want = _solution(F, G, RT, jit)
            assert np.all(W[col] == 0.0)
            assert np.abs(W - want).max() <= 1e-8 * np.abs(want).max()


@pytest.mark.parametrize("M1", [26, 126, 127, 260])
def test_repeated_columns(M1):
    """A is singular, its pivot a rounding error of either sign: the centres are the
    projection all the same, good to 1e-16 times what cancels in W, 1e-6."""
    print(f"case: M1={M1}, repeated columns", flush=True)
    T, Y0, FI, beta = _problem(M1)
    FI[:, M1 - 2] = FI[:, 1]
    FI[:, M1 // 2] = FI[:, 0]
    with dg.Engine(precision=dg.FP64, lam=0.0) as e:
        e.upload(T, FI, Y0, beta)
        e.estep(True, 1.3)
        G, RT, W, Y = _check(e, FI, T, *T.shape)
        keep = np.setdiff1d(np.arange(M1), [M1 - 2, M1 // 2])
        want = FI[:, keep] @ _solution(FI[:, keep], G, RT, 0.0)
        assert np.abs(Y - want).max() <= 1e-6 * np.abs(want).max()


@pytest.mark.parametrize("prec", [dg.FP64, dg.MIXED])
@pytest.mark.parametrize("M1", [26, 126, 127, 260])
def test_failure_and_the_step_after_it(M1, prec):
    """A basis of zeros has no solution at any jitter (tr(A) = 0): DG_ESOLVE, no
    E-step left, and a good basis put in afterwards gives a fresh context's bits."""
    print(f"case: M1={M1} precision={prec}, zero basis", flush=True)
    T, Y0, FI, beta = _problem(M1)
    W0 = np.random.default_rng(1).normal(size=(M1, T.shape[1])) * 0.1
    out = []
    for fail in (True, False):
        with dg.Engine(precision=prec, lam=0.0) as e:
            e.upload(T, np.zeros_like(FI) if fail else FI, Y0, beta)
            if fail:
                e.estep(True, 1.3)
                with pytest.raises(dg.DgError) as ex:
                    e.mstep()
                assert ex.value.code == dg.DG_ESOLVE
                with pytest.raises(dg.DgError) as ex:
                    e.mstep()
                assert ex.value.code == dg.DG_ESTATE
            e.set_basis(FI, W0)
            e.estep(True, 1.3)
            b = e.mstep()
            out.append((b,) + e.download()[:2])
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
