"""The FP64 E-step at the edges of its tiles, against the CPU oracle.

Sizes around the 16- and 64-point tiles, the 16-, 64- and 512-centre steps, the
8- and 16-wide d steps and both ways pass 1 splits its work.  Both sides
sum at most a few thousand FP64 terms of like size, and the exponents stay
below 100 in magnitude, so they agree to about 100 * 2^-52 * a few: the bars
are those of test_gpu_fp64.py (1e-11 on the qualities, 1e-10 on the sums)."""
import numpy as np
import pytest

import dagtm_gpu as dg
import oracle as O

pytestmark = pytest.mark.gpu


def _problem(N, D, K, far=0):
    rng = np.random.default_rng(1000 * N + 10 * D + K)
    T = rng.normal(size=(N, D)) / np.sqrt(D)
    Y = rng.normal(size=(K, D)) / np.sqrt(D)
    T[:far] += 60.0                    # every exp underflows: zero columns
    return T, Y, np.ones((K, 1)), 6.0


@pytest.mark.parametrize("N,D,K,far", [
    (1, 1, 1, 0), (2, 3, 5, 0), (15, 8, 63, 0), (16, 9, 64, 0), (17, 16, 65, 1),
    (63, 17, 127, 0), (64, 24, 128, 0), (65, 25, 129, 2), (127, 31, 200, 0), (129, 33, 64, 0),
    (1000, 65, 130, 3), (257, 96, 70, 0), (300, 145, 67, 0), (200, 161, 80, 0), (131, 176, 40, 1),
    (90, 177, 66, 0), (333, 192, 100, 0),
    (16500, 12, 1030, 5), (5001, 40, 515, 0),
    (262143, 4, 17, 2), (262145, 5, 131, 1),            # either side of the split of pass 1
])
def test_estep_at_tile_edges(N, D, K, far):
    print(f"case: N={N} D={D} K={K} far={far}", flush=True)
    T, Y, FI, beta = _problem(N, D, K, far)
    for isDA, temp in ((1, 1.7), (0, 1.0)):
        m = O.Model(T, FI, Y, beta)
        llh_o, nf_o, nz_o = m.estep(isDA, temp)
        with dg.Engine(precision=dg.FP64) as e:
            e.upload(T, FI, Y, beta)
            llh, nf, nz = e.estep(isDA=isDA, temp=temp)
            G, RT = e.stats()
        assert nz == nz_o == far
        if np.isfinite(llh_o):
            assert llh == pytest.approx(llh_o, rel=1e-11, abs=1e-12)
        else:
            assert llh == llh_o
        assert nf == pytest.approx(nf_o, rel=1e-11, abs=1e-12)
        assert np.allclose(G, m.R.sum(1), rtol=1e-10, atol=1e-12)
        assert np.allclose(RT, m.R @ T, rtol=1e-10, atol=1e-10)


@pytest.mark.parametrize("N,D,K,far,L", [
    (1, 1, 1, 0, 1), (15, 8, 63, 1, 2), (64, 17, 128, 0, 3), (65, 25, 129, 2, 1), (1000, 40, 1100, 3, 2),
    (333, 192, 100, 0, 3), (9000, 12, 300, 4, 2),
])
def test_outputs_at_tile_edges(N, D, K, far, L):
    """Projection and dense R (always FP64) in both precisions, and G and R T
    read after them, against the oracle: R at most 1 and K of them to a sum, so
    1e-12 on R and 1e-11 on the projection of coordinates in [-1, 1]."""
    print(f"case: N={N} D={D} K={K} far={far} L={L}", flush=True)
    T, Y, FI, beta = _problem(N, D, K, far)
    X = np.random.default_rng(N + K).uniform(-1.0, 1.0, (K, L))
    m = O.Model(T, FI, Y, beta)
    m.estep(1, 1.7)
    for prec in (dg.FP64, dg.MIXED):
        if prec == dg.MIXED and D > 128:
            continue                   # float data: the mixed path stops at 128
        with dg.Engine(precision=prec) as e:
            e.upload(T, FI, Y, beta)
            e.estep(True, 1.7)
            assert np.abs(e.map(X) - m.R.T @ X).max() < 1e-11
            assert np.abs(e.map_noalloc(X) - m.R.T @ X).max() < 1e-11
            G, RT = e.stats()
            assert np.abs(e.resp_dense() - m.R).max() < 1e-12
            assert np.array_equal(G, e.stats()[0])
        assert np.allclose(G, m.R.sum(1), rtol=1e-10, atol=1e-12)
        assert np.allclose(RT, m.R @ T, rtol=1e-10, atol=1e-10)


@pytest.mark.parametrize("N,D,K", [
    (40, 1, 3), (61, 2, 5), (64, 15, 4), (65, 16, 9), (200, 17, 5), (700, 33, 20), (90, 64, 3),
    (150, 65, 4), (300, 128, 2), (260, 192, 3),
])
def test_ctemp_at_tile_edges(N, D, K):
    """The critical temperatures of every centre from numpy's moments and
    eigvalsh, at the edges of the moments' tiles and of the eigenvalue kernel:
    both sides are off by some units of 2^-52 of a matrix' norm, n <= 192 of
    them at worst, so 1e-11 of the norm."""
    print(f"case: ctemp N={N} D={D} K={K}", flush=True)
    T, Y, FI, beta = _problem(N, D, K)
    temp, eps = 1.7, 1e-6
    m = O.Model(T, FI, Y, beta)
    m.estep(1, temp)
    g = m.R.sum(1)
    with dg.Engine(precision=dg.FP64) as e:
        e.upload(T, FI, Y, beta)
        e.estep(True, temp)
        for t in (temp, 0.05, 1e6):            # some, hardly any, all eigenvalues below
            cmax, ck = e.next_ctemp(t, eps, g)
            for k in range(K):
                x, r = T - Y[k], m.R[k][:, None]
                S1, S2 = (x * r).T @ x, (x * r * r).T @ x
                w = np.concatenate([np.linalg.eigvalsh(2 * S1), np.linalg.eigvalsh(2 * (S1 - S2))])
                norm = np.abs(w).max()
                lim = (t - eps) * g[k] * 2 / beta
                if np.abs(w - lim).min() < 1e-10 * norm:
                    continue                   # on the limit: either side may take it
                want = beta / 2 / g[k] * np.where(w >= lim, 0.0, w).max()
                assert abs(ck[k] - want) <= 1e-11 * beta / 2 / g[k] * norm
            assert cmax == ck.max()


@pytest.mark.parametrize("N,D,K,M1", [
    (40, 1, 3, 1), (60, 3, 17, 5), (200, 17, 64, 26), (150, 12, 65, 31), (300, 33, 130, 32),
    (260, 50, 127, 63), (300, 15, 500, 64), (300, 166, 260, 65), (400, 180, 600, 126),
    (300, 20, 700, 127), (300, 40, 700, 130), (400, 65, 900, 257), (300, 33, 1100, 400),
    (300, 1, 300, 128), (300, 64, 300, 192), (350, 7, 400, 191),
])
def test_mstep_at_tile_edges(N, D, K, M1):
    """One M-step at the edges of the products' and the factorisation's tiles,
    against the same equations solved by numpy from the engine's own G and R T.
    A ridge of 1e-2 tr(A) / n keeps the condition below 1e2 n, and the chains are
    at most 1100 terms long, so 1e-10 of the largest entry."""
    print(f"case: mstep N={N} D={D} K={K} M1={M1}", flush=True)
    T, Y, _, beta = _problem(N, D, K)
    FI = np.random.default_rng(M1).normal(size=(K, M1))
    lam = 1e-2 * N / K * beta * K / 10.0
    with dg.Engine(precision=dg.FP64, lam=lam) as e:
        e.upload(T, FI, Y, beta)
        e.estep(True, 1.7)
        G, RT = e.stats()
        b = e.mstep()
        W, Yn, _ = e.download()
    Wr = np.linalg.solve(FI.T @ (FI * G[:, None]) + lam / beta * np.eye(M1), FI.T @ RT)
    Yr = FI @ Wr
    assert np.abs(W - Wr).max() <= 1e-10 * np.abs(Wr).max()
    assert np.abs(Yn - Yr).max() <= 1e-10 * np.abs(Yr).max()
    s = (T * T).sum() - 2 * (Yr * RT).sum() + (G * (Yr * Yr).sum(1)).sum()
    assert b == pytest.approx(N * D / s, rel=1e-10)
