"""Critical temperatures where the eigenvalue kernel's matrices are far from order
one, or have structure, against numpy's eigvalsh of the same moments.

Weights.  A centre far from all points has responsibilities, and so moments, of
any size down to the smallest double: squares of their entries underflow from
about 1e-160 on.  The moments are built from R times 2^p, p undoing the size of
the centre's weight, and R from the exponents: at exponents of 700 and squared
distances of 2e5 both sides' R are off by at most 1e-11 (the norms' chains, D 2^-53
of a distance each, times beta / 2 = 0.01), the eigenvalues by n 2^-52 of the
norm: 1e-10 of the norm in all.

Structure.  With one centre at the origin R = 1 and the moment is T^T T: 1e-11 of
the norm, as in test_gpu_fp64_tiles.py."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 2, 12, 64, 70])
def test_ctemp_of_centres_of_hardly_any_weight(D):
    print(f"case: ctemp, far centres, D={D}", flush=True)
    rng = np.random.default_rng(D)
    N, beta = 300, 0.02
    T = rng.normal(size=(N, D)) / np.sqrt(D)
    # exponents about 0, 350 (weights 1e-150), 390, 480, 560 (1e-241), 600 and 690
    far = np.sqrt(2.0 * np.array([0.0, 350.0, 390.0, 480.0, 560.0, 600.0, 690.0]) / beta)
    u = rng.normal(size=(len(far), D))
    Y = far[:, None] * u / np.linalg.norm(u, axis=1)[:, None]
    K = len(Y)
    x = -beta / 2 * ((T[None] - Y[:, None]) ** 2).sum(2)           # K x N
    top = x.max(0)
    logR = x - top - np.log(np.exp(x - top).sum(0))
    g = np.exp(logR).sum(1)
    assert (g[1:] < 1e-140).all() and (g > 0).all() and (x > -745.0).all()
    eps = 1e-6
    with dg.Engine(precision=dg.FP64) as e:
        e.upload(T, np.ones((K, 1)), Y, beta)
        e.estep(True, 1.0)
        for t in (1.0, 0.01, 1e7):             # some, hardly any, all eigenvalues below
            cmax, ck = e.next_ctemp(t, eps, g)
            for k in range(K):
                m = logR[k].max()
                r = np.exp(logR[k] - m)[:, None]                   # R e^-m
                gk = r.sum()
                d = T - Y[k]
                S1, S2 = (d * r).T @ d, (d * r * r).T @ d * np.exp(m)
                w = np.concatenate([np.linalg.eigvalsh(2 * S1), np.linalg.eigvalsh(2 * (S1 - S2))])
                norm = np.abs(w).max()
                lim = (t - eps) * gk * 2 / beta
                if np.abs(w - lim).min() < 1e-9 * norm:
                    continue                   # on the limit: either side may take it
                want = beta / 2 / gk * np.where(w >= lim, 0.0, w).max()
                assert abs(ck[k] - want) <= 1e-10 * beta / 2 / gk * norm, (t, k, ck[k], want)
            assert cmax == ck.max()


def _structured(n):
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.normal(size=(n, n)))
    bi = np.eye(n) * rng.integers(1, 9, n)[:, None] + np.diag(np.ones(n - 1), 1)
    bi[n // 2 - 1, n // 2] = 0.0
    pair = np.kron(np.diag(rng.integers(1, 4, n // 2)), [[1.0, 1.0], [1.0, -1.0]])
    yield "diagonal", np.diag(np.arange(1.0, n + 1))
    yield "split tridiagonal", bi
    yield "repeated", pair
    yield "repeated, rotated", np.repeat([3.0, 1.0, 2.0], n)[:n, None] * Q
    yield "rank 5", rng.normal(size=(5, n))
    yield "wide", np.logspace(-6, 3, n)[:, None] * Q
    yield "one point at the centre", np.zeros((1, n))
    yield "large", 1e90 * rng.normal(size=(2 * n, n))
    yield "small", 1e-100 * rng.normal(size=(2 * n, n))


@pytest.mark.parametrize("n", [40, 166, 192])
def test_ctemp_of_structured_moments(n):
    eps = 1e-6
    for name, T in _structured(n):
        print(f"case: ctemp, {name} moment, D={n}", flush=True)
        g = np.array([float(len(T))])
        size = np.abs(T).max() or 1.0
        beta = 1.0 / size ** 2
        w = np.r_[np.sort(np.linalg.eigvalsh(2.0 * (T / size).T @ (T / size))), np.zeros(n)]
        norm = np.abs(w).max()
        with dg.Engine(precision=dg.FP64) as e:
            e.upload(T, np.ones((1, 1)), np.zeros((1, n)), beta)
            e.estep(True, 1.0)
            # limits above all of them, below the largest, and inside the spectrum
            for lim in (1e6 * (norm + 1.0), 0.999 * norm + 1e-3, w[n // 2] * 1.0001 + 1e-9 * norm):
                if np.abs(w - lim).min() < 1e-10 * norm:
                    continue
                cmax, ck = e.next_ctemp(lim / (2.0 * g[0]) + eps, eps, g)
                want = np.where(w >= lim, 0.0, w).max() / (2.0 * g[0])
                assert abs(ck[0] - want) <= 1e-11 * norm / (2.0 * g[0]) + 1e-290, (name, lim, ck[0], want)
                assert cmax == ck[0]
