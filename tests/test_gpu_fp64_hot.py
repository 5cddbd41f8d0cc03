"""The FP64 path at the hottest temperatures: every centre whose exponent does not
underflow has the same share of a point, the others none, a point without any 1/K.
Shares are reciprocals of counts: 1e-14.  Their sums are compared with sums in
extended precision (a double sum of 262200 equal shares is off by 1e-12 itself)."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,K", [(300, 12, 400), (65, 3, 1), (64, 33, 130), (262200, 2, 5)])
@pytest.mark.parametrize("temp", [1e300, np.inf])
def test_equal_shares(N, D, K, temp):
    print(f"case: temp={temp} N={N} D={D} K={K}", flush=True)
    rng = np.random.default_rng(N + K)
    T = rng.normal(size=(N, D))
    Y = rng.normal(size=(K, D))
    T[:3] += 500.0                     # no centre in reach
    if K > 3:
        Y[3] += 400.0                  # in no point's reach
        T[5:7] += 300.0
        Y[4] += 300.0                  # the only one in reach of two points
    beta = 2.0
    live = ((T[:, None] - Y[None]) ** 2).sum(2) * (beta / 2) < 745.0 if N < 1000 else None
    if live is None:
        live = np.stack([((T - y) ** 2).sum(1) * (beta / 2) < 745.0 for y in Y], 1)
    cnt = live.sum(1)
    one = np.longdouble(1.0)
    R = np.where(cnt[:, None] > 0, live * (one / np.maximum(cnt, 1))[:, None], one / K)
    X = rng.uniform(-1.0, 1.0, (K, 2))
    with dg.Engine(precision=dg.FP64) as e:
        e.upload(T, np.ones((K, 1)), Y, beta)
        llh, nf, nz = e.estep(True, temp)
        G, RT = e.stats()
        M = e.map(X)
        Rg = e.resp_dense()
    assert nz == (cnt == 0).sum() == 3
    assert not np.isnan(nf)
    assert np.abs(Rg.T - R).max() <= 1e-14
    assert np.allclose(G, R.sum(0), rtol=1e-12, atol=1e-13)
    assert np.allclose(RT, R.T @ T, rtol=1e-11, atol=1e-9)
    assert np.abs(M - R @ X).max() <= 1e-13
