"""The projection of coordinates of very different sizes: a centre far from a point
still counts if its coordinate is large enough.

All terms are positive, so every one of them shows in the sum to its own relative
error: that of R, exponents of at most 700 and distances' chains of a few terms,
below 1e-12."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [dg.FP64, dg.MIXED])
@pytest.mark.parametrize("temp", [1.0, 3.0])
def test_far_centres_with_large_coordinates(temp, prec):
    print(f"case: map, wide coordinates, temp={temp} precision={prec}", flush=True)
    rng = np.random.default_rng(7)
    N, D, K, beta = 200, 6, 700, 0.02
    T = rng.normal(size=(N, D)) / np.sqrt(D)
    Y = rng.normal(size=(K, D)) / np.sqrt(D)
    far = np.r_[304:352]                       # whole groups of 16
    x0 = np.repeat([80.0, 300.0, 680.0], 16)   # their exponents, about
    u = rng.normal(size=(48, D))
    Y[far] = np.sqrt(2.0 * x0 / beta)[:, None] * u / np.linalg.norm(u, axis=1)[:, None]
    X = rng.uniform(0.5, 2.0, (K, 3))
    for l in range(3):
        X[far[16 * l:16 * l + 16], l] *= np.exp(x0[16 * l] / temp)
    x = -beta / 2 * ((T[:, None] - Y[None]) ** 2).sum(2)
    assert (x > -745.0).all()
    p = np.exp((x - x.max(1)[:, None]) / temp)
    want = p @ X / p.sum(1)[:, None]
    near = np.setdiff1d(np.arange(K), far)
    assert (want > 1.01 * (p[:, near] @ X[near]) / p[:, near].sum(1)[:, None]).all()
    with dg.Engine(precision=prec) as e:
        e.upload(T, np.ones((K, 1)), Y, beta)
        e.estep(True, temp)
        for M in (e.map(X), e.map_noalloc(X)):
            assert np.abs(M / want - 1.0).max() <= 1e-10
