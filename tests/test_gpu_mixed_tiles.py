"""The mixed E-step where its set-up kernels and the sums of its chunk partials
have edges, against the FP64 path.

Centres around the 64 and the 4 rows (D of R T, one of G) of a summing workgroup,
more than 256 chunks, points around the 64 and 128 of the set-up kernels, in every
class of D.  The data are exact in FP16, so the bars are the binary ones of
test_gpu_mixed.py: 2e-6 on the qualities (absolute near zero), 1e-5 of the largest
entry on G and R T; the responsibilities of a point sum to 1 within FP32, 1e-5."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,K", [
    (1, 1, 1), (2, 2, 5), (63, 3, 63), (64, 4, 64), (65, 5, 65), (127, 16, 127), (128, 17, 128),
    (129, 33, 129), (1000, 48, 130), (777, 49, 257), (500, 96, 200), (300, 128, 70), (400, 166, 191),
    (260, 192, 64), (40001, 6, 40), (70003, 12, 129),
])
def test_estep_at_setup_and_sum_edges(N, D, K):
    print(f"case: N={N} D={D} K={K}", flush=True)
    rng = np.random.default_rng(1000 * N + 10 * D + K)
    T = (rng.random((N, D)) < 0.4).astype(float)
    Y = T[rng.integers(0, N, K)] + 0.2 * rng.normal(size=(K, D))
    FI, beta = np.ones((K, 1)), 30.0 / (1 + D)
    out = []
    for precision in (dg.FP64, dg.MIXED):
        with dg.Engine(precision=precision) as e:
            e.upload(T, FI, Y, beta)
            out.append(e.estep(True, 1.5) + e.stats())
    (l64, f64, z64, G64, RT64), (l16, f16, z16, G16, RT16) = out
    assert z64 == z16 == 0
    assert l16 == pytest.approx(l64, rel=2e-6, abs=2e-6)
    assert f16 == pytest.approx(f64, rel=2e-6, abs=2e-6)
    assert np.abs(G16 - G64).max() <= 1e-5 * np.abs(G64).max()
    assert np.abs(RT16 - RT64).max() <= 1e-5 * np.abs(RT64).max()
    assert G16.sum() == pytest.approx(N, rel=1e-5)
