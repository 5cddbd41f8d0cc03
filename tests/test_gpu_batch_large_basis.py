"""dg_batch_anneal where the batched M-step factorises by itself (M + 1 > 126): one
E+M step of each instance against its own dg_anneal.

The E-step's bits are those of a single context, so W differs by the two
factorisations' rounding alone: with Gaussian bases of four times as many rows and a
ridge A's condition is below 1e3, and chains of at most 300 terms leave 1e-10 of the
largest entry.  Host workers run dg_anneal itself: the same bits."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu

SIZES = [(900, 12, 127), (700, 33, 150), (800, 6, 25), (600, 20, 193), (500, 64, 260), (400, 3, 126)]


def _instances(zero=None):
    out = []
    for i, (N, D, M1) in enumerate(SIZES):
        rng = np.random.default_rng(M1)
        K = 4 * M1 + i
        T = rng.normal(size=(N, D)) / np.sqrt(D)
        FI = rng.normal(size=(K, M1))
        if zero == "basis" and M1 in (150, 126):
            FI[:] = 0.0
        if zero == "column":
            FI[:, M1 // 2] = 0.0
        out.append((T, FI, rng.normal(size=(K, D)) / np.sqrt(D), 0.5, dict(start_temp=1.5)))
    return out


@pytest.mark.parametrize("zero", [None, "column"])
@pytest.mark.parametrize("workers", [0, -1, 3])
def test_one_step(workers, zero):
    print(f"case: batch, large bases, workers={workers} zero={zero}", flush=True)
    lam = 0.0 if zero else 1e-3
    probs = _instances(zero)
    kw = dict(maxloop=1, alpha=0.9, eps=0.0)
    out, _ = dg.batch_anneal(probs, precision=dg.MIXED, lam=lam, workers=workers, **kw)
    for p, (st, r, W, Y) in zip(probs, out):
        M1 = p[1].shape[1]
        assert st == dg.DG_OK and r.nloop == 1
        with dg.Engine(precision=dg.MIXED, lam=lam) as e:
            e.upload(*p[:4])
            rs, _ = e.anneal(isDA=True, **kw, **p[4])
            Ws, Ys, _ = e.download()
        assert (r.llh, r.nfree) == (rs.llh, rs.nfree)
        if workers > 0 or M1 <= 126:
            assert r.beta == rs.beta and np.array_equal(W, Ws) and np.array_equal(Y, Ys), M1
        else:
            assert r.beta == pytest.approx(rs.beta, rel=1e-10)
            assert np.abs(W - Ws).max() <= 1e-10 * np.abs(Ws).max(), M1
            assert np.abs(Y - Ys).max() <= 1e-10 * np.abs(Ys).max(), M1
        if zero:
            assert np.all(W[M1 // 2] == 0.0)


@pytest.mark.parametrize("workers", [0, -1, 3])
def test_a_failing_basis_stops_its_own_instance_only(workers):
    print(f"case: batch, bases of zeros, workers={workers}", flush=True)
    out, _ = dg.batch_anneal(_instances("basis"), precision=dg.MIXED, lam=0.0, workers=workers,
                             maxloop=2, alpha=0.9, eps=0.0)
    want = [dg.DG_ESOLVE if M1 in (150, 126) else dg.DG_OK for _, _, M1 in SIZES]
    assert [o[0] for o in out] == want
    assert all(o[1].nloop == 2 and np.isfinite(o[3]).all() for o, w in zip(out, want) if w == dg.DG_OK)
