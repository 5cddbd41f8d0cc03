"""What the FP64 outputs of a mixed context (projection, critical temperatures, dense
R) leave for the next reader of G and R T, and for an M-step: an FP64 context's bits,
whichever of them came first or last."""
import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,K", [(700, 12, 90), (262200, 3, 20)])
@pytest.mark.parametrize("temp", [1.0, 1.6])
def test_statistics_after_fp64_outputs(N, D, K, temp):
    rng = np.random.default_rng(N)
    T = rng.normal(size=(N, D))
    T[:2] += 90.0                      # zero columns
    FI, Y, beta = rng.normal(size=(K, 9)), rng.normal(size=(K, D)), 0.9
    X, g = rng.normal(size=(K, 2)), np.ones(K)
    calls = {"map": lambda e: e.map(X), "ctemp": lambda e: e.next_ctemp(temp, 1e-6, g)}
    if N * K < 1e6:
        calls["resp"] = lambda e: e.resp_dense()

    def after(prec, names):
        with dg.Engine(precision=prec, lam=1e-3) as e:
            e.upload(T, FI, Y, beta)
            e.estep(True, 3.0)
            e.next_ctemp(3.0, 1e-6, g)         # of an E-step that is gone by then
            e.estep(True, temp)
            got = [calls[n](e) for n in names]
            G, RT = e.stats()
            G2, _ = e.stats()
            assert np.array_equal(G, G2)
            b = e.mstep()
            out = [G, RT, b, *e.download()[:2]]
            e.estep(True, temp)
            return got, out, e.stats()

    _, want, last64 = after(dg.FP64, [])
    lasts = []
    for names in (["map"], ["ctemp"], ["map", "ctemp"], ["ctemp", "map"], ["resp"], ["resp", "map", "ctemp"]):
        if not all(n in calls for n in names):
            continue
        print(f"case: N={N} temp={temp} after {names}", flush=True)
        got, out, last = after(dg.MIXED, names)
        lasts.append(last)
        ref, _, _ = after(dg.FP64, names)
        for a, b in zip(out, want):
            assert np.array_equal(a, b)
        for a, b in zip(got, ref):
            assert all(np.array_equal(x, y) for x, y in zip(a, b))
    # the next E-step is a mixed one again
    for last in lasts:
        assert all(np.array_equal(x, y) for x, y in zip(last, lasts[0]))
        assert not np.array_equal(last[1], last64[1])
