"""The work that a user of the DA-GTM engine has it do, as cases to be timed.

A case is one call, or a short run of calls, of the Python binding
(da-gtm_amd/dagtm_gpu.py) on one problem: N data points of D dimensions, a
latent grid of g^L centres and m^L basis functions plus the bias.

kind       one pass, as a program calls it
estep      one E-step at the resident state, and its statistics G and R T
iterate    resume from a saved state, `iters` E+M iterations at one
           temperature (the annealing loop with its progress rows), and the
           new W, Y and beta
map        an E-step and the projection of the points into the latent space
ctemp      the critical temperatures that the AUTO cooling schedule asks for
resp       an E-step and the whole responsibility matrix (the driver's -R)
batch      `n` uneven instances annealed in one call, set-up included

Data are Gaussian mixtures ("gmm", float data) or binary fingerprints ("fp").
The states are those of a run under way: a few EM iterations, in plain torch,
on a sample of the points.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "da-gtm_amd"))

import dagtm_gpu as dg  # noqa: E402
import datagen  # noqa: E402

LAMBDA = 1e-3                      # M-step ridge of the benchmark configurations
PRECISION = {"fp64": dg.FP64, "mixed": dg.MIXED, "mixed_r1": dg.MIXED_R1}
UNDERFLOW = -745.1332191019412     # exp(x) of a double is 0 below this


def _case(kind, data, N, D, L, g, m, precision, temp=2.0, iters=1, n=1):
    return {"kind": kind, "data": data, "N": N, "D": D, "L": L, "g": g, "m": m, "precision": precision,
            "temp": temp, "iters": iters, "n": n}


def listed():
    cases = {
        # the smallest configuration of the benchmark: launches and latency
        "estep_small_mixed": _case("estep", "gmm", 1000, 12, 2, 20, 5, "mixed"),
        # a stretch of the driver's default run (double precision) on it
        "iterate_small_fp64": _case("iterate", "gmm", 1000, 12, 2, 20, 5, "fp64", iters=20),
        # plain EM (temperature 1) on odd sizes, double precision
        "iterate_em_odd_fp64": _case("iterate", "gmm", 20011, 33, 3, 11, 4, "fp64", temp=1.0, iters=2),
        # float data of the batched workload's larger instances
        "iterate_float_mixed": _case("iterate", "gmm", 50021, 64, 2, 40, 5, "mixed", iters=4),
        # fingerprints, the benchmark's second configuration, in both precisions
        "iterate_fp_100k_mixed": _case("iterate", "fp", 100000, 166, 3, 20, 5, "mixed", iters=4),
        "estep_fp_100k_fp64": _case("estep", "fp", 100000, 166, 3, 20, 5, "fp64"),
        # the headline workload's E-step: the largest data
        "estep_fp_1m_mixed": _case("estep", "fp", 1000000, 166, 3, 20, 5, "mixed"),
        # a large grid with the largest configuration's basis (M + 1 = 1001):
        # the M-step weighs as much as the E-step
        "iterate_basis_1001_mixed": _case("iterate", "fp", 20011, 166, 3, 32, 10, "mixed", iters=2),
        # the output of a finished run: the projection, always in double precision
        "map_fp_mixed": _case("map", "fp", 30011, 166, 3, 20, 5, "mixed", temp=1.0),
        # a temperature change of the AUTO schedule
        "ctemp_float_fp64": _case("ctemp", "gmm", 5003, 32, 2, 20, 5, "fp64"),
        # the -R dump
        "resp_float_fp64": _case("resp", "gmm", 6007, 12, 2, 30, 5, "fp64", temp=1.0),
        # many small problems in one call
        "batch_mixed": _case("batch", "both", 16000, 64, 2, 20, 5, "mixed", iters=10, n=8),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["estep", "estep", "iterate", "iterate", "map", "ctemp", "resp", "batch"])
    data = "gmm" if kind in ("ctemp", "resp") else rng.choice(["gmm", "fp"])
    L = rng.choice([2, 3])
    g = rng.randint(10, 40) if L == 2 else rng.randint(5, 20)
    m = rng.randint(4, 8) if L == 2 else rng.randint(3, 5)
    D = rng.randint(4, 64) if data == "gmm" else rng.randint(100, 180)
    precision = rng.choice(["fp64", "mixed", "mixed", "mixed_r1"])
    temp = round(rng.uniform(1.5, 4.0), 3) if rng.random() < 0.7 else 1.0
    iters = rng.randint(2, 6) if kind == "iterate" else 1
    if kind == "estep":
        N = _log_int(rng, 1e3, 4e5 if precision != "fp64" else 8e4)
    elif kind == "iterate":
        N = _log_int(rng, 1e3, 1e5 if precision != "fp64" else 2e4)
    elif kind == "map":
        N = _log_int(rng, 1e3, 4e4)
    elif kind == "ctemp":
        N, precision, g = _log_int(rng, 1e3, 8e3), "fp64", min(g, 20 if L == 2 else 8)
        D = min(D, 40)
    elif kind == "resp":
        N, precision = _log_int(rng, 1e3, 8e3), rng.choice(["fp64", "mixed"])
        g = min(g, 30 if L == 2 else 10)
    else:
        return _case("batch", "both", _log_int(rng, 4e3, 2e4), 64, 2, rng.randint(10, 30), 5, "mixed",
                     temp=2.0, iters=rng.randint(5, 15), n=rng.randint(2, 8))
    return _case(kind, data, N, D, L, g, m, precision, temp, iters)


# ---- inputs ------------------------------------------------------------------

def _data(kind, N, D, seed):
    """N x D doubles on the GPU, made as da-gtm_amd/datagen.py makes them."""
    r = np.random.RandomState(seed % (1 << 31))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "gmm":
        means = torch.from_numpy(r.normal(0.0, 2.0, (3, D))).cuda()
        sds = torch.from_numpy(r.uniform(0.3, 1.0, (3, D))).cuda()
        comp = torch.randint(0, 3, (N,), generator=gen, device="cuda")
        return means[comp] + sds[comp] * torch.randn((N, D), generator=gen, device="cuda", dtype=torch.float64)
    p = r.beta(0.5, 2.0, (50, D))
    proto = torch.from_numpy(r.random_sample((50, D)) < p).cuda()
    pick = torch.randint(0, 50, (N,), generator=gen, device="cuda")
    flip = torch.rand((N, D), generator=gen, device="cuda") < 0.05
    return (proto[pick] ^ flip).double()


def _start(T, FI, X, temp, steps=6, sample=2048):
    """A state under way: the principal-plane start of datagen.pca_init and some
    EM iterations on a sample of the points.  Y and beta are rounded to single
    precision, so that they are the same numbers on every run."""
    S = T[:sample]
    mu = S.mean(0)
    ev, V = torch.linalg.eigh(torch.cov(S.T).cpu())
    ev, V, L = ev.flip(0), V.flip(1), X.shape[1]
    target = mu.cpu() + (X / X.std(0, correction=0)).cpu() @ (V[:, :L] * ev[:L].clamp(min=0).sqrt()).T
    A, B = (FI.T @ FI).cpu(), (FI.T @ target.cuda()).cpu()
    W = torch.linalg.solve(A + 1e-6 * A.diagonal().mean() * torch.eye(len(A), dtype=A.dtype), B)
    Y, beta = FI @ W.cuda(), 1.0 / max(float(ev[min(L, len(ev) - 1)]), 1e-12)
    for _ in range(steps):
        _, _, G, RT = _estep64(S, Y, beta, 1.0 / temp)
        _, Y, beta = _mstep64(S, FI, G, RT, beta)
    return Y.float().double(), float(np.float32(beta))


def _problem(case, seed):
    """(T, X, FI, Y, beta) on the GPU."""
    T = _data(case["data"], case["N"], case["D"], seed)
    X, FI = (torch.from_numpy(a).cuda() for a in
             datagen.latent_basis(case["L"], case["g"] ** case["L"], case["m"] ** case["L"], 1.0))
    Y, beta = _start(T, FI, X, case["temp"])
    return T, X, FI, Y, beta


def _instances(case, seed):
    """The batch's problems: sizes falling from N, float data and fingerprints in turn."""
    out = []
    for i in range(case["n"]):
        N = max(500, int(case["N"] * 0.7 ** i))
        data, D = ("gmm", (12, 32, 64)[i // 2 % 3]) if i % 2 == 0 else ("fp", 166)
        out.append(dict(case, data=data, N=N, D=D, temp=1.5 + 0.25 * (i % 4)))
    return [(c, _problem(c, seed * 64 + i)) for i, c in enumerate(out)]


def prepare(case, seed):
    if case["kind"] == "batch":
        items = [(T.cpu().numpy(), FI.cpu().numpy(), Y.cpu().numpy(), beta, {"start_temp": c["temp"]})
                 for c, (T, X, FI, Y, beta) in _instances(case, seed)]
        return {"case": case, "items": items}
    T, X, FI, Y, beta = _problem(case, seed)
    s = {"case": case, "isDA": case["temp"] != 1.0 or case["kind"] != "iterate", "X": X.cpu().numpy(),
         "Y": Y.cpu().numpy(), "beta": beta}
    s["engine"] = dg.Engine(precision=PRECISION[case["precision"]], lam=LAMBDA)
    s["engine"].upload(T.cpu().numpy(), FI.cpu().numpy(), s["Y"], beta)
    if case["kind"] == "ctemp":
        s["G"] = _estep64(T, Y, beta, 1.0 / case["temp"])[2].cpu().numpy()
    return s


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        done, _ = dg.batch_anneal(state["items"], precision=PRECISION[case["precision"]], lam=LAMBDA,
                                  maxloop=case["iters"], eps=0.0)
        return [{"status": st, "llh": r.llh, "nfree": r.nfree, "beta": r.beta, "W": W, "Y": Y} for st, r, W, Y in done]
    e = state["engine"]
    if case["kind"] == "iterate":
        e.set_state(state["Y"], state["beta"])
        _, rows = e.anneal(isDA=state["isDA"], maxloop=case["iters"], eps=0.0, start_temp=case["temp"])
        W, Y, beta = e.download()
        return {"nfree": np.array([r[3] for r in rows]), "llh": np.array([r[4] for r in rows]),
                "W": W, "Y": Y, "beta": beta}
    llh, nfree, nzero = e.estep(True, case["temp"])
    out = {"llh": llh, "nfree": nfree, "nzero": nzero}
    if case["kind"] == "estep":
        out["G"], out["RT"] = e.stats()
    elif case["kind"] == "map":
        out["M"] = e.map(state["X"])
    elif case["kind"] == "ctemp":
        out["max"], out["each"] = e.next_ctemp(case["temp"], 1e-6, state["G"])
    else:
        out["R"] = e.resp_dense()
    return out


# ---- what a pass cannot do without ------------------------------------------------

def work(case):
    if case["kind"] == "batch":
        parts = [work(dict(case, kind="iterate", data="", N=max(500, int(case["N"] * 0.7 ** i)),
                           D=(12, 32, 64)[i // 2 % 3] if i % 2 == 0 else 166)) for i in range(case["n"])]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    N, D, K, M1 = case["N"], case["D"], case["g"] ** case["L"], case["m"] ** case["L"] + 1
    data, model = 8.0 * N * D, 8.0 * K * D
    estep = 4.0 * K * N * D                            # the distances' cross term, and R T
    if case["kind"] == "estep":
        return {"bytes": data + 2 * model + 8.0 * K, "flops": estep}
    if case["kind"] == "iterate":
        mstep = 2.0 * K * M1 * (M1 + 2 * D) + M1 ** 3 / 3.0 + 2.0 * M1 * M1 * D
        return {"bytes": case["iters"] * data + 2 * model + 8.0 * (K * M1 + M1 * D),
                "flops": case["iters"] * (estep + mstep)}
    if case["kind"] == "map":
        return {"bytes": data + model + 8.0 * (K + N) * case["L"], "flops": estep + 2.0 * K * N * case["L"]}
    if case["kind"] == "ctemp":                        # two symmetric D x D moments for each centre
        return {"bytes": data + model + 16.0 * K, "flops": estep + 2.0 * K * N * D * (D + 1)}
    return {"bytes": data + model + 8.0 * K * N, "flops": estep}


# ---- the same in 64 bits, in plain torch -------------------------------------------

def _resp64(T, Y, beta, it):
    """Responsibilities (points x centres) and log g, log h of each point."""
    d = (Y * Y).sum(1)[None, :] - 2.0 * (T @ Y.T) + (T * T).sum(1)[:, None]
    x = d.mul_(-beta / 2.0)
    x = torch.where(x > UNDERFLOW, x, torch.full_like(x, -math.inf))
    logg, logh = torch.logsumexp(x, 1), torch.logsumexp(x * it, 1)
    return torch.exp(x.mul_(it).sub_(logh[:, None])), logg, logh


def _estep64(T, Y, beta, it):
    """(sum log g, sum log h, G, R T)."""
    G, RT = torch.zeros_like(Y[:, 0]), torch.zeros_like(Y)
    lg, lh = 0.0, 0.0
    step = max(256, (1 << 26) // len(Y))
    for i in range(0, len(T), step):
        P = T[i:i + step]
        R, logg, logh = _resp64(P, Y, beta, it)
        G += R.sum(0)
        RT += R.T @ P
        lg, lh = lg + float(logg.sum()), lh + float(logh.sum())
    return lg, lh, G, RT


def _mstep64(T, FI, G, RT, beta):
    A, B = (FI.T @ (FI * G[:, None])).cpu(), (FI.T @ RT).cpu()
    W = torch.linalg.solve(A + LAMBDA / beta * torch.eye(len(A), dtype=A.dtype), B).cuda()
    Y = FI @ W
    s = (T * T).sum() - 2.0 * (Y * RT).sum() + (G * (Y * Y).sum(1)).sum()
    return W, Y, T.numel() / float(s)


def _quality(T, Y, beta, total):
    return (T.shape[1] / 2.0) * math.log(beta / (2.0 * math.pi)) - math.log(len(Y)) + total / len(T)


def _iterate64(T, FI, Y, beta, isDA, temp, iters):
    llh, nfree, W = [], [], None
    for _ in range(iters):
        lg, lh, G, RT = _estep64(T, Y, beta, 1.0 / temp)
        llh.append(_quality(T, Y, beta, lg))
        nfree.append(_quality(T, Y, beta, temp * lh) if isDA else -llh[-1])
        W, Y, beta = _mstep64(T, FI, G, RT, beta)
    return llh, nfree, W, Y, beta


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for c, (T, X, FI, Y, beta) in _instances(case, seed):
            llh, nfree, W, Y, beta = _iterate64(T, FI, Y, beta, True, c["temp"], c["iters"])
            out.append({"status": None, "llh": llh[-1], "nfree": nfree[-1], "beta": beta, "W": W, "Y": Y})
        return out
    T, X, FI, Y, beta = _problem(case, seed)
    temp = case["temp"]
    if case["kind"] == "iterate":
        llh, nfree, W, Y, beta = _iterate64(T, FI, Y, beta, temp != 1.0, temp, case["iters"])
        return {"nfree": np.array(nfree), "llh": np.array(llh), "W": W, "Y": Y, "beta": beta}
    lg, lh, G, RT = _estep64(T, Y, beta, 1.0 / temp)
    out = {"llh": _quality(T, Y, beta, lg), "nfree": _quality(T, Y, beta, temp * lh), "nzero": None}
    if case["kind"] == "estep":
        return dict(out, G=G, RT=RT)
    step = max(256, (1 << 26) // len(Y))
    R = (_resp64(T[i:i + step], Y, beta, 1.0 / temp)[0] for i in range(0, len(T), step))
    if case["kind"] == "map":
        return dict(out, M=torch.cat([r @ X for r in R]))
    R = torch.cat(list(R)).T
    if case["kind"] == "resp":
        return dict(out, R=R.contiguous())
    # critical temperatures: the eigenvalues of [[2 S1 - S2, -S2], [-S2, 2 S1 - S2]]
    # are those of 2 S1 and of 2 S1 - 2 S2
    each = []
    for k in range(len(Y)):
        x, r, g = T - Y[k], R[k][:, None], float(G[k])
        S1, S2 = (x * r).T @ x, (x * r * r).T @ x
        w = torch.linalg.eigvalsh(torch.stack([2.0 * S1, 2.0 * (S1 - S2)]).cpu()).reshape(-1)
        w = torch.where(w >= (temp - 1e-6) * g * 2.0 / beta, torch.zeros_like(w), w)
        each.append(beta / 2.0 / g * float(w.max()))
    return dict(out, max=max(each), each=np.array(each))
