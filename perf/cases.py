"""What the framework's users run, as cases that can be timed and compared.

A case is a dict of plain values; its ``kind`` says which public entry points a
pass goes through:

* ``tick``       one MPC tick: an SQP iteration from the warm start
                 (``SQPSolver.iterate``) and the warm-start shift
                 (``SQPSolver.shift``), the tanh or LTV model family;
* ``srbd``       the same tick of the single-rigid-body quadruped controller
                 (``SRBDSolver.iterate``, ``shift_warmstart``);
* ``direction``  the direction half of an iteration on the caller's own
                 linearisation (``CallerSolver.direction``);
* ``solve``      the offline solve to the stop rule (``SQPSolver.solve``);
* ``certify``    model evaluation and KKT residual of an iterate
                 (``SQPSolver.model_eval``, ``SQPSolver.kkt``).

Inputs have the distributions of ``mpx_amd.synthetic`` and of the quadruped
controller's configuration, drawn on the device from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

H, KAPPA = 0.02, 0.1
RHO0, RHO_MAX, RHO_C, MU_B, TAU, BETA, C1, SLACK, TRIALS = 1.0, 1e8, 10.0, 1e-2, 0.995, 0.5, 1e-4, 1e-6, 10

# the quadruped controller's constants: body, stance feet, residual weights
MASS, DT = 24.637, 0.02
INERTIA = ((0.2310941359705289, -0.0014987128245817424, -0.021400468992761768),
           (-0.0014987128245817424, 1.4485084687476608, 0.0004641447134275615),
           (-0.021400468992761768, 0.0004641447134275615, 1.503217877350808))
P0 = (0.0, 0.0, 0.33)
LEGS0 = (0.27092872, 0.193, 0.0, 0.27092872, -0.193, 0.0, -0.20887128, 0.193, 0.0, -0.20887128, -0.193, 0.0)
W_SRBD = (0, 0, 1e4, 1e3, 1e3, 0, 1e3, 1e3, 1e3, 1e1, 1e1, 1e1) + (1e-2,) * 12


def listed():
    return [
        # a single small controller: every launch and every dependent stage counts
        dict(name="tick_12x12x25", kind="tick", model="tanh", n=12, m=12, N=25, p=0, box=True, B=1, dtype="f32",
             start="warm", group=0),
        # a single whole-body-sized controller with contact rows, the plain one-robot call
        dict(name="tick_36x12x50", kind="tick", model="tanh", n=36, m=12, N=50, p=8, box=False, B=1, dtype="f32",
             start="warm", group=0),
        # the serving stream's large class: a few humanoids with a long horizon in one launch group
        dict(name="serve_76x32x100", kind="tick", model="tanh", n=76, m=32, N=100, p=0, box=True, B=8, dtype="f32",
             start="warm", group=0),
        # the headline workload: a fleet of whole-body-sized instances with equality rows
        dict(name="fleet_36x12x50", kind="tick", model="tanh", n=36, m=12, N=50, p=8, box=False, B=4096,
             dtype="f32", start="warm", group=1),
        # a fleet of smaller bodies with bounded controls and a long horizon
        dict(name="fleet_24x12x100", kind="tick", model="tanh", n=24, m=12, N=100, p=0, box=True, B=1024,
             dtype="f32", start="warm", group=1),
        # humanoids in parallel environments, rows and bounds together
        dict(name="humanoid_76x32x50", kind="tick", model="tanh", n=76, m=32, N=50, p=12, box=True, B=256,
             dtype="f32", start="warm", group=0),
        # caller-supplied time-varying Jacobians and weights, ragged sizes
        dict(name="ltv_19x7x33", kind="tick", model="ltv", n=19, m=7, N=33, p=3, box=True, B=333, dtype="f32",
             start="warm", group=0),
        # double precision: the reference results of the same fleet
        dict(name="f64_36x12x50", kind="tick", model="tanh", n=36, m=12, N=50, p=8, box=False, B=64, dtype="f64",
             start="warm", group=0),
        # the quadruped controller's parallel environments (64, horizon 25)
        dict(name="srbd_25", kind="srbd", N=25, B=64, dtype="f32"),
        # whole-body quadruped with the caller's own dynamics and cost (n = 61, m = 12, horizon 25)
        dict(name="direction_61x12x25", kind="direction", n=61, m=12, N=25, p=0, cross=True, B=64, dtype="f32"),
        # the offline solve of one problem to its stop rule
        dict(name="solve_24x12x50", kind="solve", model="tanh", n=24, m=12, N=50, p=0, box=False, B=1, dtype="f64",
             start="rollout", max_iter=10),
        # costs, defects and KKT residuals of a fleet's iterates
        dict(name="certify_36x12x50", kind="certify", model="tanh", n=36, m=12, N=50, p=8, box=False, B=1024,
             dtype="f32", start="rollout", group=0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _work_units(c):
    """Dense Riccati work of one pass, up to a constant (bounds what is drawn)."""
    n, m = c["n"], c["m"]
    return c["B"] * c["N"] * (4 * n ** 3 + 6 * n * n * m + 4 * n * m * m) * (8 if c["dtype"] == "f64" else 1)


def draw(rng):
    """A further case of the same ranges: sizes over the whole range, odd ones too."""
    kind = rng.choice(["tick", "tick", "fleet", "large", "ltv", "f64", "srbd", "direction", "solve", "certify"])
    if kind == "srbd":
        return dict(kind="srbd", N=rng.randint(10, 50), B=_log_int(rng, 1, 512), dtype="f32")
    while True:
        if kind == "tick":
            c = dict(kind="tick", model="tanh", n=_log_int(rng, 6, 47), m=rng.randint(3, 14), N=rng.randint(10, 100),
                     B=_log_int(rng, 1, 64), dtype="f32", start="warm", group=0)
        elif kind == "fleet":
            c = dict(kind="tick", model="tanh", n=rng.randint(8, 47), m=rng.randint(4, 14), N=rng.randint(20, 100),
                     B=_log_int(rng, 256, 4096), dtype="f32", start="warm", group=1)
        elif kind == "large":
            c = dict(kind="tick", model="tanh", n=rng.randint(48, 78), m=rng.randint(12, 32), N=rng.randint(20, 100),
                     B=_log_int(rng, 1, 256), dtype="f32", start="warm", group=0)
        elif kind == "ltv":
            c = dict(kind="tick", model="ltv", n=rng.randint(6, 40), m=rng.randint(3, 12), N=rng.randint(10, 60),
                     B=_log_int(rng, 1, 1024), dtype="f32", start="warm", group=0)
        elif kind == "f64":
            c = dict(kind="tick", model=rng.choice(["tanh", "ltv"]), n=rng.randint(6, 40), m=rng.randint(3, 12),
                     N=rng.randint(10, 60), B=_log_int(rng, 1, 128), dtype="f64", start=rng.choice(["warm", "rollout", "tile"]),
                     group=0)
        elif kind == "direction":
            c = dict(kind="direction", n=_log_int(rng, 6, 75), m=rng.randint(3, 19), N=rng.randint(10, 50),
                     cross=rng.random() < 0.7, B=_log_int(rng, 1, 256), dtype="f32")
        elif kind == "solve":
            c = dict(kind="solve", model="tanh", n=rng.randint(6, 36), m=rng.randint(3, 12), N=rng.randint(10, 60),
                     p=0, box=False, B=_log_int(rng, 1, 16), dtype="f64", start="rollout", max_iter=10)
        else:
            c = dict(kind="certify", model="tanh", n=rng.randint(8, 60), m=rng.randint(4, 24), N=rng.randint(10, 80),
                     B=_log_int(rng, 1, 1024), dtype="f32", start="rollout", group=0)
        c.setdefault("p", rng.choice([0, rng.randint(1, max(1, min(12, c["m"] - 2)))]))
        if kind != "direction":
            # the largest bodies always with bounded controls, as humanoids have
            c.setdefault("box", kind == "large" or rng.random() < 0.5)
        if _work_units(c) <= 4096 * 50 * (4 * 36 ** 3 + 6 * 36 * 36 * 12 + 4 * 36 * 144):
            return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


class _Draw:
    """Seeded random device tensors in the case's type."""

    def __init__(self, case, seed, tag):
        self.dtype = _dtype(case)
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(1000003 * int(seed) + tag)

    def normal(self, *shape, scale=1.0):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=self.dtype) * scale

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=self.gen, device="cuda", dtype=self.dtype)


def _arrays(case, seed):
    """Problem data of the device model families: mpx_amd.synthetic's
    distributions, with control weights of the state weights' size."""
    n, m, N, p, B = case["n"], case["m"], case["N"], case["p"], case["B"]
    r = _Draw(case, seed, 11)
    eye = torch.eye(n, device="cuda", dtype=r.dtype)
    a = {}
    if case["model"] == "ltv":
        a["A"] = eye + r.normal(B, N, n, n, scale=H / math.sqrt(n))
        a["B"] = r.normal(B, N, n, m, scale=H)
        a["Q"] = torch.diag_embed(r.uniform(1, 10, B, N, n))
        a["R"] = torch.diag_embed(r.uniform(1, 10, B, N, m))
        a["QN"] = torch.diag_embed(10 * r.uniform(1, 10, B, n))
    else:
        a["A"] = r.normal(B, n, n, scale=1 / math.sqrt(n))
        a["B"] = r.normal(B, n, m)
        a["W"] = r.normal(B, n, n, scale=1 / math.sqrt(n))
        Q = torch.diag_embed(r.uniform(1, 10, B, n))
        a["Q"] = Q[:, None].contiguous()
        a["R"] = torch.diag_embed(r.uniform(1, 10, B, m))[:, None].contiguous()
        a["QN"] = 10 * Q
    a["xref"] = torch.zeros(B, N + 1, n, device="cuda", dtype=r.dtype)
    a["uref"] = torch.zeros(B, N, m, device="cuda", dtype=r.dtype)
    if p > 0:
        a["D"] = r.normal(B, N, p, n, scale=1 / math.sqrt(n))
        a["E"] = r.normal(B, N, p, m)
        a["e"] = torch.zeros(B, N, p, device="cuda", dtype=r.dtype)
    else:
        a["D"] = a["E"] = a["e"] = None
    a["ulo"] = -torch.ones(B, m, device="cuda", dtype=r.dtype) if case["box"] else None
    a["uhi"] = torch.ones(B, m, device="cuda", dtype=r.dtype) if case["box"] else None
    a["x0"] = r.normal(B, n)
    return a


def _mv(M, x):
    return torch.matmul(M, x.unsqueeze(-1)).squeeze(-1)


def _f(case, a, x, u, t):
    """The dynamics at stage t (a slice: all stages at once)."""
    if case["model"] == "ltv":
        return _mv(a["A"][:, t], x) + _mv(a["B"][:, t], u)
    if x.dim() == 2:
        return x + H * (_mv(a["A"], x) + _mv(a["B"], u) + KAPPA * torch.tanh(_mv(a["W"], x)))
    mm = lambda M, z: torch.matmul(z, M.mT.contiguous())
    return x + H * (mm(a["A"], x) + mm(a["B"], u) + KAPPA * torch.tanh(mm(a["W"], x)))


def _start(case, seed, a):
    """The iterate a pass starts from (X, U, V, Yeq, Ybox): ``warm``, a running
    controller's plan (bounded controls, their rollout, multipliers of that
    size), or ``rollout`` / ``tile``, the controllers' reset states."""
    n, m, N, p, B = case["n"], case["m"], case["N"], case["p"], case["B"]
    z = lambda *s: torch.zeros(s, device="cuda", dtype=a["x0"].dtype)
    warm = case["start"] == "warm"
    r = _Draw(case, seed, 53)
    U = r.uniform(-0.6, 0.6, B, N, m) if warm else z(B, N, m)
    if case["start"] != "tile":
        X = [a["x0"]]
        for t in range(N):
            X.append(_f(case, a, X[-1], U[:, t], t))
        X = torch.stack(X, 1)
    else:
        X = a["x0"][:, None].repeat(1, N + 1, 1)
    if warm:
        return X, U, 20 * X, r.normal(B, N, p, scale=0.3), r.uniform(0.01, 0.05, B, N, 2 * m)
    return X, U, z(B, N + 1, n), z(B, N, p), z(B, N, 2 * m)


def _certify_point(case, seed, a):
    """An iterate away from the start: perturbed states, controls and multipliers."""
    n, m, N, p, B = case["n"], case["m"], case["N"], case["p"], case["B"]
    r = _Draw(case, seed, 23)
    X = _start(case, seed, a)[0]
    return (X + r.normal(B, N + 1, n, scale=0.1), r.uniform(-0.9, 0.9, B, N, m), r.normal(B, N + 1, n),
            r.normal(B, N, p, scale=0.1), r.uniform(0.01, 0.5, B, N, 2 * m))


def _lin_arrays(case, seed):
    """A caller's linearisation: Jacobians near the identity, a definite stage Hessian with a cross term."""
    n, m, N, p, B = case["n"], case["m"], case["N"], case["p"], case["B"]
    r = _Draw(case, seed, 37)
    eye = torch.eye(n, device="cuda", dtype=r.dtype)
    a = dict(A=eye + r.normal(B, N, n, n, scale=H / math.sqrt(n)), B=r.normal(B, N, n, m, scale=H),
             Q=torch.diag_embed(r.uniform(1, 10, B, N, n)), R=torch.diag_embed(r.uniform(0.5, 1, B, N, m)),
             QN=torch.diag_embed(r.uniform(10, 100, B, n)), fbar=r.normal(B, N, n, scale=0.5),
             q=r.normal(B, N + 1, n), r=r.normal(B, N, m, scale=0.1), g=r.uniform(0, 1, B, N + 1, 1))
    a["M"] = r.normal(B, N, n, m, scale=0.3 / math.sqrt(n * m)) if case["cross"] else None
    a["D"] = r.normal(B, N, p, n, scale=1 / math.sqrt(n)) if p else None
    a["E"] = r.normal(B, N, p, m) if p else None
    a["e"] = torch.zeros(B, N, p, device="cuda", dtype=r.dtype) if p else None
    a["x0"] = r.normal(B, n)
    it = (r.normal(B, N + 1, n, scale=0.5), r.normal(B, N, m, scale=0.1), r.normal(B, N + 1, n, scale=0.5))
    return a, it


def _srbd_arrays(case, seed):
    """Trotting quadrupeds at perturbed states: (x0, reference, parameter), float64 host arrays."""
    N, B = case["N"], case["B"]
    rng = np.random.default_rng([91, int(seed)])
    v = np.stack([0.3 + 0.2 * rng.uniform(size=B), 0.1 * rng.standard_normal(B), np.zeros(B)], 1)
    t = np.arange(N + 1)
    k = t[None] + rng.integers(0, 10, size=B)[:, None]
    ref = np.zeros((B, N + 1, 17))
    ref[..., 0:3] = np.array(P0) + v[:, None] * (t * DT)[None, :, None]
    ref[..., 3] = 1.0
    ref[..., 7:10] = v[:, None]
    trot = (k // 5) % 2
    contact = np.where(trot[..., None] == 0, np.array([1.0, 0, 0, 1]), np.array([0, 1.0, 1, 0]))
    contact[k % 5 == 0] = 1.0
    ref[..., 13:17] = contact
    par = np.zeros((B, N + 1, 16))
    par[..., 0:4] = contact
    par[..., 4:] = np.array(LEGS0) + np.tile(ref[..., 0:3] * np.array([1, 1, 0]), 4)
    x0 = np.zeros((B, 13))
    x0[:, 0:3] = np.array(P0) + 0.01 * rng.standard_normal((B, 3))
    q = np.concatenate([np.ones((B, 1)), 0.02 * rng.standard_normal((B, 3))], 1)
    x0[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    x0[:, 7:13] = 0.05 * rng.standard_normal((B, 6))
    return x0, ref, par


def prepare(case, seed):
    from mpx_amd.caller import CallerBatch, CallerSolver
    from mpx_amd.problem import DeviceBatch, SQPSolver
    from mpx_amd.srbd import SRBDSolver
    kind = case["kind"]
    if kind == "srbd":
        x0, ref, par = _srbd_arrays(case, seed)
        B, N = case["B"], case["N"]
        solver = SRBDSolver(MASS, np.array(INERTIA), DT, np.diag(np.array(W_SRBD, float)), ref, par, x0,
                            dtype=_dtype(case))
        it = solver.iterate_from(np.repeat(x0[:, None], N + 1, 1), np.zeros((B, N, 12)), np.zeros((B, N + 1, 13)))
        return dict(kind=kind, solver=solver, it=it, reset=torch.zeros(B, dtype=torch.int32, device="cuda"))
    if kind == "direction":
        a, (X, U, V) = _lin_arrays(case, seed)
        host = lambda k: None if a[k] is None else a[k].cpu().numpy()
        batch = CallerBatch(case["B"], case["n"], case["m"], case["N"], host("x0"), D=host("D"), E=host("E"),
                            e=host("e"), cross=case["cross"], dtype=_dtype(case))
        batch.set_linearization(**{k: a[k] for k in ("A", "B", "fbar", "Q", "R", "M", "q", "r", "g", "QN")})
        it = batch.iterate_from(X.cpu().numpy(), U.cpu().numpy(), V.cpu().numpy())
        return dict(kind=kind, solver=CallerSolver(batch), it=it)
    a = _arrays(case, seed)
    dims = dict(n=case["n"], m=case["m"], N=case["N"], p=case["p"], model=case["model"], h=H, kappa=KAPPA)
    batch = DeviceBatch(dims, a, dtype=_dtype(case))
    solver = SQPSolver(batch, trial_group=case.get("group", 0))
    point = _certify_point(case, seed, a) if kind == "certify" else _start(case, seed, a)
    it = batch.iterate_from(*point)
    s = dict(kind=kind, solver=solver, it=it, p=case["p"], box=case["box"],
             reset=torch.zeros(case["B"], dtype=torch.int32, device="cuda"))
    if kind == "solve":
        s["start"], s["max_iter"] = point, case["max_iter"]
    return s


def run(s):
    kind, solver, it = s["kind"], s["solver"], s["it"]
    if kind == "certify":
        g, c = solver.model_eval(it["X"], it["U"])
        return dict(g=g, c=c, kkt=solver.kkt(it))
    if kind == "direction":
        dX, dU, a_max = solver.direction(it)
        return dict(dX=dX, dU=dU, a_max=a_max)
    if kind == "srbd":
        from mpx_amd.problem import shift_warmstart
        st = solver.iterate(it)
        shift_warmstart(solver.batch, it, 1, reset=s["reset"])
        return dict(X=it["X"], U=it["U"], V=it["V"], status=st["status"])
    if kind == "solve":
        # the controller's reset state, then the whole loop
        for k, v in zip(("X", "U", "V"), s["start"]):
            it[k].copy_(v)
        iters, cost, cc, _ = solver.solve(it, max_iter=s["max_iter"])
        return dict(X=it["X"], U=it["U"], V=it["V"], iters=iters, cost=cost)
    st = solver.iterate(it)
    solver.shift(it, 1, reset=s["reset"])
    out = dict(X=it["X"], U=it["U"], V=it["V"], status=st["status"])
    if s["p"]:
        out["Yeq"] = it["Yeq"]
    if s["box"]:
        out["Ybox"] = it["Ybox"]
    return out


def work(case):
    """Inputs read once, outputs written once; the arithmetic of a sequential
    Riccati iteration with one line-search trial, products with symmetric
    results at half."""
    es = 8 if case["dtype"] == "f64" else 4
    kind, N, B = case["kind"], case["N"], case["B"]
    n, m, p = (13, 12, 0) if kind == "srbd" else (case["n"], case["m"], case["p"])
    N1 = N + 1
    iterate = N1 * 2 * n + N * m
    ric = 2 * n * n * (n + m) + n * n * n + 2 * n * n * m + n * m * m + m ** 3 / 3 + 2 * m * m * n + n * n * m \
        + p * (n + m) ** 2
    model = 4 * n * n + 2 * n * m + 2 * p * (n + m)
    sweep = N * (2 * (2 * n * n + 2 * n * m) + 2 * (2 * n * n + 2 * p * (n + m)))
    rows = N * p * (n + m + 1)
    if kind == "srbd":
        data = 24 * 24 + N1 * 33 + n
        return dict(bytes=es * B * (data + 2 * iterate), flops=B * (N * ric + sweep + N1 * 2000))
    if kind == "direction":
        data = N * (n * n + n * m + n + n * n + m * m + (n * m if case["cross"] else 0) + n + m + 1) + n * n + rows + n
        return dict(bytes=es * B * (data + iterate + N1 * n + N * m), flops=B * (N * ric + sweep))
    if case["model"] == "ltv":
        data = N * (n * n + n * m + n * n + m * m)
    else:
        data = 2 * n * n + n * m + n * n + m * m
    data += n * n + iterate - N1 * n + rows + n + (2 * m if case["box"] else 0)
    duals = N * (p + (2 * m if case["box"] else 0))
    if kind == "certify":
        return dict(bytes=es * B * (data + iterate + duals + N1 * (n + 1) + 1), flops=B * N * 2 * model)
    its = 3 if kind == "solve" else 1
    return dict(bytes=es * B * (data + 2 * (iterate + duals)), flops=its * B * (N * (ric + 2 * model) + sweep))


# ---------------------------------------------------------------------------
# the same results in 64 bits, from the formulas
# ---------------------------------------------------------------------------

def _lqr(L):
    """Riccati recursion and rollout: dX, dU and the costates."""
    N = L["A"].shape[1]
    S, s = L["QN"], L["qN"]
    Ss, ss, Ks, ks = [S], [s], [], []
    for t in range(N - 1, -1, -1):
        A, Bm = L["A"][:, t], L["B"][:, t]
        At, Bt = A.mT.contiguous(), Bm.mT.contiguous()
        Sc = _mv(S, L["c"][:, t]) + s
        SA = S @ A
        G = L["M"][:, t].mT.contiguous() + Bt @ SA
        gu = L["r"][:, t] + _mv(Bt, Sc)
        Lc = torch.linalg.cholesky(L["R"][:, t] + Bt @ (S @ Bm))
        Kk = torch.cholesky_solve(torch.cat([G, gu.unsqueeze(-1)], -1), Lc)
        K, k = Kk[..., :-1].contiguous(), Kk[..., -1].contiguous()
        Gt = G.mT.contiguous()
        S = L["Q"][:, t] + At @ SA - Gt @ K
        S = 0.5 * (S + S.mT)
        s = L["q"][:, t] + _mv(At, Sc) - _mv(Gt, k)
        Ss.append(S), ss.append(s), Ks.append(K), ks.append(k)
    Ss, ss, Ks, ks = Ss[::-1], ss[::-1], Ks[::-1], ks[::-1]
    dX, dU = [L["c0"]], []
    for t in range(N):
        dU.append(-_mv(Ks[t], dX[t]) - ks[t])
        dX.append(_mv(L["A"][:, t], dX[t]) + _mv(L["B"][:, t], dU[t]) + L["c"][:, t])
    lam = torch.stack([_mv(Ss[t], dX[t]) + ss[t] for t in range(N + 1)], 1)
    return torch.stack(dX, 1), torch.stack(dU, 1), lam


def _ftb(v, dv):
    r = torch.where(dv < 0, -TAU * v / dv, torch.inf).flatten(1).amin(1)
    return torch.clamp(r, max=1.0)


def _step(L, X, U, V, phi, a_max=None):
    """The step, the penalty and the accepted step size: ``phi(X, U, V, rho)``
    is the merit; L holds the linearisation, its c the defects."""
    dX, dU, lam = _lqr(L)
    dV = lam - V
    c = torch.cat([L["c0"][:, None], L["c"]], 1)
    N = dU.shape[1]
    d_f = (L["q"] * dX[:, :N]).sum((1, 2)) + (L["r"] * dU).sum((1, 2)) + (L["qN"] * dX[:, N]).sum(1)
    d_c = ((dV - V) * c).sum((1, 2))
    cc = (c * c).sum((1, 2))
    quad = lambda x, M, y: (x * _mv(M, y)).flatten(1).sum(1)
    kap = quad(dX[:, N], L["QN"], dX[:, N]) + quad(dX[:, :N], L["Q"], dX[:, :N]) + quad(dU, L["R"], dU) \
        + 2 * quad(dX[:, :N], L["M"], dU)
    num = d_f + d_c + 0.5 * kap
    rho = torch.where(cc > 0, torch.clamp(2 * num / cc, min=RHO0), torch.full_like(cc, RHO0)).clamp(max=RHO_MAX)
    dphi = d_f + d_c - rho * cc
    top = torch.ones_like(cc) if a_max is None else a_max(dU)
    phi0 = phi(X, U, V, rho)
    limit = phi0 + SLACK * (1 + phi0.abs())
    alpha = top * BETA ** (TRIALS - 1)
    found = torch.zeros_like(cc, dtype=torch.bool)
    for j in range(TRIALS):
        a = top * BETA ** j
        e = a[:, None, None]
        ok = (phi(X + e * dX, U + e * dU, V + e * dV, rho) <= limit + C1 * a * dphi) & ~found
        alpha = torch.where(ok, a, alpha)
        found |= ok
        if bool(found.all()):
            break
    status = torch.where(found, 0, 2).to(torch.int32)
    return dX, dU, dV, alpha, status


def _quad_cost(case, a, X, U):
    N = case["N"]
    dx, du = X - a["xref"], U - a["uref"]
    g = 0.5 * (dx[:, :N] * _mv(a["Q"], dx[:, :N])).sum(-1) + 0.5 * (du * _mv(a["R"], du)).sum(-1)
    return torch.cat([g, 0.5 * (dx[:, N] * _mv(a["QN"], dx[:, N])).sum(-1)[:, None]], 1)


def _defects(case, a, X, U):
    return torch.cat([(a["x0"] - X[:, 0])[:, None], _f(case, a, X[:, :-1], U, slice(None)) - X[:, 1:]], 1)


def _jacobians(case, a, X):
    if case["model"] == "ltv":
        return a["A"], a["B"]
    B, N, n = case["B"], case["N"], case["n"]
    th = torch.tanh(torch.matmul(X[:, :N], a["W"].mT.contiguous()))
    A = torch.eye(n, device="cuda", dtype=X.dtype) \
        + H * (a["A"][:, None] + KAPPA * (1 - th * th).unsqueeze(-1) * a["W"][:, None])
    return A, (H * a["B"])[:, None].expand(B, N, n, case["m"])


def _sqp(case, a, X, U, V, Yeq, Ybox):
    """One iteration of the device model families; returns the new iterate and the line search's status."""
    N, n, m, p, B = case["N"], case["n"], case["m"], case["p"], case["B"]
    box = case["box"]
    if box:
        lo, hi = a["ulo"][:, None], a["uhi"][:, None]
        w = 1e-3 * (hi - lo)
        U = torch.where(U >= hi, hi - w, U)
        U = torch.where(U <= lo, lo + w, U)
        slack = torch.cat([hi - U, U - lo], -1)
        Ybox = torch.where(Ybox > 0, Ybox, MU_B / slack)
    A, Bm = _jacobians(case, a, X)
    c = _defects(case, a, X, U)
    Q = a["Q"].expand(B, N, n, n).clone()
    R = a["R"].expand(B, N, m, m).clone()
    M = torch.zeros(B, N, n, m, device="cuda", dtype=X.dtype)
    q = _mv(a["Q"], X[:, :N] - a["xref"][:, :N])
    r = _mv(a["R"], U - a["uref"])
    rows = None
    if p:
        Dt, Et = a["D"].mT.contiguous(), a["E"].mT.contiguous()
        rows = lambda X_, U_: _mv(a["D"], X_[:, :N]) + _mv(a["E"], U_) + a["e"]
        w_ = Yeq + RHO_C * rows(X, U)
        Q += RHO_C * Dt @ a["D"]
        R += RHO_C * Et @ a["E"]
        M += RHO_C * Dt @ a["E"]
        q = q + _mv(Dt, w_)
        r = r + _mv(Et, w_)
    a_max = None
    if box:
        r = r + MU_B / slack[..., :m] - MU_B / slack[..., m:]
        R = R + torch.diag_embed(Ybox[..., :m] / slack[..., :m] + Ybox[..., m:] / slack[..., m:])
        a_max = lambda dU: _ftb(slack, torch.cat([-dU, dU], -1))
    L = dict(A=A, B=Bm, Q=Q, R=R, M=M, q=q, r=r, c=c[:, 1:], c0=c[:, 0], QN=a["QN"],
             qN=_mv(a["QN"], X[:, N] - a["xref"][:, N]))

    def phi(X_, U_, V_, rho):
        d = _defects(case, a, X_, U_)
        v = _quad_cost(case, a, X_, U_).sum(1) + (V_ * d).sum((1, 2)) + 0.5 * rho * (d * d).sum((1, 2))
        if p:
            h = rows(X_, U_)
            v = v + (Yeq * h).sum((1, 2)) + 0.5 * RHO_C * (h * h).sum((1, 2))
        if box:
            v = v - MU_B * (torch.log(hi - U_) + torch.log(U_ - lo)).sum((1, 2))
        return v

    dX, dU, dV, alpha, status = _step(L, X, U, V, phi, a_max)
    e = alpha[:, None, None]
    Xn, Un, Vn = X + e * dX, U + e * dU, V + e * dV
    if p:
        Yeq = Yeq + RHO_C * rows(Xn, Un)
    if box:
        dY = MU_B / slack - Ybox - Ybox * torch.cat([-dU, dU], -1) / slack
        Ybox = Ybox + _ftb(Ybox, dY)[:, None, None] * dY
    return Xn, Un, Vn, Yeq, Ybox, status


def _shifted(z):
    return torch.cat([z[:, 1:], z[:, -1:]], 1)


def _exact_tick(case, a, start):
    X, U, V, Yeq, Ybox, status = _sqp(case, a, *start)
    out = dict(X=_shifted(X), U=_shifted(U), V=_shifted(V), status=status)
    if case["p"]:
        out["Yeq"] = _shifted(Yeq)
    if case["box"]:
        out["Ybox"] = _shifted(Ybox)
    return out


def _exact_solve(case, a, start):
    B = case["B"]
    cur = list(start)
    run_ = torch.ones(B, dtype=torch.bool, device="cuda")
    iters = torch.zeros(B, dtype=torch.int32, device="cuda")
    last, cost = torch.full((B,), 1e10, device="cuda", dtype=torch.float64), torch.zeros(B, device="cuda",
                                                                                         dtype=torch.float64)
    for i in range(1, case["max_iter"] + 2):
        new = _sqp(case, a, *cur)[:5]
        cur = [torch.where(run_[:, None, None], x, y) for x, y in zip(new, cur)]
        l2 = _quad_cost(case, a, cur[0], cur[1]).square().sum(1)
        cc = _defects(case, a, cur[0], cur[1]).square().sum((1, 2))
        iters = torch.where(run_, i, iters).to(torch.int32)
        cost = torch.where(run_, l2, cost)
        run_ = run_ & ~((last - l2 < 1e-3) & (cc < 1e-5))
        last = l2
        if not bool(run_.any()):
            break
    return dict(X=cur[0], U=cur[1], V=cur[2], iters=iters, cost=cost)


def _exact_certify(case, a, point):
    X, U, V, Yeq, Ybox = point
    N, m = case["N"], case["m"]
    c = _defects(case, a, X, U)
    A, Bm = _jacobians(case, a, X)
    gx = _mv(a["Q"], X[:, :N] - a["xref"][:, :N]) + _mv(A.mT, V[:, 1:]) - V[:, :N]
    gu = _mv(a["R"], U - a["uref"]) + _mv(Bm.mT, V[:, 1:])
    parts = [c, _mv(a["QN"], X[:, N] - a["xref"][:, N]) - V[:, N]]
    if case["p"]:
        gx = gx + _mv(a["D"].mT, Yeq)
        gu = gu + _mv(a["E"].mT, Yeq)
        parts.append(_mv(a["D"], X[:, :N]) + _mv(a["E"], U) + a["e"])
    if case["box"]:
        gu = gu + Ybox[..., :m] - Ybox[..., m:]
        s = torch.cat([a["uhi"][:, None] - U, U - a["ulo"][:, None]], -1)
        parts.append(Ybox * s - MU_B)
    sq = sum(z.square().flatten(1).sum(1) for z in parts + [gx, gu])
    return dict(g=_quad_cost(case, a, X, U), c=c, kkt=torch.sqrt(sq))


def _exact_direction(case, a, it):
    X, U, V = it
    N, p = case["N"], case["p"]
    B, n, m = case["B"], case["n"], case["m"]
    M = torch.zeros(B, N, n, m, device="cuda", dtype=X.dtype) if a["M"] is None else a["M"]
    Q, R, q, r = a["Q"], a["R"], a["q"][:, :N], a["r"]
    if p:
        Dt, Et = a["D"].mT.contiguous(), a["E"].mT.contiguous()
        w = RHO_C * (_mv(a["D"], X[:, :N]) + _mv(a["E"], U) + a["e"])
        Q, R, M = Q + RHO_C * Dt @ a["D"], R + RHO_C * Et @ a["E"], M + RHO_C * Dt @ a["E"]
        q, r = q + _mv(Dt, w), r + _mv(Et, w)
    dX, dU, _ = _lqr(dict(A=a["A"], B=a["B"], Q=Q, R=R, M=M, q=q, r=r, c=a["fbar"] - X[:, 1:],
                          c0=a["x0"] - X[:, 0], QN=a["QN"], qN=a["q"][:, N]))
    return dict(dX=dX, dU=dU, a_max=torch.ones(B, device="cuda", dtype=X.dtype))


# the single-rigid-body model of one stage (x 13, u 12, reference row 17, parameter row 16)

def _qmul(u, v):
    return torch.stack([u[0] * v[0] - u[1] * v[1] - u[2] * v[2] - u[3] * v[3],
                        u[0] * v[1] + u[1] * v[0] + u[2] * v[3] - u[3] * v[2],
                        u[0] * v[2] - u[1] * v[3] + u[2] * v[0] + u[3] * v[1],
                        u[0] * v[3] + u[1] * v[2] - u[2] * v[1] + u[3] * v[0]])


def _rot(q):
    w, x, y, z = q[0], q[1], q[2], q[3]
    return torch.stack([
        torch.stack([w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y)]),
        torch.stack([2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x)]),
        torch.stack([2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z])])


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _srbd_f(x, u, par, consts):
    inertia, inv, grav = consts
    contact, legs = par[:4], par[4:]
    f = [u[3 * i:3 * i + 3] for i in range(4)]
    force = sum(f[i] * contact[i] for i in range(4))
    wrench = sum(_cross(legs[3 * i:3 * i + 3] - x[:3], f[i]) * contact[i] for i in range(4))
    dp = x[7:10] + (grav + force / MASS) * DT
    om = x[10:13]
    om = om + (inv * (((_rot(x[3:7]).mT * wrench).sum(-1)) - _cross(om, (inertia * om).sum(-1)))).sum(-1) * DT
    ang = torch.sqrt((om * om).sum())
    qr = torch.cat([torch.cos(0.5 * DT * ang)[None], om * (torch.sin(0.5 * DT * ang) / ang)])
    qn = _qmul(x[3:7], qr)
    return torch.cat([x[:3] + dp * DT, qn / torch.sqrt((qn * qn).sum()), dp, om])


def _srbd_res(x, ref):
    q = _qmul(ref[3:7] * torch.tensor([1.0, -1, -1, -1], device=x.device, dtype=x.dtype), x[3:7])
    s = torch.sqrt((q[1:] * q[1:]).sum())
    ang = 2 * torch.atan2(s, q[0])
    ang = torch.where(ang > math.pi, ang - 2 * math.pi, ang)
    return torch.cat([x[:3] - ref[:3], q[1:] * (ang / s), x[7:10] - ref[7:10], x[10:13] - ref[10:13]])


def _cone(u):
    u = u.reshape(4, 3)
    return 0.7 * u[:, 2] - torch.sqrt(u[:, 0] ** 2 + u[:, 1] ** 2 + 1e-2)


def _penalty(v, alpha=0.1, sigma=5.0):
    logb = -alpha * torch.log(torch.clamp(v, 1e-10, 1e6))
    quad = alpha / 2 * (((v - 2 * sigma) / sigma) ** 2 - 1)
    return torch.clamp(torch.where(v > sigma, logb, quad + logb), 0.0, 1e8)


def _exact_srbd(case, seed):
    from torch.func import grad, jacrev, vmap
    to = lambda v: torch.as_tensor(v, device="cuda", dtype=_dtype(case)).double()
    x0, ref, par = (to(v) for v in _srbd_arrays(case, seed))
    B, N = case["B"], case["N"]
    inertia = torch.tensor(INERTIA, device="cuda", dtype=torch.float64)
    consts = (inertia, torch.linalg.inv(inertia), torch.tensor([0, 0, -9.81], device="cuda", dtype=torch.float64))
    w = torch.tensor(W_SRBD, device="cuda", dtype=torch.float64)
    Wx, Wu = w[:12], w[12:]
    f = lambda x, u, p_: _srbd_f(x, u, p_, consts)
    cost_x = lambda x, r_: 0.5 * (Wx * _srbd_res(x, r_) ** 2).sum()
    cost_u = lambda u: 0.5 * (Wu * u * u).sum() + 0.5 * torch.clamp(_penalty(_cone(u)), 1e-6, 1e6).sum()
    flat = lambda z: z.reshape((-1,) + z.shape[2:])
    back = lambda z, k: z.reshape((B, k) + z.shape[1:])
    X, U = x0[:, None].repeat(1, N + 1, 1), torch.zeros(B, N, 12, device="cuda", dtype=torch.float64)
    V = torch.zeros(B, N + 1, 13, device="cuda", dtype=torch.float64)
    xs, us, ps, rs = flat(X[:, :N]), flat(U), flat(par[:, :N]), flat(ref[:, :N])
    fx, fu = vmap(jacrev(f, argnums=(0, 1)))(xs, us, ps)
    Jx = vmap(jacrev(_srbd_res))(flat(X), flat(ref))
    JtW = Jx.mT.contiguous() * Wx
    Q = back(JtW @ Jx, N + 1)
    d2 = vmap(vmap(grad(grad(lambda v: _penalty(v)))))(vmap(_cone)(us))
    Ju = vmap(jacrev(_cone))(us)
    h = torch.clamp(d2, 1e-6, 1e6) * rs[:, 13:17]
    R = torch.diag(Wu) + (Ju.mT * h.unsqueeze(1)) @ Ju
    q = back(vmap(grad(cost_x))(flat(X), flat(ref)), N + 1)
    r = back(vmap(grad(cost_u))(us), N)

    def defects(X_, U_):
        nx = back(vmap(f)(flat(X_[:, :N]), flat(U_), ps), N)
        return torch.cat([(x0 - X_[:, 0])[:, None], nx - X_[:, 1:]], 1)

    def phi(X_, U_, V_, rho):
        d = defects(X_, U_)
        g = back(vmap(cost_x)(flat(X_), flat(ref)), N + 1).sum(1) + back(vmap(cost_u)(flat(U_)), N).sum(1)
        return g + (V_ * d).sum((1, 2)) + 0.5 * rho * (d * d).sum((1, 2))

    c = defects(X, U)
    L = dict(A=back(fx, N), B=back(fu, N), Q=Q[:, :N], R=back(R, N),
             M=torch.zeros(B, N, 13, 12, device="cuda", dtype=torch.float64), q=q[:, :N], r=r, c=c[:, 1:], c0=c[:, 0],
             QN=Q[:, N], qN=q[:, N])
    dX, dU, dV, alpha, status = _step(L, X, U, V, phi)
    e = alpha[:, None, None]
    return dict(X=_shifted(X + e * dX), U=_shifted(U + e * dU), V=_shifted(V + e * dV), status=status)


def exact(case, seed):
    kind = case["kind"]
    if kind == "srbd":
        return _exact_srbd(case, seed)
    wide = lambda d: {k: None if v is None else v.double() for k, v in d.items()}
    if kind == "direction":
        a, it = _lin_arrays(case, seed)
        return _exact_direction(case, wide(a), [v.double() for v in it])
    a = _arrays(case, seed)
    if kind == "certify":
        return _exact_certify(case, wide(a), [v.double() for v in _certify_point(case, seed, a)])
    start = [v.double() for v in _start(case, seed, a)]
    return (_exact_solve if kind == "solve" else _exact_tick)(case, wide(a), start)
