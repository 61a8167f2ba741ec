"""The block Riccati kernel on LDS operand tiles (k_lqr_tile) with its forward
chain and costates, at the edges of its tiles, against the FP64 oracle.  FP32
tolerances are those of the other FP32 kernels (tests/test_gpu_parity.py): 2e-4
of max(1, |oracle|) on X, ten times that on U and V."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from caller_problem import linearization, make_caller_instance, start  # noqa: E402
from mpx_amd import synthetic as syn  # noqa: E402
from oracle import pdilqr as orc  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = dict(X=2e-4, U=2e-3, V=2e-3)


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1.0, np.max(np.abs(b)))) if np.size(b) else 0.0


def _check(insts, start_kind, iters, dtype=torch.float32, tol=TOL, **tune):
    from mpx_amd.problem import DeviceBatch, SQPSolver
    starts = [syn.initial_iterate(d, start_kind) for d in insts]
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    solver = SQPSolver(batch, **tune)
    it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
    refs = [orc.solve(d, *s, iters) for d, s in zip(insts, starts)]
    for k in range(iters):
        st = solver.iterate(it)
        torch.cuda.synchronize()
        for i in range(len(insts)):
            assert int(st["status"][i]) == 0, (k, i)
            for key, t in tol.items():
                e = _rel(it[key][i].double().cpu().numpy(), refs[i][k][key])
                assert e < t, (k, i, key, e)


@pytest.mark.parametrize("n,m,p,box", [
    (48, 16, 0, True),     # n + 1 in a tile of its own
    (62, 3, 1, False),     # ragged rows, one control tile
    (63, 12, 16, True),    # n + 1 = 64, p = 16
    (64, 17, 5, True),     # m one past a tile
    (79, 32, 12, True),    # the largest
    (1, 18, 2, False),     # one state, one tile
    (15, 32, 0, True), (16, 20, 3, False), (33, 31, 7, True),
])
def test_tanh_model(n, m, p, box):
    print(f"tile kernel tanh n={n} m={m} p={p} box={box}", flush=True)
    _check([syn.make_instance(4, i, n=n, m=m, N=5, p=p, box=box) for i in range(2)], "rollout", 2)


@pytest.mark.parametrize("n,m", [(50, 7), (49, 18), (18, 19)])
def test_ltv_diagonals_outside_the_unit_range(n, m):
    """A_t whose diagonal entries lie inside and outside [1/2, 2]: the unit part
    is split off for some rows only, and from stage to stage."""
    print(f"tile kernel LTV n={n} m={m}", flush=True)
    insts = []
    for i in range(2):
        d = syn.make_instance(1, i, n=n, m=m, N=6)
        rng = np.random.default_rng([5, i])
        A = d["A"].copy()
        for t in range(6):
            A[t][np.arange(n), np.arange(n)] = rng.choice([0.0, 0.1, 0.5, 0.9, 1.0, 1.1, -1.0], n)
        insts.append(dict(d, A=A))
    _check(insts, "tile", 1)


@pytest.mark.parametrize("shape", [dict(n=16, m=12, N=9), dict(n=52, m=9, N=6, p=3, box=True),
                                   dict(n=20, m=18, N=6, p=2)])
def test_caller_linearisation(shape):
    """The step from the caller's linearisation, cross term included."""
    from mpx_amd.caller import CallerBatch, CallerSolver
    print(f"tile kernel caller {shape}", flush=True)
    insts = [make_caller_instance(i, **shape) for i in range(2)]
    i0 = insts[0]
    p, box = i0["p"], i0["ulo"] is not None
    st = lambda k: np.stack([d[k] for d in insts])
    batch = CallerBatch(2, i0["n"], i0["m"], i0["N"], st("x0"), D=st("D") if p else None, E=st("E") if p else None,
                        e=st("e") if p else None, ulo=st("ulo") if box else None, uhi=st("uhi") if box else None)
    solver = CallerSolver(batch)
    starts = [start(d) for d in insts]
    it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
    refs = [orc.sqp_step(d, *s) for d, s in zip(insts, starts)]
    lins = [linearization(d, s[0], r["Uin"]) for d, s, r in zip(insts, starts, refs)]
    batch.set_linearization(**{key: np.stack([l[key] for l in lins]) for key in lins[0]})
    dX, dU, _ = solver.direction(it)
    torch.cuda.synchronize()
    for i, r in enumerate(refs):
        assert _rel(dX[i].double().cpu().numpy(), r["dX"]) < TOL["X"]
        assert _rel(dU[i].double().cpu().numpy(), r["dU"]) < TOL["U"]


@pytest.mark.parametrize("wl,n,m,p", [
    (3, 1, 1, 0), (3, 15, 16, 4), (4, 16, 8, 0), (3, 20, 9, 16), (4, 47, 16, 3), (3, 63, 5, 2), (1, 33, 12, 0),
])
def test_fp64(wl, n, m, p):
    """FP64 (matrix cores): differs from the oracle by the order of sums."""
    print(f"tile kernel FP64 wl={wl} n={n} m={m} p={p}", flush=True)
    shape = dict(n=n, m=m, N=5) if wl == 1 else dict(n=n, m=m, N=5, p=p)
    _check([syn.make_instance(wl, i, **shape) for i in range(2)], "tile" if wl == 1 else "rollout", 1 if wl == 1 else 2,
           torch.float64, dict(X=1e-9, U=1e-8, V=1e-8))
