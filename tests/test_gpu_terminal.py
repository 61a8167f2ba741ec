"""A terminal weight Q_N that is not symmetric (a caller's J'WJ in FP32 is not, to
the bit): the tile recursion (k_lqr_tile) reads it by its rows, as the block
recursion does (k_lqr_seq, which flags bit 1 selects).  The two differ by the
order of sums: tolerances are those of tests/test_gpu_tile.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from caller_problem import linearization, make_caller_instance, start  # noqa: E402
from mpx_amd import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
TOL = {F32: dict(X=2e-4, U=2e-3, V=2e-3), F64: dict(X=1e-9, U=1e-8, V=1e-8)}


def _rel(a, b):
    return float((a - b).abs().max() / max(1.0, float(b.abs().max())))


def _skewed(rng, M, scale):
    """M with entries off the diagonal that differ from their mirror images."""
    E = scale * rng.standard_normal(M.shape)
    k = np.arange(M.shape[-1])
    E[..., k, k] = 0
    return M + E


@pytest.mark.parametrize("dtype,n,m,N,p,box,cross", [
    (F32, 16, 12, 9, 0, False, True), (F32, 63, 5, 4, 3, True, True), (F32, 65, 16, 1, 0, False, False),
    (F32, 20, 18, 6, 2, False, True), (F32, 79, 32, 3, 0, True, False),
    (F64, 13, 12, 5, 0, False, True), (F64, 48, 7, 3, 2, True, True),
])
def test_caller(dtype, n, m, N, p, box, cross):
    print(f"skewed Q_N caller {dtype} n={n} m={m} N={N} p={p}", flush=True)
    from mpx_amd.caller import CallerBatch, CallerSolver
    insts = [make_caller_instance(i, n=n, m=m, N=N, p=p, box=box) for i in range(2)]
    st = lambda k: np.stack([d[k] for d in insts])
    batch = CallerBatch(2, n, m, N, st("x0"), D=st("D") if p else None, E=st("E") if p else None,
                        e=st("e") if p else None, ulo=st("ulo") if box else None, uhi=st("uhi") if box else None,
                        cross=cross, dtype=dtype)
    starts = [start(d) for d in insts]
    lins = [linearization(d, s[0], s[1]) for d, s in zip(insts, starts)]
    lin = {k: np.stack([v[k] for v in lins]) for k in lins[0]}
    rng = np.random.default_rng(11)
    lin["R"] = lin["R"] + 0.5 * np.eye(m)
    lin["QN"] = _skewed(rng, lin["QN"], 0.5)
    if not cross:
        del lin["M"]
    batch.set_linearization(**lin)
    out = []
    for flags in (2, 0):
        it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
        out.append([x.clone() for x in CallerSolver(batch, flags=flags).direction(it)])
        torch.cuda.synchronize()
    (rX, rU, _), (dX, dU, _) = out
    assert torch.isfinite(rX).all() and torch.isfinite(rU).all()
    assert _rel(dX, rX) < TOL[dtype]["X"] and _rel(dU, rU) < TOL[dtype]["U"]


@pytest.mark.parametrize("dtype,model,n,m,p", [
    (F32, "tanh", 48, 12, 2), (F32, "tanh", 70, 20, 0), (F32, "ltv", 52, 9, 3), (F64, "tanh", 36, 12, 4),
    (F64, "ltv", 17, 5, 0),
])
def test_iterate(dtype, model, n, m, p):
    """The multipliers too, which the costates S_t dx + s_t give."""
    print(f"skewed Q_N {dtype} {model} n={n} m={m} p={p}", flush=True)
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(3, i, n=n, m=m, N=6, p=p, model=model) for i in range(2)]
    for i, d in enumerate(insts):
        rng = np.random.default_rng([13, i])
        d["R"] = d["R"] + 0.5 * np.eye(m)
        d["QN"] = _skewed(rng, d["QN"], 0.5)
    starts = [syn.initial_iterate(d, "rollout") for d in insts]
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    out = []
    for flags in (2, 0):
        it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
        st = SQPSolver(batch, flags=flags).iterate(it)
        torch.cuda.synchronize()
        out.append((it, st["alpha"].clone()))
    (ref, ra), (it, a) = out
    assert torch.equal(ra, a)
    for k, t in TOL[dtype].items():
        assert torch.isfinite(ref[k]).all()
        assert _rel(it[k], ref[k]) < t, k
