"""Model evaluation (g, c) and the KKT residual on the device against the FP64
oracle, in the row form (k_eval_rows), the matrix-core form (k_eval_mma) and the
general kernels, at the edges of their tiles.  FP64 differs from the oracle by
the order of sums of at most 80 terms (1e-12 of the largest entry); FP32 rounds
the inputs and those sums (80 * 2^-24 = 5e-6, with a factor of 4: 2e-5)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402
from oracle import pdilqr as orc  # noqa: E402

pytestmark = pytest.mark.gpu


def _point(d, i):
    r = np.random.default_rng([3, i])
    N, n, m, p = d["N"], d["n"], d["m"], d["p"]
    f = lambda a: a.astype(np.float32).astype(np.float64)
    return (f(r.standard_normal((N + 1, n))), f(r.uniform(-0.9, 0.9, (N, m))), f(r.standard_normal((N + 1, n))),
            f(0.1 * r.standard_normal((N, p))), f(r.uniform(0.01, 0.5, (N, 2 * m))))


def _setup(wl, dtype, B=2, **shape):
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(wl, i, **shape) for i in range(B)]
    for d in insts:   # inputs exact in FP32
        for k, v in d.items():
            if isinstance(v, np.ndarray):
                d[k] = v.astype(np.float32).astype(np.float64)
    pts = [_point(d, i) for i, d in enumerate(insts)]
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    it = batch.iterate_from(*[np.stack([q[k] for q in pts]) for k in range(5)])
    return insts, pts, SQPSolver(batch), it


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
@pytest.mark.parametrize("wl,shape", [
    (3, dict(n=1, m=1, N=1, p=1)), (3, dict(n=15, m=16, N=16, p=5)), (4, dict(n=16, m=3, N=17, p=2)),
    (4, dict(n=17, m=7, N=33, p=16)), (3, dict(n=48, m=16, N=15, p=17)), (4, dict(n=36, m=12, N=18, p=8)),
    (4, dict(n=49, m=20, N=6, p=3)), (3, dict(n=80, m=64, N=5, p=0)), (3, dict(n=81, m=5, N=4, p=2)),
    (1, dict(n=33, m=9, N=7)), (2, dict(n=20, m=17, N=9)),
])
def test_model_eval_and_kkt(wl, shape, dtype, tol):
    print(f"eval wl={wl} {shape} {dtype}", flush=True)
    insts, pts, solver, it = _setup(wl, dtype, **shape)
    g, c = solver.model_eval(it["X"], it["U"])
    kkt = solver.kkt(it)
    torch.cuda.synchronize()
    for i, (d, q) in enumerate(zip(insts, pts)):
        rg, rc = orc.model_evaluator_helper(d, q[0], q[1])
        rk = orc.kkt_residual(d, *q)
        assert np.max(np.abs(g[i].double().cpu().numpy() - rg)) <= tol * max(1.0, np.max(np.abs(rg)))
        assert np.max(np.abs(c[i].double().cpu().numpy() - rc)) <= tol * max(1.0, np.max(np.abs(rc)))
        assert abs(float(kkt[i]) - rk) <= tol * max(1.0, rk)


@pytest.mark.parametrize("n", [36, 37])
def test_nan_stays_in_its_stage(n):
    """A NaN in x_t reaches g_t and the rows c_t, c_{t+1} only."""
    insts, pts, solver, it = _setup(3, torch.float32, n=n, m=12, N=20, p=2)
    it["X"][0, 7, 0] = float("nan")
    g, c = solver.model_eval(it["X"], it["U"])
    torch.cuda.synchronize()
    bad_g, bad_c = torch.isnan(g).cpu().numpy(), torch.isnan(c).any(-1).cpu().numpy()
    assert bad_g.nonzero()[1].tolist() == [7] and not bad_g[1].any()
    assert bad_c.nonzero()[1].tolist() == [7, 8] and not bad_c[1].any()


def test_launches():
    """One launch for the model evaluation, two for the residual (the evaluation and
    its sum), the terminal stage in the matrix-core form's: evaluations of a few
    stages are bound by their launches."""
    import ctypes as C
    from mpx_amd import _lib as L
    from mpx_amd.problem import _ptr
    insts, pts, solver, it = _setup(3, torch.float32, n=12, m=12, N=25, p=0)
    b = solver.batch
    g, c = solver.model_eval(it["X"], it["U"])
    k = solver.kkt(it)
    ci, ws = b.c_iterate(it), C.c_void_p(solver.ws.data_ptr())
    hip = C.CDLL("libamdhip64.so")
    counts = []
    for what in ("model_eval", "kkt"):
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
            if what == "model_eval":
                L.check(solver.lib.mpxkkt_model_eval(st, C.byref(b.problem), _ptr(it["X"]), _ptr(it["U"]), _ptr(g), _ptr(c)))
            else:
                L.check(solver.lib.mpxkkt_kkt_residual(st, C.byref(b.problem), C.byref(solver.params), C.byref(ci), _ptr(k),
                                                       ws, solver.ws_bytes))
        n = C.c_size_t(0)
        assert hip.hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
        counts.append(n.value)
    assert counts == [1, 2]
