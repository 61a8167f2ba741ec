"""The linearisation and the trials with rows over a block's waves
(k_linearize_rows, k_trials_rows) through whole iterations against the FP64
oracle, at the edges of their row tiles, of a block's 16 stages and of a pass of
8 equality rows, from controls on and past their bounds.  Tolerances are those
of tests/test_gpu_tile.py (FP32) and tests/test_gpu_parity.py (FP64, the order
of sums: 1e-9, ten times that on U and V)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402
from oracle import pdilqr as orc  # noqa: E402

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1.0, np.max(np.abs(b)))) if np.size(b) else 0.0


@pytest.mark.parametrize("dtype,wl,n,m,N,p", [
    (torch.float32, 4, 49, 3, 16, 1), (torch.float32, 4, 80, 32, 17, 9), (torch.float32, 4, 20, 17, 33, 20),
    (torch.float32, 4, 64, 16, 1, 8), (torch.float32, 3, 78, 30, 15, 16), (torch.float32, 3, 1, 17, 2, 0),
    (torch.float64, 4, 64, 16, 17, 17), (torch.float64, 4, 1, 1, 15, 0), (torch.float64, 4, 16, 16, 16, 8),
    (torch.float64, 3, 48, 5, 33, 64), (torch.float64, 4, 37, 12, 1, 7),
])
def test_iterations(dtype, wl, n, m, N, p):
    print(f"rows {dtype} wl={wl} n={n} m={m} N={N} p={p}", flush=True)
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(wl, i, n=n, m=m, N=N, p=p) for i in range(2)]
    starts = []
    for i, d in enumerate(insts):
        s = [np.array(a) for a in syn.initial_iterate(d, "rollout")]
        if d["ulo"] is not None:   # on and past both bounds
            s[1][0, 0] = d["uhi"][0] + 0.1
            s[1][-1, -1] = d["ulo"][-1]
        starts.append(s)
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    solver = SQPSolver(batch)
    it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
    refs = [orc.solve(d, *s, 2) for d, s in zip(insts, starts)]
    tol = 2e-4 if dtype == torch.float32 else 1e-9
    for k in range(2):
        st = solver.iterate(it)
        torch.cuda.synchronize()
        for i in range(2):
            assert int(st["status"][i]) == 0, (k, i)
            for key, t in (("X", tol), ("U", 10 * tol), ("V", 10 * tol), ("Yeq", 10 * tol)):
                e = _rel(it[key][i].double().cpu().numpy(), refs[i][k][key])
                assert e < t, (k, i, key, e)
