"""The stop test's sums (sum g_t^2, sum |c|^2) that a solve returns, against the
FP64 oracle at the iterate it returns: the matrix-core form, the row form and the
general kernel at the edges of their tiles.  With e the error of an entry of g or
c (tests/test_gpu_eval.py: 2e-5 of the largest in FP32, 1e-12 in FP64) a sum of M
squares s is off by at most 2 sqrt(s M) e + M e^2."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402
from oracle import pdilqr as orc  # noqa: E402

pytestmark = pytest.mark.gpu


F32, F64 = torch.float32, torch.float64


@pytest.mark.parametrize("dtype,n,m,N,model", [
    (F32, 36, 12, 1, "tanh"), (F32, 36, 12, 15, "tanh"), (F32, 37, 5, 16, "tanh"), (F32, 48, 16, 17, "tanh"),
    (F32, 12, 4, 33, "tanh"), (F32, 49, 20, 6, "tanh"), (F32, 80, 9, 5, "tanh"), (F32, 81, 5, 4, "tanh"),
    (F32, 19, 7, 9, "ltv"), (F64, 36, 12, 15, "tanh"), (F64, 17, 16, 33, "ltv"), (F64, 63, 5, 4, "tanh"),
])
def test_sums(dtype, n, m, N, model):
    tol = 2e-5 if dtype == F32 else 1e-12
    from mpx_amd.problem import DeviceBatch, SQPSolver
    print(f"stop n={n} m={m} N={N} {model} {dtype}", flush=True)
    insts = [syn.make_instance(3, i, n=n, m=m, N=N, p=0, model=model) for i in range(2)]
    for d in insts:   # inputs exact in FP32
        for k, v in d.items():
            if isinstance(v, np.ndarray):
                d[k] = v.astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(17)
    start = [syn.initial_iterate(d, "rollout") for d in insts]
    X = np.stack([s[0] for s in start]) + rng.standard_normal((2, N + 1, n))
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    it = batch.iterate_from(X, *[np.stack([s[k] for s in start]) for k in range(1, 5)])
    iters, cost, cc, _ = SQPSolver(batch).solve(it, max_iter=0)
    torch.cuda.synchronize()
    for i, d in enumerate(insts):
        g, c = orc.model_evaluator_helper(d, it["X"][i].double().cpu().numpy(), it["U"][i].double().cpu().numpy())
        for got, v in ((float(cost[i]), g), (float(cc[i]), c)):
            s, M, e = float(np.sum(v * v)), v.size, tol * max(1.0, float(np.max(np.abs(v))))
            assert abs(got - s) <= 2 * np.sqrt(s * M) * e + M * e * e, (i, got, s)
