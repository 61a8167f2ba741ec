"""k_ls_accept with a block per part (few instances) and one block per instance
(many): the same bits, at sizes below, at and past a part of 1024 entries, with
and without equality rows and boxes, through a solve's gated iterations too."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wl,n,m,N,p", [(3, 8, 4, 127, 9), (3, 8, 4, 255, 0), (4, 31, 9, 33, 5), (4, 3, 1, 2, 0), (3, 36, 12, 28, 36)])
def test_same_bits_for_one_and_many_instances(wl, n, m, N, p):
    print(f"accept wl={wl} n={n} m={m} N={N} p={p}", flush=True)
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(wl, i, n=n, m=m, N=N, p=p) for i in range(2)]
    start = [syn.initial_iterate(d, "rollout") for d in insts]
    out = []
    for copies in (300, 1024):   # 600 instances: three blocks each; 2048: one
        batch = DeviceBatch.from_instances(insts * copies, dtype=torch.float32)
        solver = SQPSolver(batch)
        it = batch.iterate_from(*[np.stack([s[k] for s in start] * copies) for k in range(5)])
        st = solver.iterate(it)
        torch.cuda.synchronize()
        out.append([it[k][-2:].clone() for k in ("X", "U", "V", "Yeq", "Ybox")] + [st["alpha"][-2:].clone()])
        assert all(torch.equal(it[k][:2], it[k][-2:]) for k in ("X", "U", "V"))
    for a, b in zip(*out):
        assert torch.equal(a, b)
