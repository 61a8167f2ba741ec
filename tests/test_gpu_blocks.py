"""Waves of several instances in one block (batches past 512: three or four
instances per block of the wave kernels, the last block not full): every instance
gets the bits it gets alone."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,n,m,p", [("tanh", 36, 12, 8), ("tanh", 45, 14, 3), ("tanh", 24, 12, 0), ("tanh", 9, 4, 0),
                                         ("ltv", 20, 7, 3)])
def test_same_bits_in_every_block(model, n, m, p):
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(4, i, n=n, m=m, N=5, p=p, model=model) for i in range(2)]
    start = [syn.initial_iterate(d, "rollout") for d in insts]
    ref = None
    for B in (2, 514, 768, 770, 1025, 1538):
        print(f"blocks {model} n={n} m={m} B={B}", flush=True)
        k = B // 2 + 1
        batch = DeviceBatch.from_instances((insts * k)[:B], dtype=torch.float32)
        it = batch.iterate_from(*[np.stack([s[j] for s in (start * k)[:B]]) for j in range(5)])
        solver = SQPSolver(batch)
        for _ in range(2):
            solver.iterate(it)
        torch.cuda.synchronize()
        out = [it[key].clone() for key in ("X", "U", "V", "Yeq", "Ybox")]
        if ref is None:
            ref = out
            continue
        for a, r in zip(out, ref):
            assert torch.isfinite(a).all()
            assert all(torch.equal(a[j::2], r[j:j + 1].expand_as(a[j::2])) for j in range(2)), B
