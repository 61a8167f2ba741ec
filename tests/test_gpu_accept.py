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


@pytest.mark.parametrize("n,m,p", [(36, 12, 3), (24, 12, 0), (9, 4, 1)])
def test_gated_iterations(n, m, p):
    """A solve whose instances stop after different iterations, among blocks whose
    other instances go on: the bits, counts and costs of each instance alone."""
    from mpx_amd.problem import DeviceBatch, SQPSolver
    insts = [syn.make_instance(3, i, n=n, m=m, N=12, p=p, box=True) for i in range(5)]
    for d, s in zip(insts, (1.0, 0.0, 4.0, 1e-3, 0.3)):
        d["x0"] = s * d["x0"]
    start = [syn.initial_iterate(d, "tile") for d in insts]

    def solve(ds, ss):
        batch = DeviceBatch.from_instances(ds, dtype=torch.float32)
        it = batch.iterate_from(*[np.stack([s[k] for s in ss]) for k in range(5)])
        iters, cost, cc, _ = SQPSolver(batch).solve(it, max_iter=6)
        torch.cuda.synchronize()
        return [it[k] for k in ("X", "U", "V", "Yeq", "Ybox")] + [iters, cost, cc]

    alone = [solve([d], [s]) for d, s in zip(insts, start)]
    assert len({int(a[5][0]) for a in alone}) > 1
    for copies in (1, 120, 410):   # 5, 600 and 2050 instances
        print(f"gated n={n} m={m} p={p} copies={copies}", flush=True)
        out = solve(insts * copies, start * copies)
        for i, ref in enumerate(alone):
            for a, r in zip(out, ref):
                assert torch.equal(a[i::5], r.expand_as(a[i::5])), (i, copies)
