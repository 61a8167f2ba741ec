"""k_lqr_small (one wave per instance, a caller's linearisation of one tile)
returns the bits of k_lqr_seq, which flags bit 1 selects, at the edges of its
tiles; tests/test_gpu_caller.py holds both to the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from caller_problem import linearization, make_caller_instance, start  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,N,p,box,cross", [
    (13, 12, 25, 0, False, True), (13, 12, 3, 4, True, False), (15, 16, 2, 16, True, True), (15, 13, 1, 1, False, True),
    (1, 1, 5, 0, True, False), (4, 3, 7, 5, False, True), (14, 5, 6, 15, True, True), (2, 16, 4, 0, False, True),
])
def test_same_bits_as_the_block_kernel(n, m, N, p, box, cross):
    print(f"small n={n} m={m} N={N} p={p} box={box} cross={cross}", flush=True)
    from mpx_amd.caller import CallerBatch, CallerSolver
    insts = [make_caller_instance(i, n=n, m=m, N=N, p=p, box=box) for i in range(3)]
    st = lambda k: np.stack([d[k] for d in insts])
    batch = CallerBatch(3, n, m, N, st("x0"), D=st("D") if p else None, E=st("E") if p else None,
                        e=st("e") if p else None, ulo=st("ulo") if box else None, uhi=st("uhi") if box else None, cross=cross,
                        dtype=torch.float32)
    starts = [start(d) for d in insts]
    lins = [linearization(d, s[0], s[1]) for d, s in zip(insts, starts)]
    lin = {k: np.stack([v[k] for v in lins]) for k in lins[0]}
    rng = np.random.default_rng(3)   # a terminal Hessian that is not exactly symmetric
    lin["QN"] = lin["QN"] + 1e-3 * rng.standard_normal(lin["QN"].shape)
    if not cross:
        del lin["M"]
    batch.set_linearization(**lin)
    out = []
    for flags in (0, 2):
        it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
        dX, dU, amax = CallerSolver(batch, flags=flags).direction(it)
        torch.cuda.synchronize()
        out.append((dX.clone(), dU.clone(), amax.clone()))
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)
