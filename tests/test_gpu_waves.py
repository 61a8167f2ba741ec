"""k_lqr_waves (NT + 1 waves per instance, batches up to 512) returns the bits
of k_lqr_wave (larger batches): the same instances alone and among 513, at the
edges of the state tiles, of the control and equality tiles' steps, for the
tanh and the stage-varying model."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mpx_amd import synthetic as syn  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wl,n,m,p,flags", [
    (3, 1, 1, 0, 0), (3, 15, 16, 16, 0), (4, 12, 5, 0, 0), (3, 16, 4, 3, 0), (4, 31, 12, 1, 0), (3, 32, 8, 8, 0),
    (4, 33, 16, 0, 0), (3, 36, 12, 8, 0), (3, 47, 13, 16, 0), (3, 36, 12, 8, 8), (3, 44, 1, 2, 16),
    (1, 9, 3, 0, 0), (2, 19, 7, 3, 0), (1, 36, 12, 0, 0), (1, 47, 16, 0, 0),
])
def test_same_bits_for_every_batch_size(wl, n, m, p, flags):
    print(f"waves wl={wl} n={n} m={m} p={p} flags={flags}", flush=True)
    from mpx_amd.problem import DeviceBatch, SQPSolver
    shape = dict(n=n, m=m, N=4) if wl in (1, 2) else dict(n=n, m=m, N=4, p=p)
    insts = [syn.make_instance(wl, i, **shape) for i in range(2)]
    out = []
    for copies in (1, 257):   # 2 and 514 instances
        group = insts * copies
        starts = [syn.initial_iterate(d, "tile" if wl == 1 else "rollout") for d in insts] * copies
        batch = DeviceBatch.from_instances(group, dtype=torch.float32)
        solver = SQPSolver(batch, flags=flags)
        it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
        for _ in range(2):
            solver.iterate(it)
        torch.cuda.synchronize()
        out.append({k: it[k][-2:].clone() for k in ("X", "U", "V")})
    for k in out[0]:
        assert torch.isfinite(out[0][k]).all() and torch.equal(out[0][k], out[1][k]), k
