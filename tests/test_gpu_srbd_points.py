"""SRBD iterations at horizons where the trial points end inside, at and just
past a block of the cost (16 points) or of the dynamics (64), against the FP64
oracle at the tolerance of tests/test_gpu_srbd.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import pdilqr as orc  # noqa: E402
from test_gpu_srbd import KEYS, _rel, _setup  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N", [(1, 1), (2, 15), (1, 31), (5, 32), (1, 2)])
def test_iteration_fp64(B, N):
    print(f"srbd points B={B} N={N}", flush=True)
    solver, insts, it, cur = _setup(B, N, True, torch.float64)
    refs = [orc.sqp_step(d, *c) for d, c in zip(insts, cur)]
    solver.iterate(it)
    torch.cuda.synchronize()
    for i, r in enumerate(refs):
        for key in KEYS:
            e = _rel(it[key][i].double().cpu().numpy(), r[key])
            assert e < 1e-9, (i, key, e)
