"""The problem's views in layouts other than the dense instance-major one: stage-
major, padded with the base off 16 bytes, shared by the batch, and with stage
strides whose whole horizon is past one 32-bit buffer descriptor.  What lies
between a view's entries is NaN.  Results against the FP64 oracle; tolerances are
those of tests/test_gpu_tile.py (FP32 iterations), tests/test_gpu_parity.py (FP64,
the order of sums) and tests/test_gpu_eval.py (evaluation)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from caller_problem import linearization, make_caller_instance, start as caller_start  # noqa: E402
from mpx_amd import synthetic as syn  # noqa: E402
from oracle import pdilqr as orc  # noqa: E402

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1.0, np.max(np.abs(b)))) if np.size(b) else 0.0


def _lay(batch, name, layout, keep, stage_stride=0):
    """Moves view ``name`` (a tensor [B, ...] or [B, stages, ...]) to a new layout;
    ``keep`` holds the buffer while the batch is in use."""
    x = batch.t[name]
    v = getattr(batch.problem, name)
    B, es = x.shape[0], x.element_size()
    stages = x.shape[1] if v.stage_stride else 1
    length = x[0].numel() // stages
    if layout == "shared":
        assert all(torch.equal(x[0], x[i]) for i in range(B)), name
        v.batch_stride = 0
        return
    if layout == "stage":     # [stage][instance][entry], a gap after each stage
        sb, st, base = length, B * length + 4, 0
    elif layout == "pad":     # odd strides, the base one entry off an aligned address
        st = length + 1
        sb, base = stages * st + 3, 1
    else:                     # "far": stage-major, stage_stride apart
        sb, st, base = length, stage_stride, 0
    st = st if stages > 1 else 0
    buf = torch.full((base + (B - 1) * sb + (stages - 1) * st + length,), float("nan"), dtype=x.dtype, device=x.device)
    torch.as_strided(buf, (B, stages, length), (sb, st, 1), base).copy_(x.reshape(B, stages, length))
    v.ptr, v.batch_stride, v.stage_stride = buf.data_ptr() + base * es, sb, st
    keep.append(buf)


def _views(batch):
    names = ["A", "B", "Q", "R", "QN", "xref", "uref", "x0"] + (["W"] if batch.model == "tanh" else [])
    return names + (["D", "E", "e"] if batch.p else []) + (["ulo", "uhi"] if batch.box else [])


def _problem(model, dtype, layout, n, m, N, p, box, B=2, far=0):
    """Instances, their reference data and a batch in the layout."""
    from mpx_amd.problem import DeviceBatch
    insts = [syn.make_instance(4, i, n=n, m=m, N=N, p=p, box=box, model=model) for i in range(B)]
    for i, d in enumerate(insts):
        r = np.random.default_rng([7, i])
        d["xref"] = 0.1 * r.standard_normal((N + 1, n))
        d["uref"] = 0.1 * r.standard_normal((N, m))
        if p:
            d["e"] = 0.1 * r.standard_normal((N, p))
        for k, v in d.items():   # inputs exact in FP32
            if isinstance(v, np.ndarray):
                d[k] = v.astype(np.float32).astype(np.float64)
    if layout == "shared":
        insts = [dict(insts[0], x0=d["x0"]) for d in insts]
    batch = DeviceBatch.from_instances(insts, dtype=dtype)
    keep = []
    for name in _views(batch):
        if layout == "far":
            if getattr(batch.problem, name).stage_stride:
                _lay(batch, name, "far", keep, far)
        elif not (layout == "shared" and name == "x0"):
            _lay(batch, name, layout, keep)
    return insts, batch, keep


def _iterate_dict(batch, starts, off):
    """Iterate arrays whose base lies ``off`` entries past an aligned address."""
    it = batch.iterate_from(*[np.stack([s[k] for s in starts]) for k in range(5)])
    if not off:
        return it
    out = {}
    for k, x in it.items():
        buf = torch.full((x.numel() + off,), float("nan"), dtype=x.dtype, device=x.device)
        out[k] = buf[off:].view(x.shape)
        out[k].copy_(x)
    return out


def _check_iterations(insts, batch, dtype, off=0, iters=2):
    from mpx_amd.problem import SQPSolver
    starts = [syn.initial_iterate(d, "rollout") for d in insts]
    solver = SQPSolver(batch)
    it = _iterate_dict(batch, starts, off)
    refs = [orc.solve(d, *s, iters) for d, s in zip(insts, starts)]
    tol = 2e-4 if dtype == F32 else 1e-9
    for k in range(iters):
        st = solver.iterate(it)
        torch.cuda.synchronize()
        for i in range(len(insts)):
            assert int(st["status"][i]) == 0, (k, i)
            for key, t in (("X", tol), ("U", 10 * tol), ("V", 10 * tol), ("Yeq", 10 * tol)):
                e = _rel(it[key][i].double().cpu().numpy(), refs[i][k][key])
                assert e < t, (k, i, key, e)


def _check_evaluation(insts, batch, dtype, off=0):
    from mpx_amd.problem import SQPSolver
    pts = []
    for i, d in enumerate(insts):
        r = np.random.default_rng([3, i])
        N, n, m, p = d["N"], d["n"], d["m"], d["p"]
        f = lambda a: a.astype(np.float32).astype(np.float64)
        pts.append((f(r.standard_normal((N + 1, n))), f(r.uniform(-0.9, 0.9, (N, m))), f(r.standard_normal((N + 1, n))),
                    f(0.1 * r.standard_normal((N, p))), f(r.uniform(0.01, 0.5, (N, 2 * m)))))
    solver = SQPSolver(batch)
    it = _iterate_dict(batch, pts, off)
    g, c = solver.model_eval(it["X"], it["U"])
    kkt = solver.kkt(it)
    torch.cuda.synchronize()
    tol = 2e-5 if dtype == F32 else 1e-12
    for i, (d, q) in enumerate(zip(insts, pts)):
        rg, rc = orc.model_evaluator_helper(d, q[0], q[1])
        rk = orc.kkt_residual(d, *q)
        assert _rel(g[i].double().cpu().numpy(), rg) <= tol
        assert _rel(c[i].double().cpu().numpy(), rc) <= tol
        assert abs(float(kkt[i]) - rk) <= tol * max(1.0, rk)


@pytest.mark.parametrize("layout", ["stage", "pad", "shared"])
@pytest.mark.parametrize("dtype,model,n,m,p,box", [
    # wave recursion, matrix-core linearisation, trials and evaluation, adjoint
    (F32, "tanh", 36, 12, 8, True), (F32, "tanh", 17, 5, 3, False),
    # tile recursion, row forms
    (F32, "tanh", 64, 16, 12, True), (F32, "tanh", 52, 20, 3, True),
    # stage-varying: wave and tile recursion
    (F32, "ltv", 20, 8, 3, True), (F32, "ltv", 50, 18, 0, True),
    # FP64 tile recursion
    (F64, "tanh", 36, 12, 8, True), (F64, "ltv", 20, 7, 2, True),
])
def test_layouts(dtype, model, n, m, p, box, layout):
    print(f"strides {dtype} {model} n={n} m={m} p={p} {layout}", flush=True)
    insts, batch, keep = _problem(model, dtype, layout, n, m, 18, p, box)
    off = 1 if layout == "pad" else 0
    _check_evaluation(insts, batch, dtype, off)
    _check_iterations(insts, batch, dtype, off, 1 if model == "ltv" else 2)


@pytest.mark.parametrize("layout", ["stage", "pad"])
@pytest.mark.parametrize("dtype,n,m,p,cross", [(F32, 13, 12, 3, True), (F32, 15, 16, 0, False), (F32, 20, 18, 2, True),
                                               (F32, 52, 9, 3, True), (F64, 17, 5, 2, False)])
def test_caller_layouts(dtype, n, m, p, cross, layout):
    """A caller's linearisation in other layouts: the step's bits of the dense one."""
    from mpx_amd.caller import CallerBatch, CallerSolver
    print(f"strides caller {dtype} n={n} m={m} p={p} {layout}", flush=True)
    insts = [make_caller_instance(i, n=n, m=m, N=6, p=p, box=True) for i in range(2)]
    st = lambda k: np.stack([d[k] for d in insts])
    batch = CallerBatch(2, n, m, 6, st("x0"), D=st("D") if p else None, E=st("E") if p else None,
                        e=st("e") if p else None, ulo=st("ulo"), uhi=st("uhi"), cross=cross, dtype=dtype)
    starts = [caller_start(d) for d in insts]
    lins = [linearization(d, s[0], s[1]) for d, s in zip(insts, starts)]
    lin = {k: np.stack([v[k] for v in lins]) for k in lins[0]}
    if not cross:
        del lin["M"]
    batch.set_linearization(**lin)
    out, keep = [], []
    for k in range(2):
        if k:
            batch.t = {**batch.t, **batch.lin}
            for name, x in batch.t.items():
                if x is not None:
                    _lay(batch, name, layout, keep)
        it = batch.iterate_from(*[np.stack([s[j] for s in starts]) for j in range(5)])
        out.append([x.clone() for x in CallerSolver(batch).direction(it)])
        torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("n,m,N,stride", [
    (12, 4, 17, 2**26 + 4),     # past 4 GiB: 32-bit byte offsets would wrap
    (12, 4, 17, 2**25 + 64),    # past 1 GiB: the offset of absent entries would lie between two stages
    (9, 5, 67, 2**22 - 5),     # the same with strides the row forms take
])
def test_horizon_past_one_descriptor(n, m, N, stride):
    """The tanh model's per-stage views with large stage strides."""
    print(f"far stages n={n} m={m} N={N} stride={stride}", flush=True)
    insts, batch, keep = _problem("tanh", F32, "far", n, m, N, 3, True, far=stride)
    # bounds that vary with the stage take a stage stride too
    for name in ("ulo", "uhi"):
        x = batch.t[name]
        buf = torch.full(((N - 1) * stride + 2 * m,), float("nan"), dtype=x.dtype, device=x.device)
        torch.as_strided(buf, (2, N, m), (m, stride, 1)).copy_(x[:, None].expand(2, N, m))
        v = getattr(batch.problem, name)
        v.ptr, v.batch_stride, v.stage_stride = buf.data_ptr(), m, stride
        keep.append(buf)
    _check_evaluation(insts, batch, F32)
    _check_iterations(insts, batch, F32)
    keep.clear()
    torch.cuda.empty_cache()
