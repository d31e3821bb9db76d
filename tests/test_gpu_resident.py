"""The resident launch of the FP64 solve (launch "auto": one workgroup per tile of a member, members from a queue)
against the per-phase launches: the same bits in every output, over batches below, at and above the number of members
in flight, both sum orders, first guesses with halos, iteration caps, operator slots and data whose Fortran-order sums
cancel."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FIELDS = ("firstResidual", "lastResidual", "sumRHS", "rhsMax", "numIters", "converged", "outerIters")


@pytest.fixture(scope="module")
def problem():
    from mit_jax_amd import synthetic as S
    from mit_jax_amd.exchange import default_exchanger
    ex = default_exchanger()
    cls = [S.cg2d_case(0, p, nlev=n) for p, n in (("5point", 50), ("diagonal", 30), ("5point", 7))]
    slots = [torch.as_tensor(np.stack([c[1][k] for c in cls]), device="cuda") for k in range(6)]
    return ex, cls, slots


def _inputs(ex, cls, B, index):
    from mit_jax_amd import synthetic as S
    b = np.stack([S.rhs(cls[index[m]][0], 200 + m) for m in range(B)])
    x0 = np.stack([S._exch_np(ex.maps, "T", 1e-5 * S.rhs(cls[index[m]][0], 900 + m)) for m in range(B)])
    rng = np.random.default_rng(B)
    x0[:, :, :3] += 1e-6 * rng.normal(size=x0[:, :, :3].shape)  # halo values of the guess that no exchange writes
    if B > 1:
        b[1] = 0.0  # rhsNorm = 1
        b[-1] *= np.where(rng.random(b[-1].shape) < 0.5, -1e8, 1.0)  # sums that cancel
    norm = np.array([cls[k][2] for k in index])
    T = lambda a: torch.as_tensor(a, device="cuda")  # noqa: E731
    return T(b), T(x0), T(norm)


@pytest.mark.parametrize("B,order,tol,iters", [
    (1, "tile", 1e-12, 2000), (1, "fortran", 1e-7, 2000), (3, "fortran", 1e-12, 9), (18, "tile", 1e-9, 2000),
    (19, "fortran", 1e-5, 60), (20, "tile", 1e-12, 2000), (41, "tile", 1e-7, 2000), (2, "tile", 1e-12, 0),
    (2, "fortran", 1e-12, 1), (2, "tile", 1e6, 2000)])
def test_resident_equals_phases(problem, B, order, tol, iters):
    from mit_jax_amd import cg2d
    ex, cls, slots = problem
    index = np.arange(B, dtype=np.int32) % len(cls)
    b, x0, norm = _inputs(ex, cls, B, index)
    print(f"resident: B={B} order={order} tol={tol} max_iters={iters}", flush=True)
    kw = dict(cg2dNorm=norm, tolerance=tol, max_iters=iters, sum_order=order, op_index=index)
    x, d = cg2d.cg2d_fortran(ex, slots, b, x0, **kw)
    torch.cuda.synchronize()
    d.check()
    xr, dr = cg2d.cg2d_fortran(ex, slots, b, x0, launch="phases", **kw)
    torch.cuda.synchronize()
    assert int(d["launches"].max()) == 0 and int(dr["launches"].max()) > 0  # the two launch shapes
    assert torch.equal(x, xr)
    for k in FIELDS:
        assert torch.equal(d[k], dr[k]), k


def test_resident_fortran_sums_of_hard_data(problem):
    """The Fortran-order sums are chains cut into chunks that start from estimates; whatever the data, the bits are the
    chain's: ties in every addition, sums that cancel to little or nothing, magnitudes over 300 decades, sums of a few
    values among zeros, sums that pass a power of two again and again, denormal ones."""
    from mit_jax_amd import cg2d
    ex, cls, slots = problem
    wet = np.where(np.abs(cls[0][0].maskC[:, 0]) > 0, 1.0, 0.0)
    rng = np.random.default_rng(31)
    shape = wet.shape
    sign = np.where(rng.random(shape) < 0.5, -1.0, 1.0)
    data = [rng.integers(-4, 5, shape) * 0.5, sign * (1.0 + 1e-15 * rng.normal(size=shape)),
            sign * 10.0 ** rng.uniform(-150, 150, shape), np.where(rng.random(shape) < 1e-3, rng.normal(size=shape), 0.0),
            1.0 + 0.0 * sign, np.where(np.arange(shape[2]) % 2, 1.0, -1.0) * np.ones(shape), 1e-160 * rng.normal(size=shape)]
    b = torch.as_tensor(np.stack(data) * wet, device="cuda")
    B = len(data)
    norm = torch.full((B,), cls[0][2], dtype=torch.float64, device="cuda")
    index = np.zeros(B, np.int32)
    kw = dict(cg2dNorm=norm, tolerance=1e-7, max_iters=12, sum_order="fortran", op_index=index)
    print("resident: Fortran order, hard sums", flush=True)
    x, d = cg2d.cg2d_fortran(ex, slots, b, torch.zeros_like(b), **kw)
    torch.cuda.synchronize()
    xr, dr = cg2d.cg2d_fortran(ex, slots, b, torch.zeros_like(b), launch="phases", **kw)
    torch.cuda.synchronize()
    assert int(d["launches"].max()) == 0 and int(dr["launches"].max()) > 0
    bits = lambda a: a.contiguous().view(torch.int64) if a.dtype == torch.float64 else a  # noqa: E731
    assert torch.equal(bits(x), bits(xr))
    for k in FIELDS:
        assert torch.equal(bits(d[k]), bits(dr[k])), k


@pytest.mark.parametrize("B,kw", [
    (1, {}), (1, dict(tolerance=1e6)), (3, dict(max_iters=1)), (19, dict(max_iters=37)), (20, dict(max_outer=2)),
    (45, dict(inner_tolerance=1e-2)), (46, dict(max_iters=0)), (46, dict(inner_max_iters=20)), (61, {})])
def test_mixed_resident_equals_steps(problem, B, kw):
    """The mixed solve's resident launches (one workgroup per CU up to 45 members on 256 CUs, two beyond) against its
    step launches."""
    from mit_jax_amd import mixed
    ex, cls, slots = problem
    index = np.arange(B, dtype=np.int32)[::-1] % len(cls)
    b, x0, norm = _inputs(ex, cls, B, index)
    kw = dict(dict(tolerance=1e-11, max_iters=4000), **kw)
    print(f"mixed resident: B={B} {kw}", flush=True)
    x, d = mixed.cg2d_mixed(ex, slots, b, x0, cg2dNorm=norm, op_index=index, **kw)
    torch.cuda.synchronize()
    d.check()
    xr, dr = mixed.cg2d_mixed(ex, slots, b, x0, cg2dNorm=norm, op_index=index, block_threads=512, **kw)
    torch.cuda.synchronize()
    assert int(d["launches"].max()) == 0 and int(dr["launches"].max()) > 0
    assert torch.equal(x, xr)
    for k in FIELDS:
        assert torch.equal(d[k], dr[k]), k


def test_resident_member_stride_and_stream(problem):
    """Members further apart than a field, on a side stream, twice into the same workspace."""
    import ctypes
    from mit_jax_amd import _lib, cg2d
    ex, cls, slots = problem
    B, L = 5, ex.L
    index = np.zeros(B, np.int32)
    b, x0, norm = _inputs(ex, cls, B, index)
    ops = [a[0] for a in slots]
    xr, _ = cg2d.cg2d_fortran(ex, ops, b, x0, cg2dNorm=norm, tolerance=1e-10, max_iters=500, sum_order="tile",
                              launch="phases")
    stride = L.npad + 26
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        wide = [torch.full((B, stride), 7.0, dtype=torch.float64, device="cuda") for _ in range(3)]
        for w, a in zip(wide, (b, x0)):
            w[:, :L.npad] = a.reshape(B, -1)
        ops_s, keep = cg2d._ops_struct(ops, B, L, b.device)
        cfg = cg2d.config(L, B, 1e-10, 500, "tile")
        cfg.member_stride = stride
        lib = _lib.lib()
        n = lib.mj_cg2d_workspace_bytes(ctypes.byref(cfg))
        ws = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
        diag = torch.zeros(B * 48, dtype=torch.uint8, device="cuda")
        for _ in range(2):
            wide[2].fill_(7.0)
            _lib.check(lib.mj_cg2d_solve(ex.plan("T", b.device).handle, ctypes.byref(ops_s), *map(_lib.ptr, wide),
                                         _lib.ptr(norm), ctypes.byref(cfg), _lib.ptr(ws), ctypes.c_size_t(n),
                                         _lib.ptr(diag), _lib.stream_ptr()), "mj_cg2d_solve")
            side.synchronize()
            assert torch.equal(wide[2][:, :L.npad].reshape(xr.shape), xr)
            assert bool((wide[2][:, L.npad:] == 7.0).all())
    del keep


def test_resident_concurrent_streams(problem):
    """Solves on several streams at once, which together need more workgroups than the device holds."""
    from mit_jax_amd import cg2d
    ex, cls, slots = problem
    runs = []
    for i, (B, order) in enumerate(((19, "tile"), (12, "tile"), (7, "fortran"))):
        index = np.full(B, i % len(cls), np.int32)
        b, x0, norm = _inputs(ex, cls, B, index)
        kw = dict(cg2dNorm=norm, tolerance=1e-9, max_iters=400, sum_order=order, op_index=index)
        xr, _ = cg2d.cg2d_fortran(ex, slots, b, x0, launch="phases", **kw)
        runs.append((b, x0, kw, xr, torch.cuda.Stream()))
    torch.cuda.synchronize()
    print("resident: three streams", flush=True)
    out = []
    for _ in range(2):
        for b, x0, kw, _, s in runs:
            with torch.cuda.stream(s):
                out.append(cg2d.cg2d_fortran(ex, slots, b, x0, **kw))
    torch.cuda.synchronize()
    for k, (x, d) in enumerate(out):
        d.check()
        assert torch.equal(x, runs[k % 3][3]), k


GIVING_UP = [("tile", 1), ("fortran", 2), ("tile", 41), ("mixed", 3), ("mixed", 61)]


def _giving_up(problem, solve, B):
    """The call and a switch for how long its waits may take, on an exchanger (and a T plan) of its own."""
    from mit_jax_amd import _lib, cg2d, mixed
    from mit_jax_amd.exchange import Exchanger, ExchangeMaps
    _, cls, slots = problem
    ex = Exchanger(ExchangeMaps.load())
    index = np.arange(B, dtype=np.int32) % len(cls)
    b, x0, norm = _inputs(ex, cls, B, index)
    kw = dict(cg2dNorm=norm, tolerance=1e-9, max_iters=400, op_index=index)
    if solve == "mixed":
        run = lambda **o: mixed.cg2d_mixed(ex, slots, b, x0, **kw, **o)  # noqa: E731
    else:
        run = lambda **o: cg2d.cg2d_fortran(ex, slots, b, x0, sum_order=solve, **kw, **o)  # noqa: E731

    def limit(seconds):
        _lib.check(_lib.lib().mj_halo_plan_set_wait_limit(ex.plan("T", b.device).handle, seconds), "wait limit")
    return run, limit


@pytest.mark.parametrize("solve,B", GIVING_UP)
def test_resident_ends_when_its_waits_fail(problem, solve, B):
    """With a limit of 0 the first wait that is not served at once fails, in each workgroup wherever it happens to be: the
    launch ends all the same (no wave is left at a barrier that the others have passed), and the next solve with the plan
    is right."""
    run, limit = _giving_up(problem, solve, B)
    xr, _ = run(block_threads=512)
    torch.cuda.synchronize()
    for _ in range(3):
        limit(0.0)
        print(f"resident: {solve} B={B}, waits fail", flush=True)
        run()
        torch.cuda.synchronize()
        limit(20.0)
        x, d = run()
        torch.cuda.synchronize()
        assert int(d["launches"].max()) == 0
        assert torch.equal(x, xr)


@pytest.mark.parametrize("solve,B", GIVING_UP)
def test_resident_failed_waits_are_reported(problem, solve, B):
    """A solve whose waits failed says so in every member's record (the sums that it did not get read as 0, which must not
    pass for a residual), whatever the buffer held before, and the next solve does not."""
    from mit_jax_amd import _lib
    run, limit = _giving_up(problem, solve, B)
    for _ in range(3):
        limit(0.0)
        print(f"resident: {solve} B={B}, waits fail", flush=True)
        _, d = run()
        torch.cuda.synchronize()
        assert bool((d["converged"] == -2).all()), d["converged"]
        with pytest.raises(_lib.MjError, match="timed out"):
            d.check()
        limit(20.0)
        _, d = run()
        torch.cuda.synchronize()
        assert bool((d.check()["converged"] >= 0).all())
