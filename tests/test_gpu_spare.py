"""What a call can do without: with no memory to spare for it, matrices keep
their layout without a copy, and solves, batches and assemblies take the way
that needs less, with the results they have there."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl
from tests.test_gpu_gmres import _convtri
from tests.test_gpu_waits import _cg, _counts, _gmres

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx(gpu):
    yield gpu
    for name, value in (("on_chip", 1), ("spare_bytes", 2**63 - 1)):
        gpu.set_option(name, value)


# the steps' table of the 40^3 matrix takes 112,000 bytes, the positions
# 1.8 MB, the values 3.6 MB (1.8 in FP32): what is missing is all, all but the
# flags, the positions, or the values
@pytest.mark.parametrize("spare", [0, 4096, 200000, 2000000])
@pytest.mark.parametrize("st", ["row", "array", "sym"])
@pytest.mark.parametrize("c", ["d", "f"])
def test_matrix_without_its_copy(ctx, spare, st, c):
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    tdt, ndt = (torch.float64, np.float64) if c == "d" else (torch.float32, np.float32)
    A = wl.diffusion3d(40, wl.normal(40 ** 3, 4, 0.0, 0.5))
    M = wl.upper(A) if st == "sym" else A
    ctx.set_option("spare_bytes", spare)
    Ag = K.Matrix(M, storage=st, dtype=tdt)
    ctx.set_option("spare_bytes", 2**63 - 1)
    x = wl.uniform(A.m, 3).astype(ndt)
    xg = torch.tensor(x, device="cuda")
    y = torch.empty_like(xg)
    K.Mlt(Ag, xg, y)
    want = orc.mlt(M, x, storage=st, dtype=ndt)
    assert np.array_equal(y.cpu().numpy(), want)
    n0 = ctx.counter("cg_on_chip")
    it = K.Iteration(5, 1e-10)
    it.HideMessages()
    K.Cg(Ag, torch.zeros_like(xg), xg, K.Preconditioner_Base(), it)
    kept = c == "f" and spare == 2000000 and st != "sym"
    assert ctx.counter("cg_on_chip") - n0 == int(kept)


def test_large_stencil_without_its_copy(ctx):
    """The layout it had before there was a copy, and the same product."""
    from seldon_amd import krylov as K
    A = wl.convdiff3d(128)
    xg = torch.tensor(wl.uniform(A.m, 3), device="cuda")
    ys = []
    for spare, layout in ((2**63 - 1, "rows"), (1 << 20, "sliced")):
        ctx.set_option("spare_bytes", spare)
        Ag = K.Matrix(A)
        assert Ag.layout == layout
        ys.append(torch.empty_like(xg))
        K.Mlt(Ag, xg, ys[-1])
    assert torch.equal(*ys)


def test_solves_without_more_workspace(ctx):
    """Gmres, and a Cg long enough to be left, as without kernels that wait."""
    from seldon_amd import krylov as K
    A, C = wl.laplace2d(181, 233), _convtri(100003)
    ab, cb = wl.apply(A, wl.uniform(A.m, 11)), wl.apply(C, wl.uniform(C.m, 3))
    ctx.set_option("cg_iters", 10)

    def solves():
        return _cg(A, ab, None, "jacobi") + _gmres(C, cb, wl.uniform(C.m, 4), 5)

    try:
        ctx.set_option("on_chip", 0)
        want = solves()
        ctx.set_option("on_chip", 1)
        n0 = _counts(ctx, "cg_on_chip", "gmres_on_chip", "started_over")
        # the matrices keep their copies: only what the solves ask for is short
        Ag, Cg = K.Matrix(A), K.Matrix(C)
        ctx.set_option("spare_bytes", 1000)
        got = _cg(Ag, ab, None, "jacobi") + _gmres(Cg, cb, wl.uniform(C.m, 4), 5)
        assert _counts(ctx, "cg_on_chip", "gmres_on_chip", "started_over") == n0
    finally:
        ctx.set_option("cg_iters", 1 << 15)
    for a, c in zip(got, want):
        assert np.array_equal(a, c)


def test_batch_and_assembly_without_more_workspace(ctx):
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    from seldon_amd.batched import cg_batched, stack
    from tests.test_gpu_assembly import _run
    systems = [wl.aniso2d(n, n + 3, 4.0) for n in (5, 31, 45)]
    A, row_off = stack(systems)
    b = wl.apply(A, wl.uniform(A.m, 9))
    Ag, bg = K.Matrix(A, layout="rows"), torch.tensor(b, device="cuda")
    rng = np.random.default_rng(3)
    row, col = rng.integers(0, 500, 30000).astype(np.int32), rng.integers(0, 700, 30000).astype(np.int32)
    val = rng.standard_normal(30000)
    want = _run(row, col, val, 0, 0, 0, torch.float64)
    ctx.set_option("spare_bytes", 1000)
    n0 = ctx.counter("batch_on_chip")
    x = torch.zeros_like(bg)
    its, codes = cg_batched(Ag, row_off, x, bg, tol=1e-8, max_iter=5000)
    assert ctx.counter("batch_on_chip") == n0
    for s, S in enumerate(systems):
        sl = slice(row_off[s], row_off[s + 1])
        r = orc.solve("cg", S, b[sl], tol=1e-8, max_iter=5000)
        assert codes[s] == r.code == 0 and abs(int(its[s]) - r.nb_iter) <= 1
        assert np.linalg.norm(x.cpu().numpy()[sl] - r.x) <= 1e-6 * np.linalg.norm(r.x)
    got = _run(row, col, val, 0, 0, 0, torch.float64)
    assert got[:2] == want[:2]
    for a, c in zip(got[2:], want[2:]):
        assert torch.equal(a, c)
