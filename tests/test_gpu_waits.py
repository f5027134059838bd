"""What follows when a wait between work-groups runs out: a limit of zero makes
every such kernel give up and end at once, and Cg, Gmres, SOR and the batched
solve take their other way.  Also the kernels without waits by themselves, and
SOR's values exchanged through 64-bit addresses."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl
from tests.test_gpu_gmres import _convtri

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx(gpu):
    yield gpu
    for name, value in (("on_chip", 1), ("wait_us", -1), ("buffer_bytes", 2**31 - 1), ("cg_iters", 1 << 15)):
        gpu.set_option(name, value)


def _counts(ctx, *names):
    return [ctx.counter(n) for n in names]


def _cg(A, b, x0, prec, max_iter=60):
    from seldon_amd import krylov as K
    Ag, bg = A if isinstance(A, K.Matrix) else K.Matrix(A), torch.tensor(b, device="cuda")
    x = torch.full_like(bg, 7.0) if x0 is None else torch.tensor(x0, device="cuda")
    it = K.Iteration(max_iter, 1e-10)
    it.HideMessages()
    it.SetInitGuess(x0 is None)
    code = K.Cg(Ag, x, bg, K.JacobiPreconditioner() if prec == "jacobi" else K.Preconditioner_Base(), it)
    return code, it.nb_iter, it.history.copy(), x.cpu().numpy()


@pytest.mark.parametrize("prec", ["identity", "jacobi"])
@pytest.mark.parametrize("guess", [False, True])
def test_cg_starts_over(ctx, prec, guess):
    """The same bits as the launched kernels from the same start, x0 included."""
    A = wl.laplace2d(181, 233)
    b = wl.apply(A, wl.uniform(A.m, 11))
    x0 = wl.uniform(A.m, 12) if guess else None
    n0 = _counts(ctx, "cg_on_chip", "started_over")
    on_chip = _cg(A, b, x0, prec)
    assert _counts(ctx, "cg_on_chip", "started_over") == [n0[0] + 1, n0[1]]
    ctx.set_option("on_chip", 0)
    launched = _cg(A, b, x0, prec)
    assert _counts(ctx, "cg_on_chip", "started_over") == [n0[0] + 1, n0[1]]
    ctx.set_option("on_chip", 1)
    ctx.set_option("wait_us", 0)
    over = _cg(A, b, x0, prec)
    assert _counts(ctx, "cg_on_chip", "started_over") == [n0[0] + 1, n0[1] + 1]
    for a, c in zip(over, launched):
        assert np.array_equal(a, c)
    # the first residual and the first steps do not tell the two ways apart
    assert np.all(np.abs(on_chip[2][:4] - launched[2][:4]) <= 1e-12 * launched[2][:4])


def _gmres(A, b, x0, restart, max_iter=14):
    from seldon_amd import krylov as K
    Ag, bg = A if isinstance(A, K.Matrix) else K.Matrix(A), torch.tensor(b, device="cuda")
    x = torch.full_like(bg, 7.0) if x0 is None else torch.tensor(x0, device="cuda")
    it = K.Iteration(max_iter, 1e-8)
    it.SetRestart(restart)
    it.HideMessages()
    it.SetInitGuess(x0 is None)
    code = K.Gmres(Ag, x, bg, K.JacobiPreconditioner(), it)
    return code, it.nb_iter, it.history.copy(), x.cpu().numpy()


@pytest.mark.parametrize("m", [2, 33, 2049, 100003, 262147])
@pytest.mark.parametrize("restart", [5, 30])
def test_gmres_a_kernel_per_pass(ctx, m, restart):
    """Without the kernel that waits: against the oracle."""
    from oracle import oracle as orc
    A = _convtri(m)
    b = wl.apply(A, wl.uniform(m, 3))
    x0 = wl.uniform(m, 4) if restart == 5 else None
    n0 = _counts(ctx, "gmres_on_chip")
    ctx.set_option("on_chip", 0)
    code, nb, h, x = _gmres(A, b, x0, restart)
    assert _counts(ctx, "gmres_on_chip") == n0
    ref = orc.solve("gmres", A, b, precond="jacobi", tol=1e-8, max_iter=14, restart=restart, x0=x0)
    assert (code, nb, len(h)) == (ref.code, ref.nb_iter, len(ref.hist))
    # as for the kernel that waits: sums of at most 2M terms, residuals down
    # to 1e-4 of the first to 1e-9
    live = ref.hist > 1e-4
    assert np.all(np.abs(h - ref.hist)[live] <= 1e-9 * ref.hist[live])
    assert np.linalg.norm(x - ref.x) <= 1e-8 * np.linalg.norm(ref.x)


@pytest.mark.parametrize("guess", [False, True])
def test_gmres_starts_over(ctx, guess):
    m = 100003
    A = _convtri(m)
    b = wl.apply(A, wl.uniform(m, 3))
    x0 = wl.uniform(m, 4) if guess else None
    n0 = _counts(ctx, "gmres_on_chip", "started_over")
    _gmres(A, b, x0, 5)
    assert _counts(ctx, "gmres_on_chip", "started_over") == [n0[0] + 1, n0[1]]
    ctx.set_option("on_chip", 0)
    launched = _gmres(A, b, x0, 5)
    ctx.set_option("on_chip", 1)
    ctx.set_option("wait_us", 0)
    over = _gmres(A, b, x0, 5)
    assert _counts(ctx, "gmres_on_chip", "started_over") == [n0[0] + 1, n0[1] + 1]
    for a, c in zip(over, launched):
        assert np.array_equal(a, c)


@pytest.mark.parametrize("st", ["row", "array", "sym"])
@pytest.mark.parametrize("c", ["d", "f"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("rescue", [False, True])
def test_sor_rescue_and_wide_words(ctx, st, c, wide, rescue):
    """Bitwise the oracle's sweeps, by one wavefront and through 64-bit
    addresses; the next sweeps on the handle are as ever."""
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = wl.laplace2d(71, 45)
    M = wl.upper(A) if st == "sym" else A
    tdt, ndt = (torch.float64, np.float64) if c == "d" else (torch.float32, np.float32)
    Ag = K.Matrix(M, storage=st, dtype=tdt)
    b = wl.uniform(A.m, 6).astype(ndt)
    ref = wl.uniform(A.m, 5).astype(ndt)
    xg, bg = torch.tensor(ref, device="cuda"), torch.tensor(b, device="cuda")
    ctx.set_option("buffer_bytes", 0 if wide else 2**31 - 1)
    for wait, omega, iters, sweep in ((0, 1.3, 2, 0), (-1, 0.9, 1, 0), (0, 1.0, 1, 3)):
        ctx.set_option("wait_us", wait if rescue else -1)
        n0 = ctx.counter("sor_rescued")
        K.SOR(Ag, xg, bg, omega, iters, sweep)
        ref = orc.sor(M, ref, b, omega, iters, sweep, storage=st, dtype=ndt)
        assert np.array_equal(xg.cpu().numpy(), ref), (wait, omega)
        sweeps = iters * (2 if sweep == 0 else 1)
        assert ctx.counter("sor_rescued") - n0 == (sweeps if rescue and wait == 0 else 0)


@pytest.mark.parametrize("kind", ["stencil", "permuted"])
def test_batched_stall_is_an_error(ctx, kind):
    """A team whose members wait too long: the call says so, and the next one
    solves; a batch of one-member teams waits for nobody."""
    from seldon_amd import _lib as L
    from seldon_amd import krylov as K
    from seldon_amd.batched import cg_batched, stack
    from tests.test_gpu_batched import _as
    A, row_off = stack([_as(kind, wl.aniso2d(200, 200, 3.0), 1)])
    S, s_off = stack([wl.aniso2d(9, 9, 1.0), wl.aniso2d(12, 7, 1.0)])
    Ag, Sg = K.Matrix(A, layout="rows"), K.Matrix(S, layout="rows")
    bg, sg = torch.ones(A.m, dtype=torch.float64, device="cuda"), torch.ones(S.m, dtype=torch.float64, device="cuda")
    n0 = ctx.counter("batch_on_chip")
    ctx.set_option("wait_us", 0)
    with pytest.raises(L.ShkError, match="waited too long"):
        cg_batched(Ag, row_off, torch.zeros_like(bg), bg, max_iter=50)
    assert np.all(cg_batched(Sg, s_off, torch.zeros_like(sg), sg)[1] == 0)
    ctx.set_option("wait_us", -1)
    assert np.all(cg_batched(Ag, row_off, torch.zeros_like(bg), bg)[1] == 0)
    assert ctx.counter("batch_on_chip") == n0 + (2 if kind == "stencil" else 1)


def test_options_refuse_what_they_cannot_be(ctx):
    from seldon_amd import _lib as L
    for name, bad in (("on_chip", 2), ("wait_us", -2), ("buffer_bytes", 2**31), ("cg_iters", 0)):
        with pytest.raises(L.ShkError):
            ctx.set_option(name, bad)
    lib = L.load()
    assert lib.shk_ctx_set_option(ctx.h, 99, 0) == -1 and lib.shk_ctx_counter(ctx.h, 99, None) == -1


@pytest.mark.parametrize("name", ["one_member_odd", "band_wider_than_share", "four_rows_per_thread",
                                  "eight_rows_per_thread", "seven_steps", "seven_steps_four_rows"])
@pytest.mark.parametrize("prec", ["identity", "jacobi"])
def test_cg_left_and_carried_on(ctx, name, prec):
    """Launches of 1, 7 and 64 iterations give the bits of one launch."""
    from tests.test_gpu_resident import MATRICES, _solve
    A = MATRICES[name]()
    b = wl.apply(A, wl.uniform(A.m, 11))
    for dtype, x0 in ((torch.float64, None), (torch.float32, wl.uniform(A.m, 12))):
        runs = []
        for iters in (1 << 15, 1, 7, 64):
            ctx.set_option("cg_iters", iters)
            n0 = ctx.counter("cg_on_chip")
            code, it, x = _solve(A, b, "row", dtype, prec, x0, max_iter=130)
            assert ctx.counter("cg_on_chip") == n0 + 1
            runs.append((code, it.nb_iter, it.history.copy(), x))
        for run in runs[1:]:
            for a, c in zip(run, runs[0]):
                assert np.array_equal(a, c), (dtype, iters)


@pytest.mark.parametrize("side", [128, 1000])
def test_cg_noalloc_left_and_carried_on(ctx, side):
    """In the fixed work memory too, and in one launch where that has no room
    for what a solve is left with (1M FP64 rows): the same bits."""
    from seldon_amd import _lib as L
    from tests.test_zz_no_alloc import _run
    A, b, _ = wl.cg_laplace(side)
    n0 = ctx.counter("cg_on_chip")
    ref = _run(L.load().shk_cg, A, b, torch.float64, False, None)
    ctx.set_option("cg_iters", 50)
    got = _run(L.load().shk_cg_noalloc, A, b, torch.float64, False, None)
    assert ctx.counter("cg_on_chip") == n0 + 2
    for a, c in zip(got, ref):
        assert np.array_equal(a, c)


def test_long_cg_gives_way(ctx):
    """A solve that fills the GPU for a long time is left now and then: a
    short one of another thread, which needs its place, ends long before it."""
    import threading
    import time

    from seldon_amd import krylov as K
    A, S = wl.laplace2d(1000, 490), wl.laplace2d(128, 128)  # 240 and 16 work-groups
    ctxs = [K.Context(0) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    for c, s in zip(ctxs, streams):
        c.bind_stream(s)
    ctxs[0].set_option("cg_iters", 2048)
    Ag, Sg = K.Matrix(A, ctx=ctxs[0]), K.Matrix(S, ctx=ctxs[1])
    ab = torch.full((A.m,), float("nan"), dtype=torch.float64, device="cuda")
    sb = torch.tensor(wl.uniform(S.m, 2), device="cuda")
    ax, sx = torch.zeros_like(ab), torch.zeros_like(sb)

    def solve(Mg, x, b, max_iter):
        it = K.Iteration(max_iter, 1e-6)
        it.HideMessages()
        it.SetInitGuess(True)
        return K.Cg(Mg, x, b, K.Preconditioner_Base(), it)

    solve(Sg, sx, sb, 2000)
    torch.cuda.synchronize()
    spans = []

    def run():
        t = time.perf_counter()
        solve(Ag, ax, ab, 200000)  # about a second
        spans.append((t, time.perf_counter()))

    th = threading.Thread(target=run)
    th.start()
    time.sleep(0.1)
    for _ in range(3):
        solve(Sg, sx, sb, 2000)
    ended = time.perf_counter()
    th.join()
    torch.cuda.synchronize()
    print("long solve", spans[0][1] - spans[0][0], "short ones ended before it by", spans[0][1] - ended, flush=True)
    assert spans[0][1] - spans[0][0] > 0.5
    assert ended < spans[0][1] - 0.2
    assert ctxs[0].counter("started_over") == ctxs[1].counter("started_over") == 0
    for c in ctxs:
        c.synchronize()
        c.bind_stream()


def test_a_wait_that_ran_out_is_remembered(ctx):
    """One solve pays for a GPU that others use; those after it, the inner
    solves of a refinement too, do not try again at once.  Setting an option
    ends that."""
    from seldon_amd import krylov as K
    A = wl.laplace2d(181, 233)
    b = wl.apply(A, wl.uniform(A.m, 11))
    n0 = _counts(ctx, "cg_on_chip", "gmres_on_chip", "started_over")
    ctx.set_option("wait_us", 0)
    first, second = _cg(A, b, None, "jacobi"), _cg(A, b, None, "jacobi")
    C = _convtri(100003)
    _gmres(C, wl.apply(C, wl.uniform(C.m, 3)), None, 5)
    assert _counts(ctx, "cg_on_chip", "gmres_on_chip", "started_over") == [n0[0], n0[1], n0[2] + 1]
    for a, c in zip(first, second):
        assert np.array_equal(a, c)
    ctx.set_option("wait_us", 0)
    A64, A32 = K.Matrix(C), K.Matrix(C, dtype=torch.float32)
    bg = torch.tensor(wl.apply(C, wl.uniform(C.m, 3)), device="cuda")
    assert K.solve_ir(A64, A32, torch.zeros_like(bg), bg, K.JacobiPreconditioner(), tol=1e-10)["code"] == 0
    assert _counts(ctx, "cg_on_chip", "gmres_on_chip", "started_over") == [n0[0], n0[1], n0[2] + 2]
    ctx.set_option("wait_us", -1)
    _cg(A, b, None, "jacobi")
    assert _counts(ctx, "cg_on_chip", "started_over") == [n0[0] + 1, n0[2] + 2]


@pytest.mark.parametrize("method", ["cg", "gmres"])
def test_contexts_of_two_threads_run_side_by_side(ctx, method):
    """A long Cg solve of 64 work-groups in one thread does not keep short
    solves of another from running and ending meanwhile."""
    import threading
    import time

    from seldon_amd import krylov as K
    A, S = wl.laplace2d(256, 256), wl.laplace2d(64, 64)
    ctxs = [K.Context(0) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    for c, s in zip(ctxs, streams):
        c.bind_stream(s)
    Ag, Sg = K.Matrix(A, ctx=ctxs[0]), K.Matrix(S, ctx=ctxs[1])
    ab = torch.full((A.m,), float("nan"), dtype=torch.float64, device="cuda")  # never converges
    sb = torch.tensor(wl.uniform(S.m, 2), device="cuda")
    ax, sx = torch.zeros_like(ab), torch.zeros_like(sb)

    def solve(Mg, x, b, tol, max_iter):
        it = K.Iteration(max_iter, tol)
        it.HideMessages()
        it.SetRestart(20)
        it.SetInitGuess(True)
        f = K.Gmres if method == "gmres" and Mg is Sg else K.Cg
        return f(Mg, x, b, K.Preconditioner_Base(), it)

    solve(Sg, sx, sb, 1e-6, 2000)
    torch.cuda.synchronize()
    spans = []

    def run():
        t = time.perf_counter()
        solve(Ag, ax, ab, 1e-10, 300000)  # about a second
        spans.append((t, time.perf_counter()))

    th = threading.Thread(target=run)
    th.start()
    time.sleep(0.1)
    for _ in range(3):
        solve(Sg, sx, sb, 1e-6, 2000)
    ended = time.perf_counter()
    th.join()
    torch.cuda.synchronize()
    print("long solve", spans[0][1] - spans[0][0], "short ones ended before it by", spans[0][1] - ended, flush=True)
    assert spans[0][1] - spans[0][0] > 0.4
    assert ended < spans[0][1] - 0.1
    for c in ctxs:
        c.synchronize()
        c.bind_stream()
