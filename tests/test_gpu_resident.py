"""Cg held on chip (stencil matrices that fit) against the oracle's Cg: one
member and many, shares with a remainder, a band wider than a member's share,
five- and seven-step rows, every rows-per-thread setting, both types, both
preconditioners, all storages, an initial guess, max_iter and breakdown."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl

pytestmark = pytest.mark.gpu

PREC = {"identity": "id", "jacobi": "jacobi"}


def _tridiag(m):
    ptr = np.concatenate([[0], np.cumsum(np.r_[2, np.full(m - 2, 3), 2])]).astype(np.int32)
    ind = np.concatenate([[max(i - 1, 0) + k for k in range(3 if 0 < i < m - 1 else 2)] for i in range(m)])
    val = np.where(ind == np.repeat(np.arange(m), np.diff(ptr)), 2.2, -1.0)
    return wl.CSR(m, m, ptr, ind.astype(np.int32), val)


MATRICES = {
    "one_member_odd": lambda: wl.laplace2d(31, 17),
    "one_member_full": lambda: wl.laplace2d(32, 32),
    "two_members_one_row_over": lambda: _tridiag(1025),
    "band_wider_than_share": lambda: wl.aniso2d(1500, 3, 5.0),
    "many_members": lambda: wl.laplace2d(181, 233),
    "four_rows_per_thread": lambda: wl.laplace2d(400, 331),
    "eight_rows_per_thread": lambda: wl.aniso2d(100, 5300, 1.0),
    "seven_steps": lambda: wl.diffusion3d(23, wl.normal(23 ** 3, 4, 0.0, 0.5)),
    "seven_steps_four_rows": lambda: wl.diffusion3d(52, wl.normal(52 ** 3, 4, 0.0, 0.5)),
}


def _solve(A, b, storage, dtype, prec, x0=None, tol=1e-10, max_iter=4000):
    from seldon_amd import krylov as K
    Ag = K.Matrix(A, storage=storage, dtype=dtype)
    bg = torch.tensor(b, device="cuda", dtype=dtype)
    x = torch.full_like(bg, 7.0) if x0 is None else torch.tensor(x0, device="cuda", dtype=dtype)
    it = K.Iteration(max_iter, tol)
    it.HideMessages()
    it.SetInitGuess(x0 is None)
    M = K.JacobiPreconditioner() if prec == "jacobi" else K.Preconditioner_Base()
    code = K.Cg(Ag, x, bg, M, it)
    return code, it, x.cpu().numpy()


def _permuted(A, order):
    """Row and column `order` of A, each row's entries in their stored order:
    the same row sums, the dots summed in another order."""
    inv = np.empty_like(order)
    inv[order] = np.arange(A.m)
    lens = np.diff(A.ptr)[order]
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    src = np.repeat(A.ptr[:-1][order] - ptr[:-1], lens) + np.arange(A.nnz)
    return wl.CSR(A.m, A.n, ptr, inv[A.ind[src]].astype(np.int32), A.val[src])


def _spread(A, b, prec, x0, ref):
    """How far the oracle's own runs differ when only the order of the dots'
    sums does: the running maximum over the history's entries, and x."""
    from oracle import oracle as orc
    h = np.zeros(len(ref.hist))
    dx = 0.0
    rng = np.random.default_rng(5)
    for order in (np.arange(A.m)[::-1].copy(), rng.permutation(A.m), rng.permutation(A.m)):
        r = orc.solve("cg", _permuted(A, order), b[order], precond=PREC[prec], tol=1e-10, max_iter=60,
                      x0=None if x0 is None else x0[order])
        k = min(len(r.hist), len(h))
        h[:k] = np.maximum(h[:k], np.abs(r.hist[:k] - ref.hist[:k]) / ref.hist[:k])
        x = np.empty(A.m)
        x[order] = r.x
        dx = max(dx, np.linalg.norm(x - ref.x) / np.linalg.norm(ref.x))
    return np.maximum.accumulate(h), dx


@pytest.mark.parametrize("name", list(MATRICES))
@pytest.mark.parametrize("prec", ["identity", "jacobi"])
def test_resident_cg_matches_oracle(gpu, name, prec):
    from oracle import oracle as orc
    A = MATRICES[name]()
    b = wl.apply(A, wl.uniform(A.m, 11))
    for storage, guess in (("row", False), ("sym", True), ("array", False)):
        M = wl.upper(A) if storage == "sym" else A
        x0 = wl.uniform(A.m, 12) if guess else None
        # 60 iterations, entry by entry: within ten times the oracle's own
        # spread under other orders of the dots' sums (never below 1e-12)
        n0 = gpu.counter("cg_on_chip")
        code, it, x = _solve(M, b, storage, torch.float64, prec, x0, max_iter=60)
        assert gpu.counter("cg_on_chip") == n0 + 1
        ref = orc.solve("cg", M, b, precond=PREC[prec], tol=1e-10, max_iter=60, x0=x0)
        assert (code, it.nb_iter, it.hist_len) == (ref.code, ref.nb_iter, len(ref.hist))
        full = orc.solve("cg", A, b, precond=PREC[prec], tol=1e-10, max_iter=60, x0=x0)
        h, dx = _spread(A, b, prec, x0, full)
        assert np.all(np.abs(it.history - ref.hist) <= np.maximum(1e-12, 10 * h) * ref.hist)
        assert np.linalg.norm(x - ref.x) <= max(1e-12, 10 * dx) * np.linalg.norm(ref.x)


@pytest.mark.parametrize("prec", ["identity", "jacobi"])
def test_resident_cg_f32(gpu, prec):
    from oracle import oracle as orc
    A = wl.laplace2d(75, 91)
    b = wl.apply(A, wl.uniform(A.m, 11))
    n0 = gpu.counter("cg_on_chip")
    code, it, x = _solve(A, b, "row", torch.float32, prec, tol=1e-4)
    assert gpu.counter("cg_on_chip") == n0 + 1
    ref = orc.solve("cg", A, b.astype(np.float32), precond=PREC[prec], tol=1e-4, max_iter=4000, dtype=np.float32)
    assert code == ref.code == 0 and abs(it.nb_iter - ref.nb_iter) <= 2
    assert np.linalg.norm(wl.apply(A, x.astype(np.float64)) - b) <= 1e-3 * np.linalg.norm(b)


def test_resident_cg_exits(gpu):
    """A zero right-hand side leaves x at 0, A p = 0 is breakdown #2, an exact
    start ends at once, and two runs give the same bits."""
    A = wl.laplace2d(40, 61)
    code, it, x = _solve(A, np.zeros(A.m), "row", torch.float64, "identity")
    assert code == 0 and it.nb_iter == 0
    Z = wl.CSR(A.m, A.n, A.ptr, A.ind, np.zeros_like(A.val))
    code, it, _ = _solve(Z, np.ones(A.m), "row", torch.float64, "identity")
    assert code == 2 and it.nb_iter == 0
    xt = wl.uniform(A.m, 3)
    code, it, x = _solve(A, wl.apply(A, xt), "row", torch.float64, "jacobi", x0=xt)
    assert code == 0 and it.nb_iter == 0 and np.array_equal(x, xt)
    b = wl.apply(A, xt)
    runs = [_solve(A, b, "row", torch.float64, "jacobi") for _ in range(2)]
    assert np.array_equal(runs[0][2], runs[1][2]) and np.array_equal(runs[0][1].history, runs[1][1].history)


def _systems(kind):
    if kind == "one_member_each":
        return [wl.aniso2d(n, n + 3, 4.0) for n in (1, 5, 31, 32, 45)]
    if kind == "uneven_teams":
        return [wl.aniso2d(n, n, e) for n, e in ((130, 3.0), (12, 1.0), (64, 50.0), (181, 1.0), (65, 9.0))]
    if kind == "more_than_the_gpu_holds":
        return [wl.aniso2d(30 + k % 101, 40 + k % 83, 1.0 + k % 7) for k in range(330)]
    return [wl.diffusion3d(g, wl.normal(g ** 3, g, 0.0, 0.5)) for g in (5, 16, 27)]


@pytest.mark.parametrize("kind", ["one_member_each", "uneven_teams", "more_than_the_gpu_holds", "three_d"])
def test_resident_batch_matches_oracle(gpu, kind):
    """Stacked stencil systems, one work-group or a team each: the oracle's
    iteration counts within one and its solutions to the solve's accuracy; an
    empty system and a zero right-hand side among them; twice the same bits."""
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    from seldon_amd.batched import cg_batched, stack
    systems = _systems(kind)
    empty = wl.CSR(0, 0, np.zeros(1, np.int32), np.zeros(0, np.int32), np.zeros(0))
    systems.insert(2, empty)
    A, row_off = stack(systems)
    b = wl.apply(A, wl.uniform(A.m, 9))
    b[row_off[1]:row_off[2]] = 0.0
    Ag = K.Matrix(A, layout="rows")
    bg = torch.tensor(b, device="cuda")
    runs = []
    n0 = gpu.counter("batch_on_chip")
    for _ in range(2):
        x = torch.full_like(bg, 7.0)
        its, codes = cg_batched(Ag, row_off, x, bg, tol=1e-8, max_iter=5000)
        runs.append((its, codes, x.cpu().numpy()))
    assert gpu.counter("batch_on_chip") == n0 + 2
    for a, c in zip(*runs):
        assert np.array_equal(a, c)
    its, codes, x = runs[0]
    for s in list(range(min(len(systems), 12))) + [len(systems) - 1]:
        sl = slice(row_off[s], row_off[s + 1])
        if s == 1:
            assert its[s] == codes[s] == 0 and np.all(x[sl] == 7.0)
            continue
        if systems[s].m == 0:
            assert its[s] == codes[s] == 0
            continue
        r = orc.solve("cg", systems[s], b[sl], tol=1e-8, max_iter=5000)
        assert codes[s] == r.code == 0 and abs(int(its[s]) - r.nb_iter) <= 1
        assert np.linalg.norm(x[sl] - r.x) <= 1e-6 * np.linalg.norm(r.x)
