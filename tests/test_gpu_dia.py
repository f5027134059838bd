"""GPU parity of the diagonal-slice SpMV copy (AUTO layouts of stencil and
banded matrices): bitwise against the oracle at slice and group edges, for
every unrolled step count and the general one, with slices whose rows lack
some offsets, for all storages, both types and both directions."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl

pytestmark = pytest.mark.gpu

DT = {"d": (torch.float64, np.float64), "f": (torch.float32, np.float32)}


def _banded(m, n, offsets, seed, drop=0.0):
    """m x n with entries at the given offsets (those inside the matrix), a
    share `drop` of them left out; rows keep increasing columns."""
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(m), len(offsets))
    cols = rows + np.tile(np.sort(np.asarray(offsets)), m)
    keep = (cols >= 0) & (cols < n) & (rng.random(rows.size) >= drop)
    rows, cols = rows[keep], cols[keep]
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=m))]).astype(np.int32)
    return wl.CSR(m, n, ptr, cols.astype(np.int32), rng.uniform(-1, 1, cols.size))


CASES = {
    "one_row": lambda: _banded(1, 1, [0], 1),
    "63_rows": lambda: _banded(63, 63, [-1, 0, 1], 2),
    "64_rows": lambda: _banded(64, 64, [-7, 0, 2, 7], 3),
    "257_rows_gaps": lambda: _banded(257, 257, [-16, -1, 0, 1, 16], 4, drop=0.1),
    "two_offsets": lambda: _banded(500, 500, [-3, 3], 5),
    "six": lambda: _banded(1000, 1000, [-40, -5, 0, 1, 5, 40], 6),
    "nine_box": lambda: _banded(33 * 31, 33 * 31, [-34, -33, -32, -1, 0, 1, 32, 33, 34], 7),
    "thirteen": lambda: _banded(3001, 3001, list(range(-6, 7)), 8, drop=0.05),
    "thirty_two": lambda: _banded(2050, 2050, list(range(-16, 16)), 9),
    "wide_offsets": lambda: _banded(70001, 70001, [-60000, -1, 0, 9, 60000], 10),
    "rect_wide": lambda: _banded(700, 900, [0, 1, 150, 200], 11),
    "rect_tall": lambda: _banded(900, 700, [-200, -150, 0], 12),
    "laplace_odd": lambda: wl.laplace2d(61, 47),
    "convdiff_odd": lambda: wl.convdiff3d(29),
}


def _same(a, b):
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("c", ["d", "f"])
@pytest.mark.parametrize("st", ["row", "sym", "array"])
def test_dia_spmv_bitwise(gpu, name, c, st):
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = CASES[name]()
    if st == "sym":
        if A.m != A.n:
            pytest.skip("RowSymSparse is square")
        M = wl.upper(A)
        if M.nnz == 0:
            pytest.skip("no stored entry")
    else:
        M = A
    tdt, ndt = DT[c]
    x = wl.uniform(A.n, 21).astype(ndt)
    x[A.n // 2] = np.inf  # reaches the rows that hold that column, no other
    y = wl.uniform(A.m, 22).astype(ndt)
    y[A.m // 3] = np.nan
    xt, yt = wl.uniform(A.m, 23).astype(ndt), wl.uniform(A.n, 24).astype(ndt)
    Ag = K.Matrix(M, storage=st, dtype=tdt)

    def dev(v):
        return torch.tensor(v, device="cuda")

    for again in (False, True):
        for al, be in ((1.0, 0.0), (-1.0, 1.0), (0.7, -0.3)):
            yg = dev(y)
            K.MltAdd(al, Ag, dev(x), be, yg)
            assert _same(yg.cpu().numpy(), orc.mltadd(ndt(al), M, x, ndt(be), y, storage=st, dtype=ndt))
            tg = dev(yt)
            K.MltAdd(al, K.SeldonTrans, Ag, dev(xt), be, tg)
            assert _same(tg.cpu().numpy(), orc.mltadd_trans(ndt(al), M, xt, ndt(be), yt, storage=st, dtype=ndt))
        yg = torch.empty(A.m, dtype=tdt, device="cuda")
        K.Mlt(Ag, dev(x), yg)
        assert _same(yg.cpu().numpy(), orc.mlt(M, x, storage=st, dtype=ndt))
        if not again:  # new values on the same pattern
            M = wl.CSR(M.m, M.n, M.ptr, M.ind, M.val * -1.5 + 0.25, M.sym)
            Ag.set_values(M.val)


@pytest.mark.parametrize("kind", ["unsorted", "duplicate", "irregular"])
def test_dia_leaves_other_matrices_alone(gpu, kind):
    """Rows out of order, a column stored twice, or rows without common
    offsets: the other layouts' sums, in stored order."""
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = _banded(400, 400, [-20, -1, 0, 1, 20], 31)
    ind = A.ind.copy()
    a = A.ptr[200]
    if kind == "unsorted":
        ind[a:a + 2] = ind[a:a + 2][::-1].copy()
    elif kind == "duplicate":
        ind[a + 1] = ind[a]
    else:
        A = wl.powerlaw(5000, 3, kmin=3, kmax=12, half_width=700)
        ind = A.ind
    M = wl.CSR(A.m, A.n, A.ptr, ind, A.val)
    x = wl.uniform(A.n, 5)
    yg = torch.empty(A.m, dtype=torch.float64, device="cuda")
    K.Mlt(K.Matrix(M), torch.tensor(x, device="cuda"), yg)
    assert _same(yg.cpu().numpy(), orc.mlt(M, x))


@pytest.mark.parametrize("method", ["cgne", "lsqr"])
@pytest.mark.parametrize("side", [512, 301])
def test_transpose_with_a_larger_grid(gpu, method, side):
    """A in the panel layout (128 work-groups at 512^2), A^T in diagonal
    slices (1024): the solver's partial sums have room for either, and the
    bits are those of a matrix that has the slices too."""
    from seldon_amd import krylov as K
    A = wl.laplace2d(side, side)
    b = wl.apply(A, wl.uniform(A.m, 3))
    bg = torch.tensor(b, device="cuda")
    runs = []
    for layout in ("panels", "auto"):
        Ag = K.Matrix(A, layout=layout)
        x = torch.zeros_like(bg)
        it = K.Iteration(30, 1e-12)
        it.HideMessages()
        code = (K.Cgne if method == "cgne" else K.Lsqr)(Ag, x, bg, K.Preconditioner_Base(), it)
        runs.append((code, it.nb_iter, it.history.copy(), x.cpu().numpy()))
    for a, c in zip(*runs):
        assert np.array_equal(a, c)
