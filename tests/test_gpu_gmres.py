"""GMRES with the orthogonalisation of a step in one kernel, against the
oracle: every vectors-per-thread setting, one work-group and many, row counts
that end inside a vector, restarts in the middle, both types, an initial
guess, and the same bits on every run."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _convtri(m):
    """Nonsymmetric tridiagonal rows, diagonally dominant."""
    lens = np.full(m, 3)
    lens[0] = lens[-1] = 2
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    rows = np.repeat(np.arange(m), lens)
    ind = np.concatenate([[0, 1], (np.arange(1, m - 1)[:, None] + np.arange(-1, 2)).ravel(), [m - 2, m - 1]])
    val = np.where(ind == rows, 3.0 + (rows % 7) * 0.1, np.where(ind < rows, -1.4, -0.8))
    return wl.CSR(m, m, ptr, ind.astype(np.int32), val)


# rows: one work-group and a remainder; 2, 4, 8, 16 vectors per thread (FP64)
ROWS = [2, 33, 2049, 100003, 262147, 524291, 1048577, 2097157]


@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("restart", [5, 30])
def test_gmres_matches_oracle(gpu, m, restart):
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = _convtri(m)
    b = wl.apply(A, wl.uniform(m, 3))
    x0 = wl.uniform(m, 4) if restart == 5 else None
    Ag, bg = K.Matrix(A), torch.tensor(b, device="cuda")
    ref = orc.solve("gmres", A, b, precond="jacobi", tol=1e-8, max_iter=14, restart=restart, x0=x0)
    runs = []
    n0 = gpu.counter("gmres_on_chip")
    for _ in range(3):
        x = torch.full_like(bg, 7.0) if x0 is None else torch.tensor(x0, device="cuda")
        it = K.Iteration(14, 1e-8)
        it.SetRestart(restart)
        it.HideMessages()
        it.SetInitGuess(x0 is None)
        code = K.Gmres(Ag, x, bg, K.JacobiPreconditioner(), it)
        runs.append((x.cpu().numpy(), it.history.copy()))
        assert (code, it.nb_iter, it.hist_len) == (ref.code, ref.nb_iter, len(ref.hist))
    assert gpu.counter("gmres_on_chip") == n0 + 3
    for x, h in runs[1:]:
        assert np.array_equal(x, runs[0][0]) and np.array_equal(h, runs[0][1])
    # sums of up to 2M terms round by ~1e-13 of the vectors' norms; residuals
    # down to 1e-4 of the first then agree to 1e-9, x, solved to 1e-8, to that
    x, h = runs[0]
    live = ref.hist > 1e-4
    assert np.all(np.abs(h - ref.hist)[live] <= 1e-9 * ref.hist[live])
    assert np.linalg.norm(x - ref.x) <= 1e-8 * np.linalg.norm(ref.x)


@pytest.mark.parametrize("m", [77, 300007, 2097157, 4194309])
def test_gmres_f32(gpu, m):
    """FP32 to 1e-3 on the preconditioned residual (the diagonal lies within
    3.0 .. 3.6): a true residual, in FP64, of at most 3e-3, twice the same bits.
    (The oracle's sequential FP32 sums lose that accuracy past 2M terms.)"""
    from seldon_amd import krylov as K
    A = _convtri(m)
    b = wl.apply(A, wl.uniform(m, 3)).astype(np.float32)
    Ag = K.Matrix(A, dtype=torch.float32)
    bg = torch.tensor(b, device="cuda")
    out = []
    n0 = gpu.counter("gmres_on_chip")
    for _ in range(2):
        x = torch.zeros_like(bg)
        it = K.Iteration(40, 1e-3)
        it.SetRestart(20)
        it.HideMessages()
        assert K.Gmres(Ag, x, bg, K.JacobiPreconditioner(), it) == 0
        assert it.nb_iter <= 12
        out.append(x.cpu().numpy())
    assert gpu.counter("gmres_on_chip") == n0 + 2
    assert np.array_equal(out[0], out[1])
    r = wl.apply(A, out[0].astype(np.float64)) - b
    assert np.linalg.norm(r) <= 3e-3 * np.linalg.norm(b)
