"""SOR / SSOR sweeps in one kernel each, bitwise against the oracle: a chain
of one-row levels, a single level, rows of more than one batch of entries, a
pattern that is not symmetric, empty rows, row counts around a wavefront, and
sweeps after sweeps on one handle."""
import numpy as np
import pytest
import torch

from seldon_amd import workloads as wl

pytestmark = pytest.mark.gpu

DT = {"d": (torch.float64, np.float64), "f": (torch.float32, np.float32)}


def _random(m, per_row, seed, empty=0):
    """Unsymmetric pattern, sorted columns, a diagonal in every kept row."""
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(m):
        if empty and i % empty == 3:
            rows.append(np.zeros(0, np.int64))
        else:
            rows.append(np.unique(np.r_[i, rng.integers(0, m, rng.integers(0, per_row))]))
    ptr = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int32)
    ind = np.concatenate(rows).astype(np.int32)
    val = rng.uniform(-1, 1, ind.size)
    val[ind == np.repeat(np.arange(m), np.diff(ptr))] += 4.0
    return wl.CSR(m, m, ptr, ind, val)


def _tridiag(m):
    return wl.aniso2d(m, 1, 2.0)


CASES = {
    "one_row": lambda: _tridiag(1),
    "chain_300": lambda: _tridiag(300),
    "diagonal_1000": lambda: wl.CSR(1000, 1000, np.arange(1001, dtype=np.int32), np.arange(1000, dtype=np.int32),
                                    np.linspace(1, 2, 1000)),
    "random_63": lambda: _random(63, 6, 1),
    "random_65_wide": lambda: _random(65, 60, 2),
    "random_2000": lambda: _random(2000, 30, 3),
    "empty_rows": lambda: _random(500, 5, 4, empty=11),
    "laplace_odd": lambda: wl.laplace2d(71, 45),
    "convdiff_odd": lambda: wl.convdiff3d(21),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("st", ["row", "array", "sym"])
@pytest.mark.parametrize("c", ["d", "f"])
def test_sor_bitwise(gpu, name, st, c):
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = CASES[name]()
    M = wl.upper(A) if st == "sym" else A
    tdt, ndt = DT[c]
    Ag = K.Matrix(M, storage=st, dtype=tdt)
    x = wl.uniform(A.m, 5).astype(ndt)
    b = wl.uniform(A.m, 6).astype(ndt)
    xg, bg = torch.tensor(x, device="cuda"), torch.tensor(b, device="cuda")
    ref = x
    with np.errstate(all="ignore"):
        for omega, iters, sweep in ((1.0, 1, 0), (1.3, 2, 2), (0.7, 1, 3), (1.1, 2, 0)):
            ref = orc.sor(M, ref, b, omega, iters, sweep, storage=st, dtype=ndt)
            K.SOR(Ag, xg, bg, omega, iters, sweep)
            assert np.array_equal(xg.cpu().numpy(), ref, equal_nan=True), (omega, iters, sweep)


def test_sor_in_a_graph(gpu):
    """A captured sweep follows X on every replay."""
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = wl.laplace2d(40, 33)
    Ag = K.Matrix(A)
    b = wl.uniform(A.m, 6)
    bg = torch.tensor(b, device="cuda")
    xg = torch.zeros_like(bg)
    K.SOR(Ag, xg, bg, 1.2, 1, 0)  # plan
    ctx = K.Context.default()
    g = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    xg.zero_()
    torch.cuda.synchronize()
    try:
        with torch.cuda.stream(stream):
            ctx.bind_stream(stream)
            with torch.cuda.graph(g, stream=stream):
                K.SOR(Ag, xg, bg, 1.2, 1, 0)
            ref = np.zeros(A.m)
            for _ in range(4):
                g.replay()
                stream.synchronize()
                ref = orc.sor(A, ref, b, 1.2, 1, 0)
                assert np.array_equal(xg.cpu().numpy(), ref)
    finally:
        torch.cuda.synchronize()
        ctx.bind_stream()


@pytest.mark.parametrize("st", ["row", "sym"])
def test_overlapping_sweeps_of_one_matrix(gpu, st):
    """Two captured sweeps of one matrix replayed side by side on two streams,
    then one of them beside a direct call on a third: each X is its own
    sequence of sweeps, whichever way they overlap."""
    from oracle import oracle as orc
    from seldon_amd import krylov as K
    A = wl.diffusion3d(40, wl.normal(40 ** 3, 4, 0.0, 0.5))
    M = wl.upper(A) if st == "sym" else A
    Ag = K.Matrix(M, storage=st)
    b = [wl.uniform(A.m, 6 + k) for k in range(3)]
    bg = [torch.tensor(v, device="cuda") for v in b]
    xg = [torch.zeros_like(v) for v in bg]
    K.SOR(Ag, xg[2], bg[2], 1.2, 1, 0)  # plan
    ref = [np.zeros(A.m), np.zeros(A.m), orc.sor(M, np.zeros(A.m), b[2], 1.2, 1, 0, storage=st)]
    ctx = K.Context.default()
    streams = [torch.cuda.Stream() for _ in range(3)]
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    torch.cuda.synchronize()

    def check():
        torch.cuda.synchronize()
        for k in range(3):
            assert np.array_equal(xg[k].cpu().numpy(), ref[k]), k

    try:
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                ctx.bind_stream(streams[k])
                with torch.cuda.graph(graphs[k], stream=streams[k]):
                    K.SOR(Ag, xg[k], bg[k], 1.2, 1, 0)
                    K.SOR(Ag, xg[k], bg[k], 0.9, 1, 2)
        ctx.bind_stream(streams[2])
        for _ in range(4):
            for k in (0, 1, 1, 0):
                with torch.cuda.stream(streams[k]):
                    graphs[k].replay()
                for o, sweep in ((1.2, 0), (0.9, 2)):
                    ref[k] = orc.sor(M, ref[k], b[k], o, 1, sweep, storage=st)
            check()
        for _ in range(4):
            with torch.cuda.stream(streams[0]):
                graphs[0].replay()
            K.SOR(Ag, xg[2], bg[2], 1.2, 1, 0)
            for o, sweep in ((1.2, 0), (0.9, 2)):
                ref[0] = orc.sor(M, ref[0], b[0], o, 1, sweep, storage=st)
            ref[2] = orc.sor(M, ref[2], b[2], 1.2, 1, 0, storage=st)
            check()
    finally:
        torch.cuda.synchronize()
        ctx.bind_stream()
