"""CPU tests that pin the oracle (oracle/seldon_oracle.c).

Pins, each chosen so that a plausible slip (a dropped term, a wrong sign or
index, a transposed operand, a wrong stopping count) fails one of them:
  * the golden fixtures written by the real Seldon build (tests/golden):
    SpMV outputs, plain and with SeldonTrans (on a rectangular matrix), on
    three storages x two precisions x six (alpha, beta), bitwise; the CSR
    that ConvertMatrix_from_Coordinates assembles (duplicates, 1-based
    input, empty rows, no entries), bitwise; Cg / BiCgStab residual histories, iteration counts, error codes
    and solutions, bitwise against the generic-template build; Gmres against
    the MKL-linked build (the only one that compiles) within its recorded
    spread, and bitwise against its own recorded history;
  * live runs of oracle/_ref (real Seldon) on fresh random inputs when that
    build is present;
  * closed forms and textbook special cases: Laplacian eigenpairs, A = I,
    diagonal A with k distinct eigenvalues, the Givens rotation, upper
    triangular solves against numpy, small dense solves.
"""
import hashlib
import os
import tempfile

import numpy as np
import pytest

from oracle import oracle as orc
from seldon_amd import workloads as wl
from tests.conftest import GOLDEN, load_fixture
from tests.golden.make_golden import SOLVES, build_case, csr_digest

SOLVE_FIXTURES = sorted(f for f in os.listdir(GOLDEN) if f.startswith("solve_"))


def _solve(spec):
    A, b = build_case(spec)
    x0 = None if spec.get("x0seed") is None else wl.uniform(A.m, spec["x0seed"])
    return A, orc.solve(spec["method"], A, b, precond=spec["precond"], tol=spec["tol"],
                        max_iter=spec["max_iter"], restart=spec.get("restart", 10), x0=x0,
                        storage=spec.get("storage"), dtype=np.dtype(spec.get("dtype", "float64")))


def _exp_as_in_fixture(spec):
    """Whether this host can make the fixture's matrix bit for bit: the
    diffusion matrix's cell values are numpy's exp, which is numpy's own code
    on CPUs with AVX-512 (where the fixture was made) and the C library's on
    others, some last bits apart."""
    if spec["kind"] != "diffusion3d":
        return True
    assert (spec["grid"], spec["seed"]) == (16, 31)
    kappa = np.exp(wl.normal(16 ** 3, 31, 0.0, 0.5))
    return hashlib.sha256(kappa.tobytes()).hexdigest().startswith("67b8a50f9af9b733")


def test_fixture_specs_match_generator():
    left = []
    for f in SOLVE_FIXTURES:
        fx = load_fixture(f)
        if not _exp_as_in_fixture(fx["spec"]):
            left.append(f)
            continue
        A, _ = build_case(fx["spec"])
        assert csr_digest(A) == str(fx["digest"]), f
    if left:
        pytest.skip(f"numpy's exp on this CPU is not the fixture's: {left}; the others match")


@pytest.mark.parametrize("fname", SOLVE_FIXTURES)
def test_oracle_solver_matches_seldon_fixture(fname):
    fx = load_fixture(fname)
    spec = fx["spec"]
    A, r = _solve(spec)
    assert r.code == int(fx["code"])
    assert r.nb_iter == int(fx["nb_iter"])
    if str(fx["build"]) == "generic":
        # Seldon's generic templates (float vectors with Iteration<double>
        # for the FP32 family): the restatement is bitwise equal
        if not np.array_equal(r.hist, fx["hist"]) and not _exp_as_in_fixture(spec):
            pytest.skip("numpy's exp on this CPU is not the fixture's")
        assert np.array_equal(r.hist, fx["hist"])
        assert np.array_equal(r.hist_it, fx["hist_it"])
        if "x" in fx:
            assert np.array_equal(r.x, fx["x"])
        elif not spec.get("zero_rhs"):
            assert np.sum(r.x) == float(fx["x_sum"])
            assert np.array_equal(r.x[:16], fx["x_head"])
    elif str(fx["build"]) == "blas-float-iteration":
        # FP32 Gmres: Seldon's float Gmres (Iteration<float>: float
        # Hessenberg and rotations) against the oracle's, which keeps them in
        # double.  Same iteration count and Finished() sequence; histories
        # within FP32 rounding (a few hundred float ulps relative to the
        # tolerance, since both end near it); the oracle's own history is
        # pinned bitwise
        assert np.array_equal(r.hist_it, fx["hist_it"])
        assert np.array_equal(r.hist, fx["other_hist"])
        rel = np.abs(r.hist - fx["hist"]) / np.abs(fx["hist"])
        assert np.all(rel <= 2e-2), rel.max()
        assert np.all(rel[:5] <= 1e-5), rel[:5]
        xs = np.linalg.norm(fx["x"].astype(np.float64))
        assert np.linalg.norm(r.x.astype(np.float64) - fx["x"]) <= 10 * spec["tol"] * xs * 100
    else:
        # Gmres exists only in the MKL-linked build: same iteration count and
        # Finished() sequence, history within the recorded spread, and the
        # oracle's own history is pinned bitwise
        assert np.array_equal(r.hist_it, fx["hist_it"])
        assert np.array_equal(r.hist, fx["other_hist"])
        rel = np.abs(r.hist - fx["hist"]) / np.abs(fx["hist"])
        assert np.all(rel <= np.maximum(fx["spread"], 0) + 1e-300)
        assert abs(np.sum(r.x) - float(fx["x_sum"])) <= 1e-9 * max(1.0, abs(float(fx["x_sum"])))


@pytest.mark.parametrize("st", ["row", "sym", "array"])
@pytest.mark.parametrize("c", ["d", "f"])
def test_oracle_spmv_matches_seldon_fixture(st, c):
    fx = load_fixture("spmv_powerlaw300.npz")
    sp = fx["spec"]
    dt = np.float64 if c == "d" else np.float32
    A = wl.powerlaw(sp["n"], sp["seed"], kmin=sp["kmin"], kmax=sp["kmax"], half_width=sp["half_width"])
    assert csr_digest(A) == str(fx["digest"])
    M = wl.upper(A) if st == "sym" else A
    x = wl.uniform(A.m, sp["xseed"]).astype(dt)
    y = wl.uniform(A.m, sp["yseed"])
    y[sp["nan_at"]] = np.nan
    y = y.astype(dt)
    for k, (al, be) in enumerate(fx["alpha_beta"]):
        got = orc.mltadd(dt(al), M, x, dt(be), y, storage=st, dtype=dt)
        assert np.array_equal(got, fx[f"{st}_{c}_{k}"], equal_nan=True), (st, c, al, be)
    assert np.array_equal(orc.mlt(M, x, storage=st, dtype=dt), fx[f"{st}_{c}_mlt"])


def test_fixture_check_has_teeth():
    """A transposed operand or the wrong storage semantics must not pass."""
    fx = load_fixture("spmv_powerlaw300.npz")
    sp = fx["spec"]
    A = wl.powerlaw(sp["n"], sp["seed"], kmin=sp["kmin"], kmax=sp["kmax"], half_width=sp["half_width"])
    At = A.to_scipy().T.tocsr()
    T = wl.CSR(A.m, A.n, At.indptr.astype(np.int32), At.indices.astype(np.int32), At.data.copy())
    x = wl.uniform(A.m, sp["xseed"])
    assert not np.array_equal(orc.mlt(T, x), fx["row_d_mlt"])
    y = wl.uniform(A.m, sp["yseed"])
    y[sp["nan_at"]] = np.nan
    # RowSparse keeps beta*NaN, ArrayRowSparse zero-fills on beta == 0
    row = orc.mltadd(1.0, A, x, 0.0, y, storage="row")
    arr = orc.mltadd(1.0, A, x, 0.0, y, storage="array")
    assert np.isnan(row[sp["nan_at"]]) and not np.isnan(arr[sp["nan_at"]])


@pytest.mark.skipif(not orc.ref_available("generic"), reason="oracle/_ref not built (no reference tree)")
def test_oracle_bitwise_vs_live_seldon():
    rng = np.random.default_rng(7)
    with tempfile.TemporaryDirectory() as tmp:
        for seed in range(3):
            A = wl.powerlaw(2000 + 500 * seed, 100 + seed, kmin=1, kmax=60, half_width=300)
            x = rng.standard_normal(A.m)
            y = rng.standard_normal(A.m)
            for st, M in (("row", A), ("sym", wl.upper(A)), ("array", A)):
                orc.write_seldon_csr(f"{tmp}/A.bin", M)
                orc.write_seldon_vec(f"{tmp}/x.bin", x)
                orc.write_seldon_vec(f"{tmp}/y.bin", y)
                orc.run_ref(["spmv", st, "d", f"{tmp}/A.bin", f"{tmp}/x.bin", f"{tmp}/y.bin", "0.7", "-0.2",
                             f"{tmp}/o.bin"])
                ref = orc.read_seldon_vec(f"{tmp}/o.bin")
                assert np.array_equal(ref, orc.mltadd(0.7, M, x, -0.2, y, storage=st))
        A, b, _ = wl.cg_laplace(48)
        orc.write_seldon_csr(f"{tmp}/A.bin", A)
        orc.write_seldon_vec(f"{tmp}/b.bin", b)
        for meth, prec in (("cg", "jacobi"), ("bicgstab", "id")):
            out = orc.run_ref(["solve", meth, "row", prec, f"{tmp}/A.bin", f"{tmp}/b.bin", "-", 1e-9, 1000, 10,
                               f"{tmp}/x.bin"])
            h, its, code, nb = orc.parse_ref_history(out)
            r = orc.solve(meth, A, b, precond=prec, tol=1e-9, max_iter=1000)
            assert np.array_equal(h, r.hist) and code == r.code and nb == r.nb_iter
            assert np.array_equal(orc.read_seldon_vec(f"{tmp}/x.bin"), r.x)


def _spmvt_case(fx, dt):
    sp = fx["spec"]
    A = wl.powerlaw(sp["n"], sp["seed"], kmin=sp["kmin"], kmax=sp["kmax"], half_width=sp["half_width"])
    R = wl.first_columns(A, sp["ncols"])
    x = wl.uniform(sp["n"], sp["xseed"]).astype(dt)
    yr = wl.uniform(sp["ncols"], sp["yseed_rect"])
    ys = wl.uniform(sp["n"], sp["yseed_sym"])
    yr[sp["nan_at"]] = np.nan
    ys[sp["nan_at"]] = np.nan
    return A, R, x, yr.astype(dt), ys.astype(dt)


@pytest.mark.parametrize("st", ["row", "sym", "array"])
@pytest.mark.parametrize("c", ["d", "f"])
def test_oracle_spmv_trans_matches_seldon_fixture(st, c):
    """MltAdd(alpha, SeldonTrans, ...) and Mlt(SeldonTrans, ...) of the real
    Seldon build, on a 300 x 220 matrix (and a symmetric one), bitwise."""
    fx = load_fixture("spmvt_rect300x220.npz")
    dt = np.float64 if c == "d" else np.float32
    A, R, x, yr, ys = _spmvt_case(fx, dt)
    assert csr_digest(R) == str(fx["digest"])
    M, y = (wl.upper(A), ys) if st == "sym" else (R, yr)
    for k, (al, be) in enumerate(fx["alpha_beta"]):
        got = orc.mltadd_trans(dt(al), M, x, dt(be), y, storage=st, dtype=dt)
        assert np.array_equal(got, fx[f"{st}_{c}_{k}"], equal_nan=True), (st, c, al, be)
    assert np.array_equal(orc.mlt_trans(M, x, storage=st, dtype=dt), fx[f"{st}_{c}_mlt"])


def test_spmv_trans_fixture_has_teeth():
    """The transposed product is A^T x (scipy agrees to rounding), it is not
    the plain product of the transpose's storage order with other sums, and
    RowSparse keeps beta*NaN where ArrayRowSparse zero-fills."""
    fx = load_fixture("spmvt_rect300x220.npz")
    A, R, x, yr, _ = _spmvt_case(fx, np.float64)
    ref = R.to_scipy().T @ x
    got = orc.mlt_trans(R, x, storage="row")
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
    # the same sums in a different order (a column-sorted CSR of R^T summed
    # per row with a temp, as the plain RowSparse product would) round
    # differently somewhere
    Rt = R.to_scipy().T.tocsr()
    T = wl.CSR(R.n, R.m, Rt.indptr.astype(np.int32), Rt.indices.astype(np.int32), Rt.data.copy())
    plain = orc.mltadd(0.3, T, x, -1.0, yr, storage="row")
    assert not np.array_equal(plain, fx["row_d_1"], equal_nan=True)
    row = orc.mltadd_trans(1.0, R, x, 0.0, yr, storage="row")
    arr = orc.mltadd_trans(1.0, R, x, 0.0, yr, storage="array")
    nan_at = fx["spec"]["nan_at"]
    assert np.isnan(row[nan_at]) and not np.isnan(arr[nan_at])
    # RowSymSparse: MltAdd(.., SeldonTrans, ..) is the plain product, while
    # Mlt(SeldonTrans, ..) sums each full row in column order -- other sums
    U = wl.upper(A)
    assert np.array_equal(orc.mltadd_trans(1.0, U, x, 0.0, np.zeros(A.m), storage="sym"),
                          orc.mltadd(1.0, U, x, 0.0, np.zeros(A.m), storage="sym"))
    assert not np.array_equal(orc.mlt_trans(U, x, storage="sym"), orc.mlt(U, x, storage="sym"))


@pytest.mark.skipif(not orc.ref_available("generic"), reason="oracle/_ref not built (no reference tree)")
def test_oracle_trans_bitwise_vs_live_seldon():
    rng = np.random.default_rng(8)
    with tempfile.TemporaryDirectory() as tmp:
        for seed in range(2):
            A = wl.powerlaw(1500 + 700 * seed, 50 + seed, kmin=1, kmax=80, half_width=400)
            R = wl.first_columns(A, A.m - 300)
            x = rng.standard_normal(A.m)
            for st, M in (("row", R), ("array", R), ("sym", wl.upper(A))):
                y = rng.standard_normal(A.m if st == "sym" else R.n)
                orc.write_seldon_csr(f"{tmp}/A.bin", M)
                orc.write_seldon_vec(f"{tmp}/x.bin", x)
                orc.write_seldon_vec(f"{tmp}/y.bin", y)
                orc.run_ref(["spmvt", st, "d", f"{tmp}/A.bin", f"{tmp}/x.bin", f"{tmp}/y.bin", "-1.3", "0.6",
                             f"{tmp}/o.bin"])
                ref = orc.read_seldon_vec(f"{tmp}/o.bin")
                assert np.array_equal(ref, orc.mltadd_trans(-1.3, M, x, 0.6, y, storage=st))
                orc.run_ref(["mltt", st, "d", f"{tmp}/A.bin", f"{tmp}/x.bin", f"{tmp}/o.bin"])
                ref = orc.read_seldon_vec(f"{tmp}/o.bin")
                assert np.array_equal(ref, orc.mlt_trans(M, x, storage=st))


@pytest.mark.parametrize("name", ["dup", "gaps", "none"])
@pytest.mark.parametrize("c", ["d", "f"])
def test_oracle_coo_to_csr_matches_seldon_fixture(name, c):
    """ConvertMatrix_from_Coordinates (RowSparse) of the real Seldon build:
    duplicates kept in input order, 1-based input, empty rows, m / n from
    the prior size, no entries at all (m = 1 then, from GetNormInf)."""
    from tests.golden.make_golden import coo_case
    fx = load_fixture("coo_to_csr.npz")
    dt = np.float64 if c == "d" else np.float32
    row, col, val, index, m_min, n_min = coo_case(name)
    m, n, ptr, ind, out = orc.coo_to_csr(row, col, val.astype(dt), index, m_min, n_min, dtype=dt)
    assert [m, n] == list(fx[f"{name}_{c}_mn"])
    assert np.array_equal(ptr, fx[f"{name}_{c}_ptr"])
    assert np.array_equal(ind, fx[f"{name}_{c}_ind"])
    assert np.array_equal(out, fx[f"{name}_{c}_val"])


def test_oracle_coo_to_csr_is_a_stable_sort():
    """The restated MergeSort (two passes) equals numpy's stable lexsort by
    (row, column); an unstable order of the duplicates must not pass."""
    from tests.golden.make_golden import coo_case
    row, col, val, index, _, _ = coo_case("dup")
    m, n, ptr, ind, out = orc.coo_to_csr(row, col, val, index)
    o = np.lexsort((col, row))
    assert np.array_equal(ind, col[o] - index) and np.array_equal(out, val[o])
    assert np.array_equal(ptr, np.concatenate([[0], np.cumsum(np.bincount(row - index, minlength=m))]))
    rev = np.lexsort((-np.arange(len(row)), col, row))  # duplicates reversed
    assert not np.array_equal(out, val[rev])


@pytest.mark.skipif(not orc.ref_available("generic"), reason="oracle/_ref not built (no reference tree)")
def test_oracle_coo_to_csr_vs_live_seldon():
    rng = np.random.default_rng(9)
    with tempfile.TemporaryDirectory() as tmp:
        for k in range(3):
            nnz = 20000 + 5000 * k
            row = rng.integers(0, 3000, nnz).astype(np.int32)
            col = rng.integers(0, 2000 + 500 * k, nnz).astype(np.int32)
            row[: nnz // 10] = row[nnz // 10: 2 * (nnz // 10)]
            col[: nnz // 10] = col[nnz // 10: 2 * (nnz // 10)]
            val = rng.standard_normal(nnz)
            orc.write_seldon_vec(f"{tmp}/r.bin", row)
            orc.write_seldon_vec(f"{tmp}/c.bin", col)
            orc.write_seldon_vec(f"{tmp}/v.bin", val)
            orc.run_ref(["coo2csr", "d", f"{tmp}/r.bin", f"{tmp}/c.bin", f"{tmp}/v.bin", 0, 0, 0, f"{tmp}/o.bin"])
            ref = orc.read_seldon_csr(f"{tmp}/o.bin")
            got = orc.coo_to_csr(row, col, val)
            assert ref[:2] == got[:2] and all(np.array_equal(a, b) for a, b in zip(ref[2:], got[2:]))


def _sor_inputs(fx, A, dt):
    return wl.uniform(A.m, fx["spec"]["xseed"]).astype(dt), wl.uniform(A.m, fx["spec"]["bseed"]).astype(dt)


def _bytes_equal(a, b):
    return a.dtype == b.dtype and a.shape == b.shape and a.tobytes() == b.tobytes()


def test_oracle_sor_matches_seldon_fixture():
    """SOR / SSOR sweeps of the real Seldon build, bitwise: RowSparse,
    ArrayRowSparse and RowSymSparse; forward, backward, both; one and two
    sweeps; several omega; float values with a float and with a double
    omega; rows with scrambled columns, one of which hides its diagonal
    from Seldon's A(j, j)."""
    from tests.golden.make_golden import sor_fixture_cases
    fx = load_fixture("sor.npz")
    n = 0
    for key, A, st, dt, wide, om, it, ty in sor_fixture_cases():
        x, b = _sor_inputs(fx, A, dt)
        got = orc.sor(A, x, b, om, it, ty, storage=st, dtype=dt, omega_dtype=np.float64 if wide else None)
        assert _bytes_equal(got, fx[key]), key
        n += 1
    assert n == len(fx) - 1


def test_oracle_sor_fixture_has_teeth():
    """The fixture tells apart the rules a restatement could plausibly get
    wrong: taking the first diagonal entry of a row as a_jj (the scrambled
    matrix with its diagonal moved to the front of row 0 gives a finite
    x(0), Seldon's gives inf), omega in the value type where C++ promotes to
    double, and the symmetric storage's sweeps read as the general ones on
    the full matrix (equal to rounding, not bitwise)."""
    from tests.golden.make_golden import sor_case
    fx = load_fixture("sor.npz")
    C, _, cases = sor_case()["convdiff8scrambled"]
    front = C.ind.copy(), C.val.copy()
    a, b = C.ptr[0], C.ptr[1]
    o = np.argsort(C.ind[a:b] != 0, kind="stable")
    front[0][a:b], front[1][a:b] = C.ind[a:b][o], C.val[a:b][o]
    F = wl.CSR(C.m, C.n, C.ptr, *front)
    x, bb = _sor_inputs(fx, C, np.float64)
    om, it, ty = cases[0]
    got = orc.sor(F, x, bb, om, it, ty)
    assert np.isfinite(got[0]) and not np.isfinite(fx["convdiff8scrambled_row_d_0"][0])
    # omega's type: at least one float case differs between float and double omega
    A, _, cases = sor_case()["convdiff8"]
    x, bb = _sor_inputs(fx, A, np.float32)
    diffs = [not _bytes_equal(orc.sor(A, x, bb, om, it, ty, dtype=np.float32), fx[f"convdiff8_row_fw_{k}"])
             for k, (om, it, ty) in enumerate(cases)]
    assert any(diffs)
    # symmetric storage vs the general sweep on the full matrix
    U, _, cases = sor_case()["laplace16"]
    full = U.to_scipy().tocsr()
    full.sort_indices()
    G = wl.CSR(U.m, U.n, full.indptr.astype(np.int32), full.indices.astype(np.int32), full.data.astype(np.float64))
    x, bb = _sor_inputs(fx, U, np.float64)
    same = []
    for k, (om, it, ty) in enumerate(cases):
        g = orc.sor(G, x, bb, om, it, ty)
        ref = fx[f"laplace16_sym_d_{k}"]
        assert np.abs(g - ref).max() <= 1e-12 * np.abs(ref).max()
        same.append(_bytes_equal(g, ref))
    assert not all(same)


def test_oracle_sor_closed_forms():
    """With omega = 1 one forward sweep on a lower-triangular matrix is the
    forward substitution (numpy's triangular solve to rounding), and
    symmetric sweeps converge to A^-1 b on an SPD matrix, on the general and
    on the symmetric storage."""
    import scipy.linalg as sla
    A = wl.laplace2d(12)
    D = A.to_scipy().toarray()
    Lo = np.tril(D)
    rows, cols = np.nonzero(Lo)
    T = wl.CSR(A.m, A.n, np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=A.m))]).astype(np.int32),
               cols.astype(np.int32), Lo[rows, cols])
    b = wl.uniform(A.m, 3)
    x = orc.sor(T, np.zeros(A.m), b, 1.0, 1, 2)
    ref = sla.solve_triangular(Lo, b, lower=True)
    assert np.abs(x - ref).max() <= 1e-12 * np.abs(ref).max()
    sol = np.linalg.solve(D, b)
    assert np.abs(orc.sor(A, np.zeros(A.m), b, 1.5, 400, 0) - sol).max() < 1e-8
    assert np.abs(orc.sor(wl.upper(A), np.zeros(A.m), b, 1.5, 400, 0) - sol).max() < 1e-8


@pytest.mark.skipif(not orc.ref_available("generic"), reason="oracle/_ref not built (no reference tree)")
def test_oracle_sor_vs_live_seldon():
    """Fresh inputs through the reference build: general storages on
    power-law matrices, the symmetric storage on an upper Laplacian, float
    values with a double omega."""
    with tempfile.TemporaryDirectory() as tmp:
        runs = []
        for seed in range(2):
            A = wl.powerlaw(3000 + 1000 * seed, 70 + seed, kmin=2, kmax=40, half_width=300)
            runs += [(A, st, np.float64, False) for st in ("row", "array")]
        runs += [(wl.upper(wl.laplace2d(40, 30)), "sym", np.float64, False),
                 (wl.upper(wl.laplace2d(40, 30)), "sym", np.float32, True),
                 (wl.powerlaw(2000, 72, kmin=2, kmax=40, half_width=300), "row", np.float32, True)]
        for i, (A, st, dt, wide) in enumerate(runs):
            x = wl.uniform(A.m, 80 + i).astype(dt)
            b = wl.uniform(A.m, 90 + i).astype(dt)
            orc.write_seldon_csr(f"{tmp}/A.bin", A, dt)
            orc.write_seldon_vec(f"{tmp}/x.bin", x)
            orc.write_seldon_vec(f"{tmp}/b.bin", b)
            c = "d" if dt == np.float64 else "f"
            orc.run_ref(["sor", st, c, f"{tmp}/A.bin", f"{tmp}/x.bin", f"{tmp}/b.bin", "1.2", 3, 0, f"{tmp}/o.bin"]
                        + (["wide"] if wide else []))
            got = orc.sor(A, x, b, 1.2, 3, 0, storage=st, dtype=dt, omega_dtype=np.float64 if wide else None)
            assert _bytes_equal(orc.read_seldon_vec(f"{tmp}/o.bin", dt), got), (i, st)


def test_laplacian_eigenpairs():
    g = 40
    A = wl.laplace2d(g)
    i = np.arange(1, g + 1)
    for j, k in ((1, 1), (2, 5), (g, 1)):
        u = np.outer(np.sin(k * i * np.pi / (g + 1)), np.sin(j * i * np.pi / (g + 1))).ravel()
        lam = 4 - 2 * np.cos(j * np.pi / (g + 1)) - 2 * np.cos(k * np.pi / (g + 1))
        assert np.allclose(orc.mlt(A, u), lam * u, atol=1e-13)


def test_identity_and_diagonal_cases():
    n = 200
    I = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    b = wl.uniform(n, 3)
    r = orc.solve("cg", I, b, tol=1e-12, max_iter=10)
    assert r.code == 0 and r.nb_iter == 1 and np.array_equal(r.x, b)
    r = orc.solve("gmres", I, b, tol=1e-12, max_iter=10, restart=5)  # happy breakdown
    assert r.code == 0 and r.nb_iter == 1 and np.allclose(r.x, b, rtol=1e-15)
    d = np.array([1.0, 2.0, 3.5, 7.0, 11.0])[np.arange(n) % 5]
    D = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), d)
    r = orc.solve("cg", D, b, tol=1e-12, max_iter=100)
    assert r.code == 0 and r.nb_iter <= 5
    assert np.allclose(r.x, b / d, rtol=1e-12)


def test_iteration_edge_cases():
    A = wl.laplace2d(8)
    b = np.zeros(A.m)
    x0 = wl.uniform(A.m, 5)
    r = orc.solve("cg", A, b, x0=x0)          # Init fails: x untouched, code 0
    assert r.code == 0 and r.nb_iter == 0 and np.array_equal(r.x, x0)
    b = wl.uniform(A.m, 6)
    r = orc.solve("cg", A, b, tol=1e-14, max_iter=3)
    assert r.code == -2 and r.nb_iter == 3
    r = orc.solve("bicgstab", A, b, tol=1e-14, max_iter=4)
    assert r.code == -2 and r.nb_iter == 4
    E = wl.CSR(0, 0, np.zeros(1, np.int32), np.zeros(0, np.int32), np.zeros(0))
    assert orc.solve("cg", E, np.zeros(0)).code == 0


def test_givens_textbook():
    for a, b in ((3.0, 4.0), (-2.0, 0.5), (0.0, 1.0), (1e-300, -1e-300), (0.0, 0.0)):
        r, z, c, s = orc.genrot(a, b)
        if a == 0 and b == 0:
            assert (c, s, r) == (1.0, 0.0, 0.0)
            continue
        assert abs(abs(r) - np.hypot(a, b)) <= 1e-15 * np.hypot(a, b)
        assert abs(c * c + s * s - 1) < 1e-15
        assert abs(c * a + s * b - r) <= 1e-15 * abs(r)       # rotation maps (a,b) to (r,0)
        assert abs(-s * a + c * b) <= 1e-15 * abs(r)


def test_trsv_against_numpy():
    rng = np.random.default_rng(2)
    for n in (1, 5, 30):
        H = np.triu(rng.standard_normal((n + 3, n + 3))) + 5 * np.eye(n + 3)
        s = rng.standard_normal(n)
        got = orc.trsv_upper(H, s)
        assert np.allclose(H[:n, :n] @ got, s, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("method", ["cg", "bicgstab", "gmres"])
def test_small_dense_solution(method):
    A = wl.convdiff3d(6) if method != "cg" else wl.laplace2d(12)
    xt = wl.uniform(A.m, 8)
    b = wl.apply(A, xt)
    r = orc.solve(method, A, b, precond="jacobi", tol=1e-12, max_iter=2000, restart=20)
    assert r.code == 0
    ref = np.linalg.solve(A.to_scipy().toarray(), b)
    assert np.linalg.norm(r.x - ref) <= 1e-9 * np.linalg.norm(ref)


def test_gmres_matches_scipy_solution():
    import scipy.sparse.linalg as sla
    A, b, xt = wl.convdiff(10)
    r = orc.solve("gmres", A, b, precond="id", tol=1e-11, max_iter=3000, restart=30)
    xs = sla.spsolve(A.to_scipy().tocsc(), b)
    assert np.linalg.norm(r.x - xs) <= 1e-8 * np.linalg.norm(xs)


def test_sddmm_matches_dense_outer_product():
    A = wl.powerlaw(300, 4, kmin=2, kmax=20, half_width=30)
    lam = wl.uniform(A.m, 1)
    x = wl.uniform(A.m, 2)
    g = orc.sddmm(A, lam, x)
    dense = -np.outer(lam, x)
    rows = np.repeat(np.arange(A.m), np.diff(A.ptr))
    assert np.array_equal(g, dense[rows, A.ind])


# ------------------------------------------------------- Harwell-Boeing --

def test_oracle_hb_writer_matches_seldon():
    """WriteHarwellBoeing's text, byte for byte: RowSparse (sorted and
    scrambled rows, square and rectangular), ArrayRowSparse, RowSymSparse
    (written whole), FP64 and FP32."""
    from tests.golden.make_golden import hb_cases
    fx = load_fixture("harwell_boeing.npz")
    writers, _ = hb_cases()
    for name, (A, st) in writers.items():
        for dt, c in ((np.float64, "d"), (np.float32, "f")):
            assert orc.hb_write_text(A, st, dt) == fx[f"w_{name}_{c}"].tobytes(), (name, c)


def test_oracle_hb_reader_matches_seldon():
    """ReadHarwellBoeing + the coordinate conversion to RowSparse: E values,
    an RHS line, a pattern matrix, a rectangular one, rows unsorted within
    columns with a duplicate (kept, in file order)."""
    from tests.golden.make_golden import hb_cases
    fx = load_fixture("harwell_boeing.npz")
    _, readers = hb_cases()
    for name, text in readers.items():
        assert fx[f"r_{name}_text"].tobytes() == text
        for dt, c in ((np.float64, "d"), (np.float32, "f")):
            m, n, ptr, ind, val = orc.hb_read(text, dt)
            assert [m, n] == list(fx[f"r_{name}_{c}_dims"]), name
            assert np.array_equal(ptr, fx[f"r_{name}_{c}_ptr"]) and np.array_equal(ind, fx[f"r_{name}_{c}_ind"])
            assert fx[f"r_{name}_{c}_val"].tobytes() == val.astype(dt).tobytes(), (name, c)


def test_oracle_hb_teeth():
    """What the fixtures rule out: the symmetric storage written as its upper
    triangle only, and a column sort that is not stable (the duplicated
    entry's two copies differ, so their order shows); and Seldon's reader
    refuses Seldon's own D-format value line."""
    from tests.golden.make_golden import hb_cases
    fx = load_fixture("harwell_boeing.npz")
    writers, readers = hb_cases()
    U, _ = writers["laplace12_sym"]
    assert orc.hb_write_text(U, "row") != fx["w_laplace12_sym_d"].tobytes()
    m, n, ptr, ind, val = orc.hb_read(readers["unsorted_dup"])
    r = next(i for i in range(m) if len(set(ind[ptr[i]:ptr[i + 1]])) < ptr[i + 1] - ptr[i])
    a, b = ptr[r], ptr[r + 1]
    dup = [k for k in range(a, b) if list(ind[a:b]).count(ind[k]) > 1]
    assert val[dup[0]] != val[dup[1]]  # the two copies differ, so their order is pinned
    swapped = val.copy()
    swapped[dup[0]], swapped[dup[1]] = val[dup[1]], val[dup[0]]
    assert swapped.tobytes() != fx["r_unsorted_dup_d_val"].tobytes()
    with pytest.raises(ValueError, match="could not be parsed"):
        orc.hb_read(fx["w_powerlaw150_row_d"].tobytes())


@pytest.mark.skipif(not orc.ref_available("generic"), reason="oracle/_ref not built (no reference tree)")
def test_oracle_hb_vs_live_seldon():
    from tests.golden.make_golden import hb_text_e
    with tempfile.TemporaryDirectory() as tmp:
        A = wl.powerlaw(3000, 91, kmin=2, kmax=30, half_width=400)
        orc.write_seldon_csr(f"{tmp}/A.bin", A)
        orc.run_ref(["hbwrite", "row", "d", f"{tmp}/A.bin", f"{tmp}/o.rua"])
        assert open(f"{tmp}/o.rua", "rb").read() == orc.hb_write_text(A, "row")
        S = A.to_scipy().tocsc()
        text = hb_text_e(S.shape[0], S.shape[1], S.indptr, S.indices, S.data, "R", (8, 10), (8, 10), (4, 24, 16))
        with open(f"{tmp}/i.rua", "wb") as f:
            f.write(text)
        orc.run_ref(["hbread", "d", f"{tmp}/i.rua", f"{tmp}/o.bin"])
        ref = orc.read_seldon_csr(f"{tmp}/o.bin")
        got = orc.hb_read(text)
        assert ref[:2] == got[:2] and all(np.array_equal(x, y) for x, y in zip(ref[2:], got[2:]))


# ---------------------------------------------- FP32 family: invariants --

def test_fp32_identity_and_diagonal_cases():
    """A = I: Cg in one step, Gmres in one step through the happy breakdown
    (h_{1,0} = 0); diagonal A with k distinct values: both in at most k
    steps (the Krylov space of b holds the solution after k)."""
    n = 256
    b = wl.uniform(n, 3).astype(np.float32)
    I = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    for method in ("cg", "gmres", "bicgstab"):
        r = orc.solve(method, I, b, tol=1e-6, max_iter=10, restart=5, dtype=np.float32)
        assert r.code == 0 and r.nb_iter == 1, (method, r.code, r.nb_iter)
        assert np.allclose(r.x, b, rtol=1e-6)
    vals = np.array([1.0, 2.0, 3.5, 7.0])
    d = vals[np.arange(n) % vals.size]
    D = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), d)
    for method in ("cg", "gmres"):
        r = orc.solve(method, D, b, tol=1e-5, max_iter=50, restart=10, dtype=np.float32)
        assert r.code == 0 and r.nb_iter <= vals.size, (method, r.nb_iter)
        assert np.allclose(r.x, b / d.astype(np.float32), rtol=1e-5, atol=1e-6)


def _arnoldi_residuals(A, V, H, diag):
    """|| M^{-1} A V_k - V_{k+1} Hbar_k ||_F / ||Hbar||_F and V^T V - I, in
    double from the recorded basis (Gmres.cxx:120-135 with the left
    preconditioner M = diag(A))."""
    k = H.shape[1]
    S = A.to_scipy()
    V64 = V.astype(np.float64)
    AV = np.stack([(S @ V64[i]) / diag for i in range(k)])      # rows = vectors
    rel = np.linalg.norm(AV - H.T @ V64) / np.linalg.norm(H)
    return rel, V64 @ V64.T - np.eye(k + 1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_gmres_arnoldi_relation(dtype):
    """The first restart cycle of the oracle's Gmres satisfies M^-1 A V_k =
    V_{k+1} Hbar_k to the rounding of its vector type (FP32: the inner
    solver of the mixed-precision path); its basis vectors have unit norm
    and the first ones are orthogonal to rounding; modified Gram-Schmidt
    then loses orthogonality in inverse proportion to the residual it has
    reached (Paige, Rozloznik and Strakos, SIAM J. Matrix Anal. Appl. 28,
    2006), so the whole basis is held to eps / (relative residual)."""
    A = wl.convdiff3d(10)
    b = wl.apply(A, wl.uniform(A.m, 17))
    r = orc.solve("gmres", A, b, precond="jacobi", tol=1e-12, max_iter=40, restart=25, dtype=dtype, arnoldi=True)
    V, H = r.arnoldi
    assert H.shape == (26, 25) and V.shape == (26, A.m)
    eps = float(np.finfo(dtype).eps)
    diag = orc.jacobi_diag(A).astype(np.float64)
    rel, G = _arnoldi_residuals(A, V, H, diag)
    assert rel <= 100 * eps, rel
    assert np.abs(np.diag(G)).max() <= 20 * eps
    # after j steps the cycle's residual estimate is hist[j]: the leading
    # (j+1) x (j+1) block of V^T V - I stays below 20 eps / hist[j]
    for j in range(1, 26):
        assert np.abs(G[:j + 1, :j + 1]).max() <= 20 * eps / r.hist[j], (j, np.abs(G[:j + 1, :j + 1]).max())
    # and it is not exact: FP32 loses far more than FP64 (the basis really
    # is built in the vector type)
    assert np.abs(G).max() >= 10 * eps


def test_gmres_arnoldi_check_has_teeth():
    """Slips a restatement could make, applied to the recorded cycle, each
    break the relation by orders of magnitude more than FP32 rounding: a
    sign flip of an MGS coefficient, a dropped sub-diagonal norm, the
    Hessenberg transposed in its upper part, the preconditioner left out."""
    A = wl.convdiff3d(10)
    b = wl.apply(A, wl.uniform(A.m, 17))
    r = orc.solve("gmres", A, b, precond="jacobi", tol=1e-12, max_iter=40, restart=25, dtype=np.float32,
                  arnoldi=True)
    V, H = r.arnoldi
    diag = orc.jacobi_diag(A).astype(np.float64)
    k = H.shape[1]
    bad = []
    H1 = H.copy(); H1[2, 5] = -H1[2, 5]; bad.append((H1, diag))
    H2 = H.copy(); H2[4, 3] = 0.0; bad.append((H2, diag))
    H3 = H.copy(); H3[:k, :k] = np.triu(H[:k, :k]).T + np.tril(H[:k, :k], -1); bad.append((H3, diag))
    bad.append((H, np.ones_like(diag)))
    for Hb, db in bad:
        rel, _ = _arnoldi_residuals(A, V, Hb, db)
        assert rel > 10 * 100 * float(np.finfo(np.float32).eps), rel  # 10x the relation's bar


@pytest.mark.parametrize("method,precond", [("cg", "id"), ("bicgstab", "jacobi"), ("gmres", "jacobi")])
def test_fp32_solution_within_kappa_eps(method, precond):
    """FP32 solves land within kappa(A) * eps_32 (times a modest factor) of the
    FP64 oracle's solution, the forward-error bound of a backward-stable
    solve; kappa from numpy's dense 2-norm condition number."""
    A = wl.laplace2d(20) if method == "cg" else wl.convdiff3d(8)
    b = wl.apply(A, wl.uniform(A.m, 41))
    r64 = orc.solve(method, A, b, precond=precond, tol=1e-13, max_iter=5000, restart=40)
    r32 = orc.solve(method, A, b, precond=precond, tol=1e-6, max_iter=5000, restart=40, dtype=np.float32)
    assert r64.code == 0 and r32.code == 0
    kappa = np.linalg.cond(A.to_scipy().toarray())
    err = np.linalg.norm(r32.x.astype(np.float64) - r64.x) / np.linalg.norm(r64.x)
    eps32 = float(np.finfo(np.float32).eps)
    assert err <= 10 * kappa * max(eps32, 1e-6), (err, kappa)
    assert err >= eps32 / 10  # it is an FP32 solve, not an FP64 one


def test_fp32_cg_and_bicgstab_use_float_arithmetic():
    """The FP32 family's arithmetic is float, not a rounded FP64 run: its
    history departs from the FP64 oracle's after the first steps by far more
    than FP64 rounding, while staying on the same convergence curve."""
    A = wl.laplace2d(32)
    b = wl.apply(A, wl.uniform(A.m, 5))
    h64 = orc.solve("cg", A, b, tol=1e-6, max_iter=500).hist
    h32 = orc.solve("cg", A, b, tol=1e-6, max_iter=500, dtype=np.float32).hist
    n = min(h64.size, h32.size)
    rel = np.abs(h32[:n] - h64[:n]) / h64[:n]
    assert rel[1:].max() > 1e-9 and rel[:10].max() < 1e-3


def test_diffusion_grad_reference_against_its_own_finite_differences():
    """The oracle's FP64 gradient of L = |x - x_obs|^2, x = A(theta)^{-1} b
    (its Cg forward and adjoint, its SDDMM, and the numpy chain rule through
    the harmonic-mean faces) against central finite differences of the
    oracle's own solve on the C generator's matrix: every theta component
    of a 5^3 grid (interior, face, edge and corner cells, so every branch of
    the chain rule) and every b component."""
    n = 5
    N = n ** 3
    theta = wl.normal(N, 3, 0.0, 0.5)
    b = wl.uniform(N, 4, 0.0, 1.0)
    x_obs = orc.solve("cg", wl.diffusion3d(n, theta + wl.normal(N, 5, 0.0, 0.1)), b, precond="jacobi",
                      tol=1e-15, max_iter=5000).x
    A = wl.diffusion3d(n, theta)
    ref = orc.diffusion_grad_reference(n, theta, A.val, A, b, x_obs, tol=1e-15, max_iter=5000)

    def L(th, bb):
        x = orc.solve("cg", wl.diffusion3d(n, th), bb, precond="jacobi", tol=1e-15, max_iter=5000).x
        return float(np.sum((x - x_obs) ** 2))

    h = 1e-6
    gt = np.array([(L(theta + h * e, b) - L(theta - h * e, b)) / (2 * h) for e in np.eye(N)])
    gb = np.array([(L(theta, b + h * e) - L(theta, b - h * e)) / (2 * h) for e in np.eye(N)])
    assert np.linalg.norm(gt - ref["grad_theta"]) <= 1e-6 * np.linalg.norm(gt)
    assert np.linalg.norm(gb - ref["grad_b"]) <= 1e-6 * np.linalg.norm(gb)
    # componentwise too: a dropped term (a face's neighbour share, a boundary
    # face) shows in the components it touches, not only in the norm
    assert np.max(np.abs(gt - ref["grad_theta"])) <= 1e-6 * np.max(np.abs(gt))


# ------------------------------------------------------- Cgs and BiCg ----

def _overlay_fixture():
    return np.load(os.path.join(GOLDEN, "overlay_cpu.npz"), allow_pickle=False)


@pytest.mark.parametrize("method", ["cgs", "bicg"])
def test_oracle_cgs_bicg_match_seldon_fixture(method):
    """Seldon's own Cgs / BiCg (Cgs.cxx:46-137, BiCg.cxx:47-131, generic
    templates, run by the overlay program on its CPU storages) on the 24 x 24
    upwind convection-diffusion system: residual history, iteration numbers,
    count and code, bitwise."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve(method, A, b, tol=1e-8, max_iter=2000)
    assert r.code == int(fx[f"{method}_cpu_code"]) == 0
    assert r.nb_iter == int(fx[f"{method}_cpu_nb"])
    assert np.array_equal(r.hist_it, fx[f"{method}_cpu_its"])
    assert np.array_equal(r.hist, fx[f"{method}_cpu_hist"])


def test_oracle_cgs_bicg_fixture_check_has_teeth():
    """The same comparison fails for a slightly different system (one entry
    moved by one ulp) and for the other method's history."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    val = A.val.copy()
    val[100] = np.nextafter(val[100], 0.0)
    B = wl.CSR(A.m, A.n, A.ptr, A.ind, val)
    assert not np.array_equal(orc.solve("bicg", B, b, tol=1e-8, max_iter=2000).hist, fx["bicg_cpu_hist"])
    assert not np.array_equal(orc.solve("cgs", A, b, tol=1e-8, max_iter=2000).hist[:20], fx["bicg_cpu_hist"][:20])


@pytest.mark.parametrize("method", ["cgs", "bicg"])
def test_oracle_cgs_bicg_one_loop_cases(method):
    """A = 2.5 I with the identity, and a diagonal A with the Jacobi
    preconditioner (M^-1 A = I): one loop of either method solves the system
    exactly (two of Seldon's iterations: both methods count the two products
    of a loop), and the identity on the diagonal A needs at most one loop per
    distinct value."""
    n = 120
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    b = wl.uniform(n, 8)
    r = orc.solve(method, wl.CSR(n, n, *eye, np.full(n, 2.5)), b, tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, b / 2.5, rtol=1e-15)
    d = np.array([1.0, 2.0, 3.5, 7.0])[np.arange(n) % 4]
    D = wl.CSR(n, n, *eye, d)
    r = orc.solve(method, D, b, precond="jacobi", tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, b / d, rtol=1e-14)
    r = orc.solve(method, D, b, tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter <= 2 * 4 and np.allclose(r.x, b / d, rtol=1e-10)


@pytest.mark.parametrize("precond", ["id", "jacobi"])
def test_oracle_bicg_on_spd_follows_cg(precond):
    """On a symmetric positive definite A, BiCg with r~0 = r0 builds the same
    Krylov recurrences as Cg (p~ = p, r~ = r) with two iteration counts per
    loop: its residual history at iteration 2k equals Cg's at k up to
    rounding (A^T p~ is summed in the transposed order), with the identity
    and with Jacobi.  A wrong sign or a swapped operand in the r~ / p~
    updates breaks the match at once."""
    A = wl.aniso2d(20, 20, 3.0)
    b = wl.apply(A, wl.uniform(A.m, 12))
    cg = orc.solve("cg", A, b, precond=precond, tol=1e-10, max_iter=2000)
    bi = orc.solve("bicg", A, b, precond=precond, tol=1e-10, max_iter=4000)
    assert cg.code == bi.code == 0
    assert abs(bi.nb_iter - 2 * cg.nb_iter) <= 2
    assert np.array_equal(bi.hist_it[:30], 2 * cg.hist_it[:30])
    rel = np.abs(bi.hist[:30] - cg.hist[:30]) / cg.hist[:30]
    assert rel.max() < 1e-9, rel.max()


def test_oracle_cgs_squares_the_bicg_residual_polynomial_early():
    """Cgs's residual is the square of BiCg's residual polynomial applied to
    r0 (Sonneveld): in exact arithmetic both need the same number of loops on
    a system whose Krylov space has small dimension -- here a diagonal A with
    five distinct values and the identity: at most five loops each."""
    n = 250
    d = np.array([1.0, 1.5, 3.0, 4.0, 9.0])[np.arange(n) % 5]
    D = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), d)
    b = wl.uniform(n, 21)
    for m in ("cgs", "bicg"):
        r = orc.solve(m, D, b, tol=1e-11, max_iter=100)
        assert r.code == 0 and r.nb_iter <= 10, (m, r.nb_iter)
        assert np.allclose(r.x, b / d, rtol=1e-9)


@pytest.mark.parametrize("method", ["cgs", "bicg"])
def test_oracle_cgs_bicg_fp32_within_kappa_eps(method):
    """The FP32 versions land within kappa * eps_32 of the FP64 oracle's
    solution and are float solves (not a rounded FP64 run)."""
    A, b, _ = wl.upwind(16)
    r64 = orc.solve(method, A, b, precond="jacobi", tol=1e-13, max_iter=4000)
    r32 = orc.solve(method, A, b, precond="jacobi", tol=1e-5, max_iter=4000, dtype=np.float32)
    assert r64.code == 0 and r32.code == 0
    kappa = np.linalg.cond(A.to_scipy().toarray())
    err = np.linalg.norm(r32.x.astype(np.float64) - r64.x) / np.linalg.norm(r64.x)
    eps32 = float(np.finfo(np.float32).eps)
    assert eps32 / 10 <= err <= 10 * kappa * max(eps32, 1e-5), (err, kappa)


# ------------------------------------------------------------- TfQmr ----

def test_oracle_tfqmr_matches_seldon_fixture():
    """Seldon's own TfQmr (TfQmr.cxx:45-240, generic templates, the overlay
    program's CPU leg) on the 24 x 24 upwind system: history (its kappa
    bounds), iteration numbers, count and code, bitwise."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve("tfqmr", A, b, tol=1e-8, max_iter=2000)
    assert r.code == int(fx["tfqmr_cpu_code"]) == 0
    assert r.nb_iter == int(fx["tfqmr_cpu_nb"])
    assert np.array_equal(r.hist_it, fx["tfqmr_cpu_its"])
    assert np.array_equal(r.hist, fx["tfqmr_cpu_hist"])


def test_oracle_tfqmr_closed_forms():
    """A = 2.5 I, and a diagonal A under Jacobi (M^-1 A = I): the first half
    step gives w = 0, so theta = tau = kappa = 0 and x = b / a exactly at
    iteration 0.  On a general system the quasi-residual bound holds: the
    true (left-preconditioned) residual at the end is at most the last
    kappa-based estimate Finished() saw."""
    n = 90
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    b = wl.uniform(n, 4)
    r = orc.solve("tfqmr", wl.CSR(n, n, *eye, np.full(n, 2.5)), b, tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter == 0 and np.allclose(r.x, b / 2.5, rtol=1e-15)
    d = np.array([1.0, 2.0, 3.5, 7.0])[np.arange(n) % 4]
    r = orc.solve("tfqmr", wl.CSR(n, n, *eye, d), b, precond="jacobi", tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter == 0 and np.allclose(r.x, b / d, rtol=1e-15)
    for precond in ("id", "jacobi"):
        A, b, _ = wl.upwind(20)
        r = orc.solve("tfqmr", A, b, precond=precond, tol=1e-9, max_iter=3000)
        assert r.code == 0
        res = b - orc.mlt(A, r.x)
        dg = orc.jacobi_diag(A, None, np.float64) if precond == "jacobi" else np.ones(A.m)
        rel = np.linalg.norm(res / dg) / np.linalg.norm(b / dg)
        assert rel <= r.hist[-1] * (1 + 1e-6) + 1e-14, (rel, r.hist[-1])


def test_oracle_tfqmr_bound_has_teeth():
    """The same bound fails when the last x update is skipped (a plausible
    slip: applying x += eta d only when the solve continues)."""
    A, b, _ = wl.upwind(20)
    r = orc.solve("tfqmr", A, b, tol=1e-6, max_iter=3000)
    r_short = orc.solve("tfqmr", A, b, tol=1e-6, max_iter=int(r.hist_it[-1]))
    assert r_short.code == -2
    rel = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert rel <= r.hist[-1] * (1 + 1e-6)
    # the iterate of the previous half step is further from b than the bound
    prev = orc.solve("tfqmr", A, b, tol=1e-30, max_iter=max(int(r.hist_it[-1]) - 1, 0))
    relp = np.linalg.norm(b - orc.mlt(A, prev.x)) / np.linalg.norm(b)
    assert relp > r.hist[-1]


def test_oracle_tfqmr_fp32_within_kappa_eps():
    A, b, _ = wl.upwind(16)
    r64 = orc.solve("tfqmr", A, b, precond="jacobi", tol=1e-13, max_iter=4000)
    r32 = orc.solve("tfqmr", A, b, precond="jacobi", tol=1e-5, max_iter=4000, dtype=np.float32)
    assert r64.code == 0 and r32.code == 0
    kappa = np.linalg.cond(A.to_scipy().toarray())
    err = np.linalg.norm(r32.x.astype(np.float64) - r64.x) / np.linalg.norm(r64.x)
    eps32 = float(np.finfo(np.float32).eps)
    assert eps32 / 10 <= err <= 10 * kappa * 1e-5, (err, kappa)


# --------------------------------------------------------------- Qmr ----

def test_oracle_qmr_matches_seldon_fixture():
    """Seldon's own Qmr (Qmr.cxx:42-190, the overlay program's CPU leg) on
    the 24 x 24 upwind system: history, iteration numbers, count and code,
    bitwise."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve("qmr", A, b, tol=1e-8, max_iter=2000)
    assert r.code == int(fx["qmr_cpu_code"]) == 0
    assert r.nb_iter == int(fx["qmr_cpu_nb"])
    assert np.array_equal(r.hist_it, fx["qmr_cpu_its"])
    assert np.array_equal(r.hist, fx["qmr_cpu_hist"])


def test_oracle_qmr_closed_forms_and_residual():
    """A = 2.5 I: one loop gives v = w = 0, eta = |b| / 2.5 and x = b / 2.5
    exactly, r = 0 at iteration 2.  A diagonal A with four distinct values:
    at most four loops, x = b / d.  On a general system the residual Qmr
    carries (r -= s) stays the true one: its last recorded norm matches
    |b - A x| / |b| to rounding, with the identity and Jacobi -- a slip in
    the d / s / x updates breaks that at once."""
    n = 100
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    b = wl.uniform(n, 6)
    r = orc.solve("qmr", wl.CSR(n, n, *eye, np.full(n, 2.5)), b, tol=1e-12, max_iter=50)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, b / 2.5, rtol=1e-14)
    d = np.array([1.0, 2.0, 3.5, 7.0])[np.arange(n) % 4]
    for precond in ("id", "jacobi"):
        r = orc.solve("qmr", wl.CSR(n, n, *eye, d), b, precond=precond, tol=1e-12, max_iter=50)
        assert r.code == 0 and r.nb_iter <= 8 and np.allclose(r.x, b / d, rtol=1e-10), (precond, r.nb_iter)
    A, b, _ = wl.upwind(20)
    for precond in ("id", "jacobi"):
        r = orc.solve("qmr", A, b, precond=precond, tol=1e-9, max_iter=3000)
        assert r.code == 0
        true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
        assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15, (precond, true, r.hist[-1])


def test_oracle_qmr_fp32_within_kappa_eps():
    A, b, _ = wl.upwind(16)
    r64 = orc.solve("qmr", A, b, precond="jacobi", tol=1e-13, max_iter=4000)
    r32 = orc.solve("qmr", A, b, precond="jacobi", tol=1e-5, max_iter=4000, dtype=np.float32)
    assert r64.code == 0 and r32.code == 0
    kappa = np.linalg.cond(A.to_scipy().toarray())
    err = np.linalg.norm(r32.x.astype(np.float64) - r64.x) / np.linalg.norm(r64.x)
    eps32 = float(np.finfo(np.float32).eps)
    assert eps32 / 10 <= err <= 10 * kappa * 1e-5, (err, kappa)


# ------------------------------------------------------- Cgne and Lsqr ----

@pytest.mark.parametrize("method", ["cgne", "lsqr"])
def test_oracle_cgne_lsqr_match_seldon_fixture(method):
    """Seldon's own Cgne (Cgne.cxx:41-124) and Lsqr (Lsqr.cxx:41-150), the
    overlay program's CPU legs on the 24 x 24 upwind system (4000
    iterations allowed): history, iteration numbers, count and code,
    bitwise."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve(method, A, b, tol=1e-8, max_iter=4000)
    assert r.code == int(fx[f"{method}_cpu_code"]) == 0
    assert r.nb_iter == int(fx[f"{method}_cpu_nb"])
    assert np.array_equal(r.hist_it, fx[f"{method}_cpu_its"])
    assert np.array_equal(r.hist, fx[f"{method}_cpu_hist"])


def test_oracle_cgne_is_cg_on_the_normal_equations():
    """Cgne's loop is Cg on A^T A x = A^T b (two iterations per loop): its
    history at 2k matches the oracle's Cg on the explicit A^T A with A^T b
    (as a CSR matrix) up to rounding, with the identity; its solution is
    A^-1 b.  A = 2.5 I takes one loop."""
    A, b, xt = wl.upwind(10)
    D = A.to_scipy().toarray()
    N = D.T @ D
    rows, cols = np.nonzero(N)
    ptr = np.searchsorted(rows, np.arange(A.m + 1)).astype(np.int32)
    AtA = wl.CSR(A.m, A.m, ptr, cols.astype(np.int32), N[rows, cols])
    atb = orc.mlt_trans(A, b) if hasattr(orc, "mlt_trans") else D.T @ b
    cg = orc.solve("cg", AtA, atb, tol=1e-10, max_iter=2000)
    ne = orc.solve("cgne", A, b, tol=1e-10, max_iter=4000)
    assert cg.code == ne.code == 0
    k = min(30, len(cg.hist), len(ne.hist))
    assert np.array_equal(ne.hist_it[:k], 2 * cg.hist_it[:k])
    assert np.max(np.abs(ne.hist[:k] - cg.hist[:k]) / cg.hist[:k]) < 1e-8
    assert np.allclose(ne.x, xt, rtol=0, atol=1e-7)
    n = 50
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    bb = wl.uniform(n, 2)
    r = orc.solve("cgne", wl.CSR(n, n, *eye, np.full(n, 2.5)), bb, tol=1e-12, max_iter=20)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, bb / 2.5, rtol=1e-14)


def test_oracle_lsqr_residual_estimate_and_breakdown():
    """Lsqr's rnorm = |phi_bar| is the true residual norm: at the end it
    matches |b - A x| / |b| to rounding and the solution is A^-1 b.  A = 2.5 I
    takes one loop.  With A = 2 I and b = e_0 every step is exact, so the
    first u1 = A v - alpha u is exactly 0: breakdown #1 with x still zero, as
    the template has it."""
    A, b, xt = wl.upwind(12)
    r = orc.solve("lsqr", A, b, tol=1e-10, max_iter=6000)
    assert r.code == 0
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15, (true, r.hist[-1])
    assert np.allclose(r.x, xt, rtol=0, atol=1e-6)
    n = 40
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    bb = wl.uniform(n, 3)
    r = orc.solve("lsqr", wl.CSR(n, n, *eye, np.full(n, 2.5)), bb, tol=1e-12, max_iter=20)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, bb / 2.5, rtol=1e-14)
    e0 = np.zeros(n)
    e0[0] = 1.0
    r = orc.solve("lsqr", wl.CSR(n, n, *eye, np.full(n, 2.0)), e0, tol=1e-12, max_iter=20)
    assert r.code == 1 and r.nb_iter == 0 and np.all(r.x == 0)


@pytest.mark.parametrize("method", ["cgne", "lsqr"])
def test_oracle_cgne_lsqr_fp32_within_kappa_eps(method):
    A, b, _ = wl.upwind(8)
    r64 = orc.solve(method, A, b, tol=1e-13, max_iter=8000)
    r32 = orc.solve(method, A, b, tol=1e-5, max_iter=8000, dtype=np.float32)
    assert r64.code == 0 and r32.code == 0
    kappa = np.linalg.cond(A.to_scipy().toarray())
    err = np.linalg.norm(r32.x.astype(np.float64) - r64.x) / np.linalg.norm(r64.x)
    eps32 = float(np.finfo(np.float32).eps)
    assert eps32 / 10 <= err <= 10 * kappa ** 2 * 1e-5, (err, kappa)


def test_oracle_cg_is_seldons_cocg_on_reals():
    """Seldon's CoCg (CoCg.cxx:44-115, the overlay program's CPU leg on the
    64 x 64 Laplacian) has Cg's loop for real values: the oracle's Cg
    reproduces its history, iteration numbers and count bitwise, which is
    why the library runs CoCg as its fused Cg."""
    import math
    fx = _overlay_fixture()
    A = wl.laplace2d(64)
    xt = np.array([math.sin(0.37 * i) + 0.1 * math.cos(1.3 * i) for i in range(A.m)])
    b = orc.mlt(A, xt)
    assert np.array_equal(np.frombuffer(fx["b_cpu"].tobytes()[4:], np.float64), b)  # Vector::Write: int n, then b
    r = orc.solve("cg", A, b, tol=1e-8, max_iter=2000)
    assert r.nb_iter == int(fx["cocg_cpu_nb"]) and r.code == int(fx["cocg_cpu_code"]) == 0
    assert np.array_equal(r.hist_it, fx["cocg_cpu_its"]) and np.array_equal(r.hist, fx["cocg_cpu_hist"])


def test_oracle_bicgcr_matches_seldon_fixture_and_closed_forms():
    """Seldon's own BiCgcr (BiCgcr.cxx:45-117, the overlay program's CPU leg
    on the 64 x 64 Laplacian): history, iteration numbers, count, bitwise.
    A = 2.5 I: the first loop solves it (x = b / 2.5); where v rounds to
    exactly 0, tau = (w, A s) is 0 and the template reports its breakdown #2
    at iteration 1, else Finished() ends it at iteration 2.  The carried
    residual v stays the true one."""
    import math
    fx = _overlay_fixture()
    A = wl.laplace2d(64)
    xt = np.array([math.sin(0.37 * i) + 0.1 * math.cos(1.3 * i) for i in range(A.m)])
    b = orc.mlt(A, xt)
    r = orc.solve("bicgcr", A, b, tol=1e-8, max_iter=2000)
    assert r.nb_iter == int(fx["bicgcr_cpu_nb"]) and r.code == int(fx["bicgcr_cpu_code"]) == 0
    assert np.array_equal(r.hist_it, fx["bicgcr_cpu_its"]) and np.array_equal(r.hist, fx["bicgcr_cpu_hist"])
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-4 * r.hist[-1] + 1e-15
    n = 60
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    bb = wl.uniform(n, 9)
    for precond in ("id", "jacobi"):
        r = orc.solve("bicgcr", wl.CSR(n, n, *eye, np.full(n, 2.5)), bb, precond=precond, tol=1e-12, max_iter=20)
        assert (r.code, r.nb_iter) in ((2, 1), (0, 2)) and np.allclose(r.x, bb / 2.5, rtol=1e-14)


def test_oracle_qmrsym_matches_seldon_fixture_and_residual():
    """Seldon's own QmrSym (QmrSym.cxx:42-166, the overlay program's CPU leg
    on the 64 x 64 Laplacian): history, iteration numbers, count, bitwise;
    its carried residual (r -= s) stays the true one; A = 2.5 I is solved
    in one loop."""
    import math
    fx = _overlay_fixture()
    A = wl.laplace2d(64)
    xt = np.array([math.sin(0.37 * i) + 0.1 * math.cos(1.3 * i) for i in range(A.m)])
    b = orc.mlt(A, xt)
    r = orc.solve("qmrsym", A, b, tol=1e-8, max_iter=2000)
    assert r.nb_iter == int(fx["qmrsym_cpu_nb"]) and r.code == int(fx["qmrsym_cpu_code"]) == 0
    assert np.array_equal(r.hist_it, fx["qmrsym_cpu_its"]) and np.array_equal(r.hist, fx["qmrsym_cpu_hist"])
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15
    n = 60
    eye = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
    bb = wl.uniform(n, 19)
    r = orc.solve("qmrsym", wl.CSR(n, n, *eye, np.full(n, 2.5)), bb, tol=1e-12, max_iter=20)
    assert r.code == 0 and r.nb_iter == 1 and np.allclose(r.x, bb / 2.5, rtol=1e-14)


def test_oracle_minres_matches_seldon_fixture_and_estimate():
    """Seldon's own MinRes (MinRes.cxx:47-151, the overlay program's CPU leg
    on the 64 x 64 Laplacian): history, iteration numbers, count, bitwise.
    Its stopping quantity np = |b| prod |s| is the true residual norm of
    the iterate in exact arithmetic: at the end it matches |b - A x| to
    rounding (identity), and the iterate solves A x = b."""
    import math
    fx = _overlay_fixture()
    A = wl.laplace2d(64)
    xt = np.array([math.sin(0.37 * i) + 0.1 * math.cos(1.3 * i) for i in range(A.m)])
    b = orc.mlt(A, xt)
    r = orc.solve("minres", A, b, tol=1e-8, max_iter=2000)
    assert r.nb_iter == int(fx["minres_cpu_nb"]) and r.code == int(fx["minres_cpu_code"]) == 0
    assert np.array_equal(r.hist_it, fx["minres_cpu_its"]) and np.array_equal(r.hist, fx["minres_cpu_hist"])
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15, (true, r.hist[-1])
    assert np.linalg.norm(r.x - xt) <= 1e-8 * 2e3 * np.linalg.norm(xt)  # kappa(A) ~ 1.7e3 times the tolerance


def test_oracle_symmlq_matches_seldon_fixture():
    """Seldon's own Symmlq (Symmlq.cxx:45-161, the overlay program's CPU leg
    on the 64 x 64 Laplacian): history, iteration numbers, count, bitwise;
    after its last step x solves A x = b to kappa times the tolerance; and
    without that step (max_iter reached) x is further from it."""
    import math
    fx = _overlay_fixture()
    A = wl.laplace2d(64)
    xt = np.array([math.sin(0.37 * i) + 0.1 * math.cos(1.3 * i) for i in range(A.m)])
    b = orc.mlt(A, xt)
    r = orc.solve("symmlq", A, b, tol=1e-8, max_iter=2000)
    assert r.nb_iter == int(fx["symmlq_cpu_nb"]) and r.code == int(fx["symmlq_cpu_code"]) == 0
    assert np.array_equal(r.hist_it, fx["symmlq_cpu_its"]) and np.array_equal(r.hist, fx["symmlq_cpu_hist"])
    assert np.linalg.norm(r.x - xt) <= 1e-8 * 2e3 * np.linalg.norm(xt)
    r2 = orc.solve("symmlq", A, b, tol=1e-8, max_iter=60)
    assert r2.code == -2 and np.linalg.norm(r2.x - xt) > np.linalg.norm(r.x - xt)


def test_oracle_qcgs_matches_seldon_fixture():
    """Seldon's own QCgs (QCgs.cxx:47-164, the overlay program's CPU leg on
    the 24 x 24 upwind system): history, iteration numbers, count, bitwise;
    the smoothed residual r_qcgs it stops on is the true residual of
    x = x_qcgs at the end (identity), and a diagonal A is solved."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve("qcgs", A, b, tol=1e-8, max_iter=2000)
    assert r.code == int(fx["qcgs_cpu_code"]) == 0 and r.nb_iter == int(fx["qcgs_cpu_nb"])
    assert np.array_equal(r.hist_it, fx["qcgs_cpu_its"]) and np.array_equal(r.hist, fx["qcgs_cpu_hist"])
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15, (true, r.hist[-1])
    n = 80
    d = np.array([1.0, 2.0, 3.5, 7.0])[np.arange(n) % 4]
    D = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), d)
    bb = wl.uniform(n, 13)
    r = orc.solve("qcgs", D, bb, tol=1e-11, max_iter=100)
    assert r.code == 0 and np.allclose(r.x, bb / d, rtol=1e-9)


def test_oracle_gcr_matches_seldon_fixture():
    """Seldon's own Gcr (Gcr.cxx:45-139, restart 10, the overlay program's
    CPU leg on the 24 x 24 upwind system): history -- the outer and inner
    Finished() calls, three entries at each restart -- iteration numbers,
    count, bitwise; its residual r stays the true one."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve("gcr", A, b, tol=1e-8, max_iter=2000, restart=10)
    assert r.code == int(fx["gcr_cpu_code"]) == 0 and r.nb_iter == int(fx["gcr_cpu_nb"])
    assert np.array_equal(r.hist_it, fx["gcr_cpu_its"]) and np.array_equal(r.hist, fx["gcr_cpu_hist"])
    assert list(r.hist_it[:9]) == [0, 0, 2, 4, 6, 8, 10, 10, 10]
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-15


def test_oracle_bicgstabl_matches_seldon_fixture_and_closed_forms():
    """Seldon's own BiCgStabl (BiCgStabl.cxx:43-180, l = 10, the overlay
    program's CPU leg on the 24 x 24 upwind system): history -- one
    Finished() per cycle of 2 l iterations -- count and code, bitwise.  The
    recurrence residual r_0 stays the true one.  Closed forms: with Jacobi on
    a diagonal matrix A M^{-1} = I, so BiCgStab(1)'s first cycle solves the
    system and only the final change of coordinates x = M^{-1} y gives
    x = b / d (a dropped final map or a sign slip in the x update fails it);
    without a preconditioner the BiCG polynomial gains degree l per cycle, so
    four distinct eigenvalues stop BiCgStab(l) after ceil(4 / l) cycles of
    2 l iterations, with x = b / d."""
    fx = _overlay_fixture()
    A, b, _ = wl.upwind(24)
    r = orc.solve("bicgstabl", A, b, tol=1e-8, max_iter=2000, restart=10)
    assert r.code == int(fx["bicgstabl_cpu_code"]) == 0 and r.nb_iter == int(fx["bicgstabl_cpu_nb"])
    assert np.array_equal(r.hist_it, fx["bicgstabl_cpu_its"]) and np.array_equal(r.hist, fx["bicgstabl_cpu_hist"])
    assert list(r.hist_it) == [0, 20, 40, 60, 80, 100]
    # (the last entry, 1.3e-11, is near the rounding floor of the true
    # residual, so the gap is bounded absolutely there)
    true = np.linalg.norm(b - orc.mlt(A, r.x)) / np.linalg.norm(b)
    assert abs(true - r.hist[-1]) <= 1e-3 * r.hist[-1] + 1e-11
    n = 80
    d = np.array([1.0, 2.0, 3.5, 7.0])[np.arange(n) % 4]
    D = wl.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), d)
    bb = wl.uniform(n, 13)
    r = orc.solve("bicgstabl", D, bb, precond="jacobi", tol=1e-12, max_iter=100, restart=1)
    assert r.code == 0 and r.nb_iter == 2 and np.allclose(r.x, bb / d, rtol=1e-12)
    for l, cycles in ((1, 4), (2, 2), (3, 2), (4, 1)):
        r = orc.solve("bicgstabl", D, bb, tol=1e-11, max_iter=100, restart=l)
        assert r.code == 0 and r.nb_iter == 2 * l * cycles, (l, r.nb_iter)
        assert np.allclose(r.x, bb / d, rtol=1e-9)
    # the float restatement (orc_s_bicgstabl) on the same closed forms
    # (errors relative to the largest entry: FP32 rounding)
    xs = bb / d
    r = orc.solve("bicgstabl", D, bb, precond="jacobi", tol=1e-5, max_iter=100, restart=1, dtype=np.float32)
    assert r.code == 0 and r.nb_iter == 2 and np.abs(r.x - xs).max() <= 1e-6 * np.abs(xs).max()
    for l, cycles in ((1, 4), (2, 2), (3, 2), (4, 1)):
        r = orc.solve("bicgstabl", D, bb, tol=1e-5, max_iter=100, restart=l, dtype=np.float32)
        assert r.code == 0 and r.nb_iter == 2 * l * cycles, (l, r.nb_iter)
        assert np.abs(r.x - xs).max() <= 2e-6 * np.abs(xs).max()
