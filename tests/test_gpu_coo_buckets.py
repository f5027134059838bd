"""The assembly's bucket path against the definition of the order, bitwise, where
its pieces meet: rows longer than are counted through, a bucket just within
and just over the work-group's LDS, many buckets and more than are counted,
keys of 64 bits and more, empty rows, one column, dimensions larger than the
entries', a non-zero base index."""
import numpy as np
import pytest
import torch

from tests.test_gpu_assembly import _run

pytestmark = pytest.mark.gpu


def _case(name):
    rng = np.random.default_rng(11)
    ints = lambda hi, k: rng.integers(0, hi, k)
    if name == "one entry":
        return np.array([2]), np.array([1]), 0, 0, 0
    if name == "one column":  # no column bits; every row a run of duplicates
        return ints(3000, 20000), np.zeros(20000, int), 0, 0, 0
    if name == "a row a bucket":
        return np.arange(5 * 4097) % 5, ints(5000, 5 * 4097), 0, 0, 0
    if name == "few":  # the last count that is sorted, and the first that is not
        return ints(500, 16384), ints(500, 16384), 0, 0, 0
    if name == "not few":
        return ints(500, 16385), ints(500, 16385), 0, 0, 0
    if name == "long rows":  # 127, 128 and 129 entries: four runs of 32, one more for the last
        return np.repeat(np.arange(600), 127 + np.arange(600) % 3), ints(90, int((127 + np.arange(600) % 3).sum())), 0, 0, 0
    if name == "one long row":  # a bucket of 6542 entries: within the second LDS size
        return np.concatenate([ints(20000, 60000), np.full(5000, 777)]), ints(20000, 65000), 0, 0, 0
    if name == "over the LDS":  # 9000 entries in one row: the general sort
        return np.concatenate([ints(20000, 60000), np.full(9000, 777)]), ints(20000, 69000), 0, 0, 0
    if name == "full bucket":  # the last 544 rows: exactly 8192 entries
        return np.concatenate([np.arange(20000), np.full(7648, 19999)]), ints(20000, 27648), 0, 0, 0
    if name == "empty rows":  # 2051 buckets, dealt in two splits
        return 40 * ints(50000, 30000), ints(7, 30000), 0, 2100000, 0
    if name == "wide":  # 24 column bits: a 51-bit key
        return ints(70000, 200000), ints(1 << 24, 200000), 0, 0, 0
    if name == "widest":  # 31 column bits
        return ints(900, 20000), np.concatenate([ints(1 << 30, 19999), [2**31 - 2]]), 0, 0, 0
    if name == "many buckets":  # 2048 of them, a 60-bit key
        return ints(1 << 21, 100000), ints(1 << 27, 100000), 0, 0, 0
    if name == "too many buckets":  # 39063, over the 36864 that are counted: the general sort
        return ints(40000000, 100000), ints(7, 100000), 0, 40000000, 0
    if name == "64-bit key":  # 6 bits of the bucket, 10 of the row, 31 of the column, 17 of the place
        return ints(1 << 21, 100000), np.concatenate([ints(1 << 30, 99999), [2**31 - 2]]), 0, 1 << 21, 0
    if name == "65-bit key":  # one more for the place: the general sort
        return ints(1 << 21, 200000), np.concatenate([ints(1 << 30, 199999), [2**31 - 2]]), 0, 1 << 21, 0
    if name == "base one":
        return 1 + ints(5000, 80000), 1 + ints(300, 80000), 1, 0, 0
    assert name == "part of a pass"
    return ints(9000, 4096 * 33 + 5), ints(9000, 4096 * 33 + 5), 0, 9000, 9500


# cases that take the general sort
SORTED = ("one entry", "few", "over the LDS", "too many buckets", "65-bit key")


@pytest.mark.parametrize("c", ["d", "f"])
@pytest.mark.parametrize("name", ["one entry", "one column", "a row a bucket", "few", "not few", "long rows", "one long row", "over the LDS",
                                  "full bucket", "empty rows", "wide", "widest", "many buckets", "base one",
                                  "part of a pass", "too many buckets", "64-bit key", "65-bit key"])
def test_coo_buckets(gpu, name, c):
    row, col, index, m_min, n_min = _case(name)
    rng = np.random.default_rng(7)
    perm = rng.permutation(len(row))
    row, col = row[perm].astype(np.int32), col[perm].astype(np.int32)
    tdt, ndt = (torch.float64, np.float64) if c == "d" else (torch.float32, np.float32)
    val = rng.standard_normal(len(row)).astype(ndt)
    print(f"[coo] {name} {c}: {len(row)} entries", flush=True)
    n0 = gpu.counter("coo_buckets")
    m, n, ptr, ind, out = _run(row, col, val, index, m_min, n_min, tdt)
    assert gpu.counter("coo_buckets") - n0 == (name not in SORTED)
    # the definition itself: entries by (row, column), equal ones in their
    # input order
    order = np.lexsort((np.arange(len(row)), col, row))
    want_m, want_n = max(int(row.max()) - index + 1, m_min), max(int(col.max()) - index + 1, n_min)
    assert (m, n) == (want_m, want_n)
    counts = np.bincount(row - index, minlength=want_m)
    assert np.array_equal(ptr.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    assert np.array_equal(ind.cpu().numpy(), col[order] - index)
    assert np.array_equal(out.cpu().numpy(), val[order])


def test_coo_larger_buckets(gpu):
    """19.5M rows of 2.3 entries: buckets of 512 rows would be 38086, more than
    are counted, so they hold 1024 rows (19043 of them).  Against torch's
    stable sort of the (row, column) keys."""
    from seldon_amd import krylov as K
    m, n, nnz = 19500000, 1000, 45000000
    g = torch.Generator(device="cuda").manual_seed(5)
    row = torch.randint(0, m, (nnz,), generator=g, device="cuda", dtype=torch.int32)
    col = torch.randint(0, n, (nnz,), generator=g, device="cuda", dtype=torch.int32)
    val = torch.randn(nnz, generator=g, device="cuda", dtype=torch.float64)
    n0 = gpu.counter("coo_buckets")
    got_m, got_n, ptr, ind, out = K.ConvertMatrix_from_Coordinates(row, col, val, index=0, m=m, n=n)
    assert gpu.counter("coo_buckets") == n0 + 1 and (got_m, got_n) == (m, n)
    order = torch.sort(row.to(torch.int64) * n + col, stable=True).indices
    assert torch.equal(ind, col[order]) and torch.equal(out, val[order])
    counts = torch.bincount(row, minlength=m)
    assert ptr[0] == 0 and torch.equal(ptr[1:].to(torch.int64), torch.cumsum(counts, 0))
