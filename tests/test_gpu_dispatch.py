"""The sizes at which a kernel or a rule of a dispatch can go wrong: edges of tiles, remainders, both sides of a
threshold - against the oracle or numpy."""
import ctypes as C
import time

import numpy as np
import pytest

from comet_amd import gen
from comet_amd import runtime as rt
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, scope="module")
def _device():
    rt.init(0)


@pytest.mark.parametrize("nbytes", [1, 512, 513, 8192, 8193, 1 << 20, (1 << 20) + 8, 37_000_001])
def test_freed_blocks_come_back_only_when_nothing_uses_them(nbytes):
    a = rt.DeviceArray(nbytes, np.uint8)
    a.free()
    b, c = rt.DeviceArray(nbytes, np.uint8), rt.DeviceArray(nbytes, np.uint8)
    assert b.ptr != c.ptr
    ones, twos = np.full(nbytes, 1, np.uint8), np.full(nbytes, 2, np.uint8)
    for d, v in ((b, ones), (c, twos)):
        rt._check(rt.lib().comet_hip_memcpy(d.ptr, rt._vptr(v), nbytes, 0))
    assert np.array_equal(b.to_numpy(), ones) and np.array_equal(c.to_numpy(), twos)
    old = b.ptr
    b.free()
    assert rt.lib().comet_hip_free(old) != 0          # a second time
    assert np.array_equal(c.to_numpy(), twos)


EXTENTS = [dict(a=5, b=7, c=3, d=11, e=16, f=2), dict(a=1, b=1, c=129, d=1, e=17, f=1), dict(a=8, b=16, c=8, d=17, e=16, f=3),
           dict(a=16, b=9, c=32, d=4, e=32, f=16), dict(a=2, b=64, c=4, d=32, e=15, f=1), dict(a=3, b=43, c=1, d=1, e=7, f=31)]


@pytest.mark.parametrize("forced", [None, "0,1", "1,1", "2,1", "3,1", "0,3", "1,2", "2,5", "3,4"])
@pytest.mark.parametrize("a,b,c", [("ef", "fc", "ec"), ("aebf", "dfce", "abcd"), ("aebf", "efcd", "abcd"), ("eabf", "cdfe", "cdab"),
                                   ("feab", "efcd", "dcba"), ("abef", "ef", "ab"), ("ab", "cd", "acbd"), ("ef", "f", "e"), ("f", "fa", "a")])
def test_contraction_every_tile_shape_and_layout(a, b, c, forced, monkeypatch):
    for i, extent in enumerate(EXTENTS):
        rng = np.random.default_rng(i)
        A, B = (rng.uniform(-1, 1, [extent[x] for x in lab]) for lab in (a, b))
        C0 = rng.uniform(-1, 1, [extent[x] for x in c])
        want, bound = (np.einsum(f"{a},{b}->{c}", f(A), f(B)) for f in (np.array, np.abs))
        if forced:
            monkeypatch.setenv("COMET_HIP_GETT", forced)
        for beta in (0.0, 1.0):
            dC = rt.DeviceArray.from_numpy(C0)
            rt.ttgt_contract(a, b, c, rt.DeviceArray.from_numpy(A), rt.DeviceArray.from_numpy(B), dC, beta=beta)
            assert np.all(np.abs(dC.to_numpy() - want - beta * C0) <= 1e-13 * (bound + 1.0)), (extent, beta)


@pytest.mark.parametrize("forced", ["0,1", "1,1", "1,3", "2,1", "2,5", "3,1", "3,2"])
@pytest.mark.parametrize("m,n,k", [(1100, 200, 40), (2200, 33, 33), (70, 2100, 96), (1030, 1030, 17), (129, 16, 130)])
def test_contraction_takes_every_tile_once(m, n, k, forced, monkeypatch):
    # tiles by bands of sixteen rows, an eighth of the list to an XCD: last bands of few rows, lists of no multiple of eight
    monkeypatch.setenv("COMET_HIP_GETT", forced)
    rng = np.random.default_rng(m)
    A, B, C0 = rng.uniform(-1, 1, (m, k)), rng.uniform(-1, 1, (k, n)), rng.uniform(-1, 1, (m, n))
    want, bound = A @ B, np.abs(A) @ np.abs(B)
    for beta in (0.0, 1.0):
        dC = rt.DeviceArray.from_numpy(C0)
        rt.ttgt_contract("ef", "fc", "ec", rt.DeviceArray.from_numpy(A), rt.DeviceArray.from_numpy(B), dC, beta=beta)
        assert np.all(np.abs(dC.to_numpy() - want - beta * C0) <= 1e-13 * (bound + 1.0))


@pytest.mark.parametrize("pieces", [2, 3, 7])
@pytest.mark.parametrize("a,b,c", [("ef", "fc", "ec"), ("aebf", "dfce", "abcd"), ("aebf", "efcd", "abcd"), ("feab", "efcd", "dcba"),
                                   ("abef", "ef", "ab"), ("ab", "cd", "acbd"), ("f", "fa", "a")])
def test_contraction_in_pieces(a, b, c, pieces, monkeypatch):
    # operands beyond 4 GiB are cut; here small ones are, along every index
    for i, extent in enumerate(EXTENTS + [dict(a=300, b=1, c=2, d=2, e=1, f=260), dict(a=3, b=1, c=280, d=1, e=2, f=530)]):
        rng = np.random.default_rng(i)
        A, B = (rng.uniform(-1, 1, [extent[x] for x in lab]) for lab in (a, b))
        C0 = rng.uniform(-1, 1, [extent[x] for x in c])
        want, bound = (np.einsum(f"{a},{b}->{c}", f(A), f(B)) for f in (np.array, np.abs))
        monkeypatch.setenv("COMET_HIP_GETT_SPAN", str(max(A.size, B.size) // pieces + 1))
        for beta in (0.0, 1.0):
            dC = rt.DeviceArray.from_numpy(C0)
            rt.ttgt_contract(a, b, c, rt.DeviceArray.from_numpy(A), rt.DeviceArray.from_numpy(B), dC, beta=beta)
            assert np.all(np.abs(dC.to_numpy() - want - beta * C0) <= 1e-13 * (bound + 1.0)), (extent, beta)


def test_contraction_of_an_operand_beyond_4_gib():
    # 1,500,672 x 361 doubles, the same 1536 rows over and over
    block, times, k = 1536, 977, 361
    A, B = (np.random.default_rng(i).uniform(-1, 1, s) for i, s in enumerate([(block, k), (k, 3)]))
    dA, dB = rt.DeviceArray((block * times, k)), rt.DeviceArray.from_numpy(B)
    assert 8 * block * times * k > 1 << 32
    for i in range(times):
        rt._check(rt.lib().comet_hip_memcpy(dA.ptr + 8 * i * block * k, rt._vptr(A), A.nbytes, 0))
    C, _ = rt.ttgt_contract("ab", "bc", "ac", dA, dB)
    got = C.to_numpy().reshape(times, block, 3)
    assert np.all(np.abs(got - A @ B) <= 1e-13 * (np.abs(A) @ np.abs(B)))


def test_contraction_over_an_index_beyond_31_bits():
    block, times = 1 << 21, 1025
    a, b = (np.random.default_rng(i).uniform(-1, 1, block) for i in (3, 4))
    dA, dB = rt.DeviceArray((1, block * times)), rt.DeviceArray((block * times, 1))
    for d, h in ((dA, a), (dB, b)):
        for i in range(times):
            rt._check(rt.lib().comet_hip_memcpy(d.ptr + 8 * block * i, rt._vptr(h), h.nbytes, 0))
    C, _ = rt.ttgt_contract("ak", "kb", "ab", dA, dB)
    assert abs(C.to_numpy()[0, 0] - times * (a @ b)) <= 1e-13 * times * (np.abs(a) @ np.abs(b))


@pytest.mark.parametrize("extent", [dict(a=24, b=23, c=22, d=21, e=25, f=26), dict(a=32, b=16, c=32, d=17, e=32, f=16)])
def test_contraction_with_a_turned_operand(extent):
    rng = np.random.default_rng(7)
    A, B = (rng.uniform(-1, 1, [extent[x] for x in lab]) for lab in ("aebf", "dfce"))
    C, _ = rt.ttgt_contract("aebf", "dfce", "abcd", rt.DeviceArray.from_numpy(A), rt.DeviceArray.from_numpy(B))
    want = np.tensordot(A, B, axes=([1, 3], [3, 1])).transpose(0, 1, 3, 2)
    assert np.abs(C.to_numpy() - want).max() <= 1e-11


@pytest.mark.parametrize("nbytes", [1, 15, 16, (1 << 18) - 1, (1 << 18) + 1, (1 << 20) + 7, (1 << 20) * 7 + 16, (1 << 20) * 19 + 5])
@pytest.mark.parametrize("offset", [0, 1, 4, 8, 15, 16, 27])
def test_copies_between_host_and_device(nbytes, offset):
    host = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    d = rt.DeviceArray(nbytes + 64, np.uint8, zero=True)
    rt._check(rt.lib().comet_hip_memcpy(d.ptr + offset, rt._vptr(host), nbytes, 0))
    back = np.zeros(nbytes, np.uint8)
    rt._check(rt.lib().comet_hip_memcpy(d.ptr + offset, rt._vptr(back), nbytes, 1))
    whole = d.to_numpy()
    assert np.array_equal(back, host) and not whole[:offset].any() and not whole[offset + nbytes:].any()
    assert np.array_equal(whole[offset:offset + nbytes], host)


def test_copies_are_as_fast_wherever_they_begin():
    # byte by byte it would take twice as long
    nbytes = 60 << 10
    host = np.zeros(nbytes, np.uint8)
    d = rt.DeviceArray(nbytes + 64, np.uint8)
    def best(offset):
        times = []
        for _ in range(50):
            t = time.perf_counter()
            rt._check(rt.lib().comet_hip_memcpy(d.ptr + offset, rt._vptr(host), nbytes, 0))
            times.append(time.perf_counter() - t)
        return min(times)
    best(0)
    assert best(8) <= 1.5 * best(0)


@pytest.mark.parametrize("idt", [np.int64, np.int32])
@pytest.mark.parametrize("n,mean", [(1, 1.0), (700, 3.0), (90_001, 9.0), (400_000, 8.0)])
def test_csr_goes_up_and_comes_back(n, mean, idt):
    pos, crd, val = gen.poisson_csr(n=n, mean=mean, seed=3)
    got = rt.CsrMatrix.from_arrays((n, n), pos.astype(idt), crd.astype(idt), val).to_arrays(idt)
    assert all(np.array_equal(g, w) for g, w in zip(got, (pos, crd, val)))
    if idt is np.int64 and len(crd):
        for bad in (n, -1, (1 << 32) + int(crd[-1])):          # the last one would pass for a column in 32 bits
            wrong = crd.copy()
            wrong[-1] = bad
            with pytest.raises(rt.CometHipError, match="outside"):
                rt.CsrMatrix.from_arrays((n, n), pos, wrong, val)


def _rows(rng, n, lengths):
    """A matrix whose first rows have the given lengths, columns drawn from all n."""
    pos = np.concatenate([[0], np.cumsum(lengths), np.full(n - len(lengths), sum(lengths))]).astype(np.int64)
    return pos, np.concatenate([np.sort(rng.choice(n, l, replace=False)) for l in lengths]).astype(np.int32)


@pytest.mark.parametrize("only", [None, "workgroup", "wavefront"])
@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("double_b,double_m", [(False, False), (True, False), (False, True)])
def test_masked_sum_of_every_list_and_table_length(only, weights, double_b, double_m, monkeypatch):
    # lists around one quad, a row of 64 quads, a turn; tables around what a wavefront's holds; rows with pairs for one
    # fetch and one more, and many; columns stored twice, where pairs may not change sides
    if only:
        monkeypatch.setenv("COMET_HIP_MASKED_SUM_ONLY", only)
    n, rng = 6000, np.random.default_rng(5)
    lengths = [1, 2, 3, 4, 5, 63, 64, 65, 191, 192, 193, 255, 256, 257, 511, 513, 1023, 1025, 2047, 2049, 4100] + [0, 7] * 60
    bpos, bcrd = _rows(rng, n, lengths)
    mpos, mcrd = _rows(rng, n, lengths[::-1])
    apos, acrd = _rows(rng, n, [1, 64, 65, 129, 0, 900] * 24)
    twice = lambda pos, crd: (2 * pos, np.repeat(crd, 2))
    if double_b:
        bpos, bcrd = twice(bpos, bcrd)
    if double_m:
        mpos, mcrd = twice(mpos, mcrd)
    aval = rng.uniform(0.5, 1.5, len(acrd)) if weights else np.full(len(acrd), 0.25)
    a, b, m = (apos, acrd, aval), (bpos, bcrd, np.full(len(bcrd), 1.5)), (mpos, mcrd, np.ones(len(mcrd)))
    A, B, M = (rt.CsrMatrix.from_arrays((n, n), *x) for x in (a, b, m))
    want = orc.reduce_sum(orc.spgemm(*a, *b, n, mask=(mpos, mcrd))[2])
    got = [rt.spgemm_masked_sum(A, B, M) for _ in range(3)]
    assert got[0] == got[1] == got[2] and abs(got[0] - want) <= 1e-12 * want


@pytest.mark.parametrize("nnz", [0, 1, 3])
def test_masked_sum_of_nearly_empty_matrices(nnz):
    pos = np.array([0] + [nnz] * 5, np.int64)
    x = (pos, np.arange(nnz, dtype=np.int32), np.ones(nnz))
    A = rt.CsrMatrix.from_arrays((5, 5), *x)
    assert rt.spgemm_masked_sum(A, A, A) == (nnz if nnz else 0)


def test_masked_sum_of_a_matrix_beyond_31_bits_of_entries():
    # 1,048,577 rows of 2051 columns, the same 4096 rows over and over; the lists asked for lie at both ends of the arrays
    # and where entry 2^31 is
    rng = np.random.default_rng(9)
    ncols, per, block = 5000, 2051, 4096
    n = (1 << 20) + 1
    nnz = n * per
    assert nnz > 1 << 31
    cols = np.sort(np.argsort(rng.random((block, ncols)), axis=1)[:, :per].astype(np.int32), axis=1)
    crd, val = rt.DeviceArray(nnz, np.int32), rt.DeviceArray(nnz)
    threes = np.full(block * per, 3.0)
    L = rt.lib()
    for r in range(0, n, block):
        rows = min(block, n - r)
        rt._check(L.comet_hip_memcpy(crd.ptr + 4 * r * per, rt._vptr(cols), 4 * rows * per, 0))
        rt._check(L.comet_hip_memcpy(val.ptr + 8 * r * per, rt._vptr(threes), 8 * rows * per, 0))
    pos = rt.DeviceArray.from_numpy(np.arange(n + 1, dtype=np.int64) * per)
    b = L.comet_hip_csr_wrap(n, ncols, nnz, pos.ptr, crd.ptr, val.ptr)
    assert b, L.comet_hip_last_error()
    middle = (1 << 31) // per
    ks = np.unique(np.concatenate([[0, 1, n - 2, n - 1], middle + np.arange(-3, 4), rng.integers(0, n, 400)])).astype(np.int32)
    mrows = [np.sort(rng.choice(ncols, l, replace=False)).astype(np.int32) for l in (4000, 100, 1)]
    csr = lambda rows, m, v: rt.CsrMatrix.from_arrays((len(rows), m), np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64),
                                                      np.concatenate(rows), np.full(sum(map(len, rows)), v))
    A, M = csr([ks] * 3, n, 2.0), csr(mrows, ncols, 1.0)
    got = C.c_double(0.0)
    rt.profile_reset()
    rt.profile_enable(True)
    rt._check(L.comet_hip_spgemm_masked_sum(A.handle, b, M.handle, C.byref(got)))
    taken = rt.profile_report()
    rt.profile_enable(False)
    rt._check(L.comet_hip_csr_destroy(b))
    hits = sum(np.isin(cols[ks % block], r).sum() for r in mrows)
    assert got.value == 6.0 * hits
    assert "spgemm_pair_plan" in taken


@pytest.mark.parametrize("semiring", [None, ("min", "plus")])
@pytest.mark.parametrize("k", [1, 63, 6000, 300_001, 640_001, 1 << 20])
def test_masked_product_of_every_list_and_table_length(k, semiring):
    # tables in a wavefront's buckets, in a workgroup's with the values beside it and without, with a count for every word
    # and for every eight; lists around a quad and a turn; mask rows for one fetch of pairs and more
    rng = np.random.default_rng(9)
    sizes = [x for x in (1, 2, 3, 4, 5, 63, 64, 65, 191, 192, 193, 255, 257, 900, 4000, 15_000) if x <= k]
    la, lb = np.array(sizes * 3 + [0, 7 % (k + 1)] * 8), np.array(sizes[::-1] * 2 + [0, 1] * 40)
    pick = np.sort(rng.choice(k, min(k, 20_000), replace=False))
    rows = lambda lengths: (np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64),
                            np.concatenate([np.sort(rng.choice(pick, l, replace=False)) for l in lengths]).astype(np.int32))
    apos, acrd = rows(la)
    bt_pos, bt_crd = rows(lb)          # B by columns
    col = np.repeat(np.arange(len(lb)), lb)
    order = np.lexsort((col, bt_crd))
    bpos = np.concatenate([[0], np.cumsum(np.bincount(bt_crd, minlength=k))]).astype(np.int64)
    a, b = (apos, acrd, rng.uniform(-1, 1, len(acrd))), (bpos, col[order].astype(np.int32), rng.uniform(-1, 1, len(col)))
    n, m = len(la), len(lb)
    for keep in (0.0, 0.01, 0.5, 1.0):
        mask = rng.random((n, m)) < keep
        mp, mc = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int64), np.nonzero(mask)[1].astype(np.int32)
        A, B, M = (rt.CsrMatrix.from_arrays(shape, *x) for shape, x in (((n, k), a), ((k, m), b), ((n, m), (mp, mc, np.ones(len(mc))))))
        wp, wc, wv = orc.spgemm(*a, *b, m, mask=(mp, mc), semiring=semiring)
        p, c, v = rt.spgemm(A, B, M, semiring=semiring).to_arrays()
        assert np.array_equal(p, wp) and np.array_equal(c, wc)
        if semiring:
            assert np.array_equal(v, wv)
        else:
            bound = orc.spgemm(a[0], a[1], np.abs(a[2]), b[0], b[1], np.abs(b[2]), m, mask=(mp, mc))[2]
            assert np.all(np.abs(v - wv) <= 1e-12 * bound)


@pytest.mark.parametrize("semiring", [None, ("min", "plus")])
def test_masked_product_by_stretches_of_its_lists(semiring):
    # lists of more than 14 MiB; long rows in several parts, some of which have no list; short rows beside them
    n = 16_000
    rng = np.random.default_rng(5)
    lens = np.full(n, 82)
    lens[[0, 77, 8000, 15_999]] = 8000, 15_000, 3000, 9000

    def matrix(columns):
        crd = np.concatenate([np.sort(rng.permutation(columns[i])[:l]) if l > 82 else np.unique(rng.integers(0, n, l))
                              for i, l in enumerate(lens)])
        pos = np.concatenate([[0], np.cumsum([len(r) for r in np.split(crd, np.flatnonzero(np.diff(crd) < 0) + 1)])])
        return pos.astype(np.int64), crd.astype(np.int32), rng.uniform(1, 2, len(crd))

    low = {i: n for i in range(n)}
    low[8000] = 3500                       # all of its columns are in front: the last parts of the row are empty
    a, b, m = matrix(low), matrix(low), matrix(low)
    assert all(len(x[1]) * 12 > 14 << 20 and len(x[0]) == n + 1 for x in (a, b, m))
    A, B, M = (rt.CsrMatrix.from_arrays((n, n), *x) for x in (a, b, m))
    want = orc.spgemm(*a, *b, n, mask=m[:2], **({"semiring": semiring} if semiring else {}))
    for _ in range(2):
        p, c, v = rt.spgemm(A, B, M, semiring=semiring).to_arrays()
        assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
        assert np.array_equal(v, want[2]) if semiring else np.all(np.abs(v - want[2]) <= 1e-12 * np.abs(want[2]))


@pytest.mark.parametrize("semiring", [None, ("min", "plus")])
@pytest.mark.parametrize("rows", [40, 1152 * 3])
@pytest.mark.parametrize("n", [600, 2048, 2049, 4096, 4097, 8192, 8193])
def test_rows_of_many_products_of_a_matrix_within_a_block(n, rows, semiring):
    # the columns of a wavefront by those there are, two workgroups a CU from 4.5 such rows a CU on; rows of A of fewer and
    # of more entries than either has lanes, the first and the last column taken
    rng = np.random.default_rng(n)
    long_rows, short_rows = 10, 1100
    crd = [np.unique(np.r_[0, rng.permutation(n)[:548], n - 1]) for _ in range(long_rows)]
    crd += [np.sort(rng.permutation(n)[:4]) for _ in range(short_rows)]
    k = len(crd)
    b = (np.concatenate([[0], np.cumsum([len(c) for c in crd])]).astype(np.int64), np.concatenate(crd).astype(np.int32),
         rng.integers(1, 9, sum(len(c) for c in crd)).astype(np.float64))
    kinds = [np.array([0, 2, 3, 5, 7]), np.arange(k), np.arange(long_rows, long_rows + 513), np.arange(3)]
    picked = [kinds[i % 40 if i % 40 < 4 else 0] for i in range(rows)]
    a = (np.concatenate([[0], np.cumsum([len(r) for r in picked])]).astype(np.int64), np.concatenate(picked).astype(np.int32), None)
    a = a[:2] + (rng.integers(1, 9, len(a[1])).astype(np.float64),)
    want = orc.spgemm(*a, *b, n, **({"semiring": semiring} if semiring else {}))
    A, B = rt.CsrMatrix.from_arrays((rows, k), *a), rt.CsrMatrix.from_arrays((k, n), *b)
    for _ in range(2):
        for g, w in zip(rt.spgemm(A, B, semiring=semiring).to_arrays(), want):
            assert np.array_equal(g, w)


@pytest.mark.parametrize("counted", [True, False])
@pytest.mark.parametrize("rows,long_row,b_entries", [(60, 120, 900), (10_240, 120, 900), (10_242, 120, 900), (60, 2, 900),
                                                     (9000, 2, 900), (60, 120, 3), (7, 0, 900)])
def test_the_structure_of_rows_of_few_products(rows, long_row, b_entries, counted, monkeypatch):
    # by turns rows of no entry, of two, of a hundred that mostly meet empty rows of B, of entries without a product and (of
    # 120) of more products than a workgroup has lanes; up to 4096 rows of few products join the last kind
    if not counted:
        monkeypatch.setenv("COMET_HIP_SPGEMM_NO_LIST_CACHE", "1")
    k, n = 600, 777
    rng = np.random.default_rng(rows)
    full = 300 if b_entries == 900 else 1          # rows of B that have entries, the others are empty
    b = (np.minimum(np.arange(k + 1), full).astype(np.int64) * 3, np.sort(rng.random((full, n)).argsort(1)[:, :3]).ravel().astype(np.int32),
         rng.integers(1, 9, b_entries).astype(np.float64))
    empty = np.arange(full, k)
    kinds = [np.zeros(0, int), np.arange(min(full, 2)), np.concatenate([np.arange(min(full, 20)), empty[:80]]), empty[:3],
             np.arange(min(full, long_row))]
    picked = [kinds[i % 5] for i in range(rows)] if long_row else [kinds[0]] * rows
    pos = np.concatenate([[0], np.cumsum([len(r) for r in picked])]).astype(np.int64)
    crd = np.concatenate(picked).astype(np.int32)
    a = (pos, crd, rng.integers(1, 9, len(crd)).astype(np.float64))
    want = orc.spgemm(*a, *b, n)
    A, B = rt.CsrMatrix.from_arrays((rows, k), *a), rt.CsrMatrix.from_arrays((k, n), *b)
    for _ in range(2):
        for g, w in zip(rt.spgemm(A, B).to_arrays(), want):
            assert np.array_equal(g, w)


@pytest.mark.parametrize("nnz", [1, 2047, 2048, 2049, 6144])
def test_masked_product_gathers_its_result_by_chunks(nnz):
    # a diagonal A keeps every second row's mask entries; rows of one entry, empty rows, a row longer than a chunk
    rng = np.random.default_rng(nnz)
    lengths = np.bincount(rng.integers(0, 40, nnz), minlength=50) + np.where(np.arange(50) == 45, 2500, 0)
    mp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    mc = np.concatenate([np.sort(rng.choice(9000, l, replace=False)) for l in lengths]).astype(np.int32)
    a = (np.repeat(np.arange(26), 2)[1:].astype(np.int64), np.zeros(25, np.int32), np.full(25, 3.0))
    b = (np.array([0, 9000], np.int64), np.arange(9000, dtype=np.int32), rng.uniform(1, 2, 9000))
    A, B, M = rt.CsrMatrix.from_arrays((50, 1), *a), rt.CsrMatrix.from_arrays((1, 9000), *b), rt.CsrMatrix.from_arrays(
        (50, 9000), mp, mc, np.ones(len(mc)))
    want = orc.spgemm(*a, *b, 9000, mask=(mp, mc))
    assert all(np.array_equal(g, w) for g, w in zip(rt.spgemm(A, B, M).to_arrays(), want))


@pytest.mark.parametrize("empty", [None, "row", "column"])
@pytest.mark.parametrize("pairs", [64 * 2048 - 1, 64 * 2048, 64 * 2048 + 1, 2048, 7])
def test_masked_product_with_and_without_pairs_of_no_side(pairs, empty):
    # up to 64 chunks of 2048 pairs are counted and placed by one launch; the marks are cleared first only where a pair's
    # row of A or column of B is empty; the same handles with another mask in between leave marks behind
    rows, k, n = 40, 3, 5000
    rng = np.random.default_rng(pairs)
    cells = np.sort(rng.permutation(rows * n)[:pairs])
    mask = (np.searchsorted(cells, np.arange(rows + 1) * n).astype(np.int64), (cells % n).astype(np.int32), np.ones(pairs))
    full = (np.arange(rows + 1, dtype=np.int64) * 4000, np.tile(np.arange(4000, dtype=np.int32), rows), np.ones(rows * 4000))
    a_full, b_full = rng.integers(1, 9, (rows, k)).astype(float), rng.integers(1, 9, (k, n)).astype(float)
    a_full[::3, 1:] = 0.0                        # those rows do not meet the columns without an entry in the first row of B
    b_full[0, ::2] = 0.0
    if empty == "row":
        a_full[[0, 17, rows - 1]] = 0.0
    if empty == "column":
        b_full[:, n // 2:] = 0.0

    def csr(x):
        return np.concatenate([[0], np.cumsum((x != 0).sum(1))]).astype(np.int64), np.nonzero(x)[1].astype(np.int32), x[x != 0]

    a, b = csr(a_full), csr(b_full)
    A, B, M, F = (rt.CsrMatrix.from_arrays(shape, *x) for shape, x in (((rows, k), a), ((k, n), b), ((rows, n), mask), ((rows, n), full)))
    want, between = (orc.spgemm(*a, *b, n, mask=m[:2]) for m in (mask, full))
    for handle, w in ((F, between), (M, want), (F, between), (M, want)):
        assert all(np.array_equal(g, x) for g, x in zip(rt.spgemm(A, B, handle).to_arrays(), w))


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("c,n,shares", [(17, 15, 1), (19, 27, 1), (31, 33, 1), (61, 47, 1), (61, 47, 2), (61, 47, 3), (61, 47, 17),
                                        (61, 47, 64), (61, 47, 180)])
def test_contractions_over_irregular_k(shape, c, n, shares, monkeypatch):
    # k in two dimensions that no sixteen divide: sixteen turns of offsets at a time, less, more, up to eleven times; shares of
    # one turn and more, added by one thread an output and by several with steps left over
    monkeypatch.setenv("COMET_HIP_GETT", "%d,%d" % (shape, shares))
    rng = np.random.default_rng(c + shares)
    A, B = rng.uniform(-1, 1, (13, c, n)), rng.uniform(-1, 1, (n, c, 21))
    got = rt.ttgt_contract("icn", "nca", "ia", rt.DeviceArray.from_numpy(A), rt.DeviceArray.from_numpy(B))[0].to_numpy()
    want, bound = np.einsum("icn,nca->ia", A, B), np.einsum("icn,nca->ia", np.abs(A), np.abs(B))
    assert np.all(np.abs(got - want) <= 2 * c * n * 2.0 ** -53 * bound)          # two sums of c * n products in any order


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("K", [1, 2, 3, 5, 21, 22, 33, 63, 64, 65, 130])
@pytest.mark.parametrize("nrows", [1, 40, 4000, 14_000])
def test_spmm_chunks_of_every_length_and_width(nrows, K, accumulate):
    # chunks of 64, 128 and 256 nonzeros; rows that end with a chunk, that it would cut but that lie inside a block, that go
    # through several blocks, empty ones in front, between and behind; groups of every number of lanes
    rng = np.random.default_rng(nrows + K)
    lens = np.resize([0, 0, 60, 4, 64, 0, 130, 62, 256, 1, 0, 511, 1, 700, 3, 1, 0], nrows)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    crd, val = rng.integers(0, 500, pos[-1]).astype(np.int32), rng.uniform(-1, 1, pos[-1])
    crd = np.concatenate([np.sort(r) for r in np.split(crd, pos[1:-1])]).astype(np.int32)
    B, C0 = rng.uniform(-1, 1, (500, K)), rng.uniform(-1, 1, (nrows, K))
    A, dB = rt.CsrMatrix.from_arrays((nrows, 500), pos, crd, val), rt.DeviceArray.from_numpy(B)
    want = orc.spmm(pos, crd, val, B, C0 if accumulate else None)
    bound = orc.spmm(pos, crd, np.abs(val), np.abs(B), np.abs(C0))
    whole = (lens == 0) | (pos[:-1] // 256 == (pos[1:] - 1) // 256)          # summed in the order of the nonzeros
    for _ in range(3):
        dC = rt.DeviceArray.from_numpy(C0)
        rt.spmm(A, dB, dC, accumulate=accumulate)
        got = dC.to_numpy()
        assert np.all(np.abs(got - want) <= 1e-12 * bound)
        if K < 16 or K % 2 or pos[-1] < 1 << 19:
            assert np.array_equal(got[whole], want[whole])


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("K", [1, 3, 16, 17, 33, 64, 70])
@pytest.mark.parametrize("nrows", [130, 3000, 26_000])
def test_spmm_rows_that_are_not_cut(nrows, K, accumulate):
    # rows below 128 nonzeros across the blocks of 256, alone in their chunk or with many short ones; chunks of 64, 128 and 256
    rng = np.random.default_rng(nrows + K)
    lens = np.resize([1, 1, 127, 1, 2, 1, 96, 3, 120, 5, 1, 1, 40], nrows)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    crd = np.concatenate([np.sort(rng.choice(500, l, replace=False)) for l in lens]).astype(np.int32)
    val, B, C0 = rng.uniform(-1, 1, pos[-1]), rng.uniform(-1, 1, (500, K)), rng.uniform(-1, 1, (nrows, K))
    dC = rt.DeviceArray.from_numpy(C0)
    rt.spmm(rt.CsrMatrix.from_arrays((nrows, 500), pos, crd, val), rt.DeviceArray.from_numpy(B), dC, accumulate=accumulate)
    assert np.array_equal(dC.to_numpy(), orc.spmm(pos, crd, val, B, C0 if accumulate else None))


@pytest.mark.parametrize("K", [1, 3, 33, 64, 130])
@pytest.mark.parametrize("nrows,filled", [(70, 1), (20_000, 3), (20_000, 300), (4_000, 3_900), (100, 100)])
def test_spmm_empty_rows_belong_to_one_chunk_each(nrows, filled, K):
    # in front, between and behind, few and thousands of them to a chunk, fewer rows than chunks; C's padding is not touched
    rng = np.random.default_rng(nrows + filled)
    lens = np.zeros(nrows, np.int64)
    lens[rng.choice(np.arange(nrows // 3, nrows) if 2 * filled < nrows else nrows, filled, replace=False)] = 1
    lens[np.flatnonzero(lens)[::3]] = 90 if nrows < 200 else 7
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    crd = np.concatenate([np.sort(rng.choice(500, l, replace=False)) for l in lens]).astype(np.int32)
    val, B, ldc = rng.uniform(-1, 1, pos[-1]), rng.uniform(-1, 1, (500, K)), K + 3
    A, dB, dC = rt.CsrMatrix.from_arrays((nrows, 500), pos, crd, val), rt.DeviceArray.from_numpy(B), rt.DeviceArray((nrows, ldc))
    for _ in range(2):
        rt._check(rt.lib().comet_hip_memcpy(dC.ptr, rt._vptr(np.full((nrows, ldc), 7.0)), dC.nbytes, 0), "upload")
        rt._check(rt.lib().comet_hip_spmm_csr_f64(A.handle, K, dB.ptr, K, dC.ptr, ldc, 0), "spmm")
        got = dC.to_numpy()
        assert np.array_equal(got[:, :K], orc.spmm(pos, crd, val, B)) and np.all(got[:, K:] == 7.0)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("nlong,ncols,K", [(40, 20_000, 7), (40, 9_000, 16), (300, 9_000, 21), (300, 4_100, 64), (700, 9_000, 33),
                                           (700, 120_000, 32), (700, 120_001, 31)])
def test_spmm_chunks_by_columns(nlong, ncols, K, accumulate, monkeypatch):
    # from the second product on; chunks of 64, 128 and 256 nonzeros, and 128 in place of 256 for a large B; rows below 128
    # nonzeros across the blocks of 256, empty rows in front, between and behind
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    rng = np.random.default_rng(nlong + K)
    lens = np.resize([0, 0, 60, 4, 127, 0, 128, 1, 256, 1, 3, 100, 511], 13 * nlong)
    lens[rng.choice(len(lens) - 1, nlong, replace=False)] = 3000
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    crd = np.concatenate([np.sort(rng.choice(ncols, l, replace=False)) for l in lens]).astype(np.int32)
    val, B, C0 = rng.uniform(-1, 1, pos[-1]), rng.uniform(-1, 1, (ncols, K)), rng.uniform(-1, 1, (len(lens), K))
    A, dB = rt.CsrMatrix.from_arrays((len(lens), ncols), pos, crd, val), rt.DeviceArray.from_numpy(B)
    want = orc.spmm(pos, crd, val, B, C0 if accumulate else None)
    bound = orc.spmm(pos, crd, np.abs(val), np.abs(B), np.abs(C0))
    whole = (lens < 128) | (pos[:-1] // 256 == (pos[1:] - 1) // 256)
    first, sorted_at = None, []
    for _ in range(3):
        dC = rt.DeviceArray.from_numpy(C0)
        rt.profile_reset()
        rt.profile_enable(True)
        rt.spmm(A, dB, dC, accumulate=accumulate)
        rt.sync()
        sorted_at.append("radix_sort_pairs" in rt.profile_report())
        rt.profile_enable(False)
        got = dC.to_numpy()
        assert np.all(np.abs(got - want) <= 1e-12 * bound)
        assert np.array_equal(got[whole], want[whole])
        first = got if first is None else first
        if ncols < 100_000:          # the same chunks: the same sums
            assert np.array_equal(got, first)
    assert sorted_at == [False, True, False]


@pytest.mark.parametrize("columns,K,ordered", [("graph", 17, False), ("graph", 32, False), ("graph at random places", 17, False),
                                               ("uniform", 17, True), ("uneven", 32, True), ("one", 32, False), ("far apart", 14, True)])
def test_spmm_chunks_go_by_columns_unless_few_hold_much_of_the_matrix(columns, K, ordered, monkeypatch):
    # rows of four chunks hold half of each of these; where the columns are as uneven, the chunks stay as stored
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    rng = np.random.default_rng(8)
    if columns.startswith("graph"):
        n = 1 << 13
        pos, crd, val = gen.rmat_symmetric_csr(scale=13, edge_factor=32, seed=2)
        if columns != "graph":
            place = rng.permutation(n)
            rows, cols = place[np.repeat(np.arange(n), np.diff(pos))], place[crd]
            order = np.lexsort((cols, rows))
            crd, pos = cols[order], np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
        ncols = n
    else:
        n, ncols = 3000, 500_000 if columns == "far apart" else 20_000
        lens = np.where(np.arange(n) % 3 == 0, 1200, 9)
        u = rng.random(lens.sum()) ** (4 if columns == "uneven" else 1)
        rows, cols = np.repeat(np.arange(n), lens), (u * ncols).astype(np.int64)
        if columns == "one":              # half of the entries in columns that are in every row
            cols[::2] = np.arange(len(cols[::2])) % 700
        key = np.unique(rows * ncols + cols)
        crd, pos = key % ncols, np.concatenate([[0], np.cumsum(np.bincount(key // ncols, minlength=n))])
        val = rng.uniform(-1, 1, len(crd))
    lens, four_chunks = np.diff(pos), {"graph": 256, "uneven": 512}.get(columns.split()[0], 1024)
    assert lens[lens >= four_chunks].sum() * 2 >= len(crd)
    A, B = rt.CsrMatrix.from_arrays((n, ncols), pos.astype(np.int64), crd.astype(np.int64), val), rng.uniform(-1, 1, (ncols, K))
    dB, dC = rt.DeviceArray.from_numpy(B), rt.DeviceArray((n, K))
    bound = orc.spmm(pos, crd, np.abs(val), np.abs(B))
    for call in range(3):
        rt.profile_reset()
        rt.profile_enable(True)
        rt.spmm(A, dB, dC, accumulate=False)
        rt.sync()
        rep = rt.profile_report()
        rt.profile_enable(False)
        assert "spmm_csr_nnzsplit" in rep and "spmm_heavy_sweep" not in rep, sorted(rep)
        assert ("radix_sort_pairs" in rep) == (ordered and call == 1), call
        assert np.all(np.abs(dC.to_numpy() - orc.spmm(pos, crd, val, B)) <= 1e-12 * bound)


def test_spmm_launches_are_listed_by_the_kernel_that_runs(monkeypatch):
    # a first product and chunks by columns: the chunk kernel; a B beyond those, or the switch that turns them off: the sweep
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    n = 120_000
    pos, crd, val = gen.zipf_csr(n=n, mean=16.0, cap=4096, seed=7)
    A, B = rt.CsrMatrix.from_arrays((n, n), pos, crd, val), np.random.default_rng(3).uniform(-1, 1, (n, 64))
    for K, columns, swept in [(32, True, False), (32, True, False), (64, True, True), (32, True, False), (32, False, True)]:
        if not columns:
            monkeypatch.setenv("COMET_HIP_SPMM_NO_COLUMNS", "1")
        b = np.ascontiguousarray(B[:, :K])
        dB, dC = rt.DeviceArray.from_numpy(b), rt.DeviceArray((n, K))
        rt.profile_reset()
        rt.profile_enable(True)
        rt.spmm(A, dB, dC, accumulate=False)
        rt.sync()
        rep = rt.profile_report()
        rt.profile_enable(False)
        assert ("spmm_heavy_sweep" in rep) == ("spmm_heavy_combine" in rep) == swept, (K, columns, sorted(rep))
        assert swept or "spmm_csr_nnzsplit" in rep, (K, columns, sorted(rep))
        bound = orc.spmm(pos, crd, np.abs(val), np.abs(b))
        assert np.all(np.abs(dC.to_numpy() - orc.spmm(pos, crd, val, b)) <= 1e-12 * bound)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("K", [8, 33])
def test_spmm_of_a_matrix_without_entries_again_and_again(K, accumulate, monkeypatch):
    # with a B of the size for which chunks go by columns: there are none, and no call leaves an error behind
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    nrows, ncols = 70, 40_000
    A = rt.CsrMatrix.from_arrays((nrows, ncols), np.zeros(nrows + 1, np.int64), np.zeros(0, np.int64), np.zeros(0))
    C0, dB = np.random.default_rng(K).uniform(-1, 1, (nrows, K)), rt.DeviceArray((ncols, K), zero=True)
    for _ in range(3):
        dC = rt.DeviceArray.from_numpy(C0)
        rt.spmm(A, dB, dC, accumulate=accumulate)
        assert np.array_equal(dC.to_numpy(), C0 if accumulate else np.zeros((nrows, K)))


@pytest.mark.parametrize("K", [1, 2, 3, 5, 16, 17, 31, 32, 33, 63, 64, 65, 66, 130])
@pytest.mark.parametrize("nnz", [1, 15, 17, 63, 65, 4097])
def test_sddmm_of_every_tile_and_width(nnz, K):
    rng = np.random.default_rng(nnz + K)
    n, m = 70, 130
    cells = np.sort(rng.choice(n * m, nnz, replace=False))
    pos = np.concatenate([[0], np.cumsum(np.bincount(cells // m, minlength=n))]).astype(np.int64)
    crd, val = (cells % m).astype(np.int32), rng.uniform(-1, 1, nnz)
    C, D = rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (K, m))
    out = rt.DeviceArray.from_numpy(np.full(nnz + 1, 7.0))
    rt.sddmm(rt.CsrMatrix.from_arrays((n, m), pos, crd, val), rt.DeviceArray.from_numpy(C), rt.DeviceArray.from_numpy(D), out_values=out)
    got = out.to_numpy()
    assert np.array_equal(got[:nnz], orc.sddmm(pos, crd, val, C, D)) and got[nnz] == 7.0


@pytest.mark.parametrize("K", [1, 2, 15, 16, 17, 33, 47, 64])
@pytest.mark.parametrize("nnz", [(1 << 19) - 1, 1 << 19, (1 << 19) + 37])
def test_sddmm_of_many_entries(nnz, K):
    # the numbers of entries from which on a wavefront takes 64 of them; rows of one entry and rows of thousands
    rng = np.random.default_rng(nnz + K)
    n, m = 1500, 2000
    share = rng.pareto(1.0, n) + 1e-3
    lens = np.minimum(m, np.floor(share / share.sum() * nnz)).astype(np.int64)
    lens = lens + np.bincount(np.repeat(np.arange(n), m - lens)[: nnz - lens.sum()], minlength=n)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    crd = np.concatenate([np.sort(rng.permutation(m)[:l]) for l in lens]).astype(np.int32)
    val, C, D = rng.uniform(-1, 1, nnz), rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (K, m))
    out = rt.DeviceArray.from_numpy(np.full(nnz + 1, 7.0))
    rt.sddmm(rt.CsrMatrix.from_arrays((n, m), pos, crd, val), rt.DeviceArray.from_numpy(C), rt.DeviceArray.from_numpy(D), out_values=out)
    got = out.to_numpy()
    assert np.array_equal(got[:nnz], orc.sddmm(pos, crd, val, C, D)) and got[nnz] == 7.0


@pytest.mark.parametrize("kind", ["band", "one tile", "hub", "two rounds", "widest tile"])
@pytest.mark.parametrize("K", [1, 2, 7, 15, 16, 17, 31, 33, 48, 70])
def test_sddmm_by_tiles_of_columns(kind, K, monkeypatch):
    # runs of entries of one row in tiles of 16 columns to 512, entries of a tile in one part or several, the last one of a
    # wavefront or two; pieces of sixteen columns of C and every kind of rest; operands wider than they need be
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    rng = np.random.default_rng(K)
    n, m, run = {"band": (2500, 2600, 70), "one tile": (9000, 16, 15), "hub": (20_000, 5000, 12), "two rounds": (4600, 131_073, 40),
                 "widest tile": (5000, 131_072, 40)}[kind]
    first = rng.integers(0, m - run + 1, n)
    if kind == "hub":
        first[:15_000] = rng.integers(0, 4, 15_000)
    crd = (first[:, None] + np.arange(run)).ravel()
    lens = np.full(n, run)
    drop = rng.choice(n, n // 50, replace=False)
    keep = np.ones((n, run), bool)
    keep[drop] = False                    # empty rows
    lens[drop] = 0
    crd = crd[keep.ravel()].astype(np.int32)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    assert pos[-1] >= 1 << 15
    val, C, D = rng.uniform(-1, 1, pos[-1]), rng.uniform(-1, 1, (n, K + 3)), rng.uniform(-1, 1, (K, m + 5))
    S, out = rt.CsrMatrix.from_arrays((n, m), pos, crd, val), rt.DeviceArray.from_numpy(np.full(pos[-1] + 1, 7.0))
    dC, dD = rt.DeviceArray.from_numpy(C), rt.DeviceArray.from_numpy(D)
    want = orc.sddmm(pos, crd, val, np.ascontiguousarray(C[:, :K]), np.ascontiguousarray(D[:, :m]))
    tiled = []
    for _ in range(3):
        rt._check(rt.lib().comet_hip_memcpy(out.ptr, rt._vptr(np.full(pos[-1] + 1, 7.0)), 8 * (int(pos[-1]) + 1), 0))
        rt.profile_reset()
        rt.profile_enable(True)
        rt._check(rt.lib().comet_hip_sddmm_csr_values_f64(S.handle, K, dC.ptr, K + 3, dD.ptr, m + 5, out.ptr), "sddmm")
        rt.sync()
        tiled.append("sddmm_tile_kernel" in rt.profile_report())
        rt.profile_enable(False)
        got = out.to_numpy()
        assert np.array_equal(got[:-1], want) and got[-1] == 7.0
    by_tiles = (kind != "two rounds" or (K > 16 and K % 16 <= 12)) and (K <= 40 or pos[-1] >= 1 << 17)
    assert tiled == [False, by_tiles, by_tiles]


@pytest.mark.parametrize("wide", [False, True])
def test_sddmm_of_every_piece_and_rest(wide):
    # every number of columns up to three pieces: whole ones, a last one with lanes behind its end, a rest of one or two a lane;
    # wide: rows of C so far apart that an address is no 24-bit product
    rng = np.random.default_rng(9)
    n, m, nnz = 13, 40, 200
    cells = np.sort(rng.choice(n * m, nnz, replace=False))
    pos = np.concatenate([[0], np.cumsum(np.bincount(cells // m, minlength=n))]).astype(np.int64)
    crd, val = (cells % m).astype(np.int32), rng.uniform(-1, 1, nnz)
    S = rt.CsrMatrix.from_arrays((n, m), pos, crd, val)
    for K in range(1, 49):
        C, D = rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (K, m))
        ldc = (1 << 21) + 5 if wide else K
        flat = np.full((n - 1) * ldc + K, np.inf)          # what lies between the rows is nobody's
        np.lib.stride_tricks.as_strided(flat, (n, K), (8 * ldc, 8))[:] = C
        dC, dD, out = rt.DeviceArray.from_numpy(flat), rt.DeviceArray.from_numpy(D), rt.DeviceArray.from_numpy(np.full(nnz + 1, 7.0))
        rt._check(rt.lib().comet_hip_sddmm_csr_values_f64(S.handle, K, dC.ptr, ldc, dD.ptr, m, out.ptr), "sddmm")
        got = out.to_numpy()
        assert np.array_equal(got[:nnz], orc.sddmm(pos, crd, val, C, D)) and got[nnz] == 7.0, K


@pytest.mark.parametrize("K", [16, 17, 18, 24, 25, 31, 32])
def test_sddmm_of_rows_from_beyond_the_l2(K):
    # many entries as stored and a large D: 32 entries a wavefront
    rng = np.random.default_rng(K)
    n = 80_000
    pos = np.arange(0, 7 * n + 1, 7).astype(np.int64)
    crd = np.sort(rng.integers(0, n // 7, (n, 7)) + np.arange(7) * (n // 7), axis=1).ravel().astype(np.int32)
    val, C, D = rng.uniform(-1, 1, len(crd)), rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (K, n))
    assert len(crd) >= 1 << 19 and n * K * 8 >= 8 << 20
    out = rt.DeviceArray(len(crd))
    S = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    rt.sddmm(S, rt.DeviceArray.from_numpy(C), rt.DeviceArray.from_numpy(D), out_values=out)
    assert np.array_equal(out.to_numpy(), orc.sddmm(pos, crd, val, C, D))


@pytest.mark.parametrize("K", [27, 31, 32, 33, 64, 65])
@pytest.mark.parametrize("hub", [False, True])
def test_sddmm_in_an_order_that_keeps_columns_close(K, hub):
    # enough entries in long rows, and a D that is too large for an L2: the second call takes them by blocks of columns; with
    # a hub half of them name columns of one block, which several XCDs then share
    rng = np.random.default_rng(K)
    n, m = 2500, 40_000
    lens = np.where(np.arange(n) % 25 == 3, 6000, rng.integers(0, 9, n))
    rows = [np.sort(rng.choice(m, l, replace=False)) if not hub or l < 100 else
            np.sort(np.concatenate([rng.choice(4000, l // 2, replace=False), 4000 + rng.choice(m - 4000, l // 2, replace=False)]))
            for l in lens]
    pos, crd = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64), np.concatenate(rows).astype(np.int32)
    val, C, D = rng.uniform(-1, 1, len(crd)), rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (K, m))
    S, dC, dD = rt.CsrMatrix.from_arrays((n, m), pos, crd, val), rt.DeviceArray.from_numpy(C), rt.DeviceArray.from_numpy(D)
    want = orc.sddmm(pos, crd, val, C, D)
    for _ in range(3):
        out = rt.DeviceArray(len(crd), zero=True)
        rt.sddmm(S, dC, dD, out_values=out)
        assert np.array_equal(out.to_numpy(), want)


@pytest.mark.parametrize("semiring", [None, ("min", "plus"), ("max", "times"), ("any", "second")])
@pytest.mark.parametrize("ncols", [1, 31, 33, 1000, 65_535, 65_536, 65_537])
@pytest.mark.parametrize("kept", [True, False])
def test_spgemm_rows_with_few_products(ncols, semiring, kept, monkeypatch):
    # rows around the number of products, and matrices around the number of columns, that the small workgroups take; the
    # host knows how many rows are small only where the list of rows is kept
    if not kept:
        monkeypatch.setenv("COMET_HIP_SPGEMM_NO_LIST_CACHE", "1")
    rng = np.random.default_rng(ncols)
    csr = lambda rows: (np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64),
                        np.concatenate(rows).astype(np.int32), rng.uniform(0.5, 1.5, sum(map(len, rows))))
    k, most = 1100, min(ncols, 1000)          # rows of B: two of 1000 entries (if there is room), a hundred of one, others
    b = csr([np.sort(rng.choice(ncols, min(l, ncols), replace=False)) for l in [most] * 2 + [1] * 100 + [7, 15, 16, 17, 64, 513] * 166 + [3] * 2])
    picks = [[], [0], [5], range(102, 110), range(102, 168)] + [[0, 1, *range(2, 2 + n)] for n in (0, 7, 47, 48, 49, 100)]
    picks += [[0, 1, *range(2, 2 + n), *sorted([*range(107, 125, 6), *range(106, 154, 6)])] for n in (44, 45, 46)]
    a = csr([np.array(p, np.int64) for p in picks * 5])
    A, B = rt.CsrMatrix.from_arrays((5 * len(picks), k), *a), rt.CsrMatrix.from_arrays((k, ncols), *b)
    want = orc.spgemm(*a, *b, ncols, semiring=semiring)
    for _ in range(2):
        p, c, v = rt.spgemm(A, B, semiring=semiring).to_arrays()
        assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
        if semiring is None:
            assert np.all(np.abs(v - want[2]) <= 1e-12 * want[2])
        else:
            assert np.array_equal(v, want[2])


@pytest.mark.parametrize("ncols", [8192, 8193, 20_011, 65_535, 65_536])
def test_spgemm_structure_of_rows_with_long_rows_of_b(ncols):
    # rows of B around a sixty-fourth of the columns, the first and the last column among them, some with every column
    # twice; rows of A with none to nine of those, beyond the 512 entries that are looked at together, and with nothing else
    rng = np.random.default_rng(ncols)
    least = -(-ncols // 64)
    lens = np.array([least - 1, least, least + 1, 4 * least, ncols // 2, 0] * 2 + [7] * 900)
    cols = [np.sort(rng.choice(ncols, l, replace=False)) for l in lens]
    cols[1][0], cols[2][-1] = 0, ncols - 1
    cols[7] = np.repeat(np.sort(rng.choice(ncols, least, replace=False)), 2)
    bpos = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int64)
    b = (bpos, np.concatenate(cols).astype(np.int64), rng.uniform(0.5, 1.5, bpos[-1]))
    picks = [range(h, 12) for h in range(13)] + [[*range(h), *range(12, 12 + n)] for h in (0, 3, 9, 12) for n in (300, 511, 512, 513, 800)]
    picks += [[0, 6, *range(12, 700)], [1, 3, 4, 5, *range(300, 912)]]
    apos = np.concatenate([[0], np.cumsum([len(p) for p in picks])]).astype(np.int64)
    acrd = np.concatenate([np.array(p, np.int64) for p in picks])
    a = (apos, acrd, rng.uniform(0.5, 1.5, len(acrd)))
    A, B = rt.CsrMatrix.from_arrays((len(picks), len(lens)), *a), rt.CsrMatrix.from_arrays((len(lens), ncols), *b)
    want = orc.spgemm(*a, *b, ncols)
    for _ in range(2):
        p, c, v = rt.spgemm(A, B).to_arrays()
        assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
        assert np.all(np.abs(v - want[2]) <= 1e-12 * want[2])


@pytest.mark.parametrize("semiring", [None, ("min", "plus")])
@pytest.mark.parametrize("rows", [1020, 1030])          # around four to a CU of 256
@pytest.mark.parametrize("ncols", [1 << 17, (1 << 17) + 1])
def test_masked_dots_two_workgroups_a_cu(ncols, rows, semiring):
    # rows of more entries than a wavefront's table holds, as many of them and as many columns as decide whether two
    # workgroups share a CU; one row whose values fit a whole CU's LDS and not half of it, one that fits neither
    rng = np.random.default_rng(rows)
    pool = np.sort(rng.choice(ncols, 16_000, replace=False))
    pool[-1] = ncols - 1
    lens = np.full(rows, 200)
    lens[5], lens[9], lens[11] = 6000, 16_000, 0
    apos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    acrd = np.concatenate([np.sort(rng.choice(pool, l, replace=False)) for l in lens]).astype(np.int64)
    m = 70
    near = np.unique(np.concatenate([acrd[apos[r]:apos[r + 1]][:40] for r in range(0, rows, 20)]))
    bcols = [np.sort(rng.choice(near, l, replace=False)) for l in rng.integers(0, 199, m)]
    k = np.concatenate(bcols)
    order = np.lexsort((np.repeat(np.arange(m), [len(c) for c in bcols]), k))
    bcrd = np.repeat(np.arange(m), [len(c) for c in bcols])[order].astype(np.int64)
    bpos = np.concatenate([[0], np.cumsum(np.bincount(k, minlength=ncols))]).astype(np.int64)
    keep = rng.random((rows, m)) < 0.8
    mpos = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int64)
    mcrd = np.nonzero(keep)[1].astype(np.int64)
    a, b = (apos, acrd, rng.uniform(0.5, 1.5, len(acrd))), (bpos, bcrd, rng.uniform(0.5, 1.5, len(bcrd)))
    A, B = rt.CsrMatrix.from_arrays((rows, ncols), *a), rt.CsrMatrix.from_arrays((ncols, m), *b)
    M = rt.CsrMatrix.from_arrays((rows, m), mpos, mcrd, np.ones(len(mcrd)))
    want = orc.spgemm(*a, *b, m, mask=(mpos, mcrd), semiring=semiring)
    assert want[0][-1] > 1000
    for _ in range(2):
        p, c, v = rt.spgemm(A, B, M, semiring=semiring).to_arrays()
        assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
        if semiring is None:          # positive terms, 198 at most
            assert np.all(np.abs(v - want[2]) <= 200 * 2.0 ** -53 * want[2])
        else:
            assert np.array_equal(v, want[2])


@pytest.mark.parametrize("semiring", [None, ("min", "plus"), ("max", "times"), ("any", "second"), ("plus", "first")])
@pytest.mark.parametrize("repeats", [1, 40])
def test_spgemm_block_by_block_slices(semiring, repeats, monkeypatch):
    # slices of every length around a quad and a turn, the last entries of B, rows of A around the entries that are staged
    # at a time; columns stored more than once make slices longer than the block is wide.  Values are whole numbers and
    # zeros of either sign: sums are exact, and those of nothing but zeros and cancelled ones stay stored.
    monkeypatch.setenv("COMET_HIP_SPGEMM_WIDE", "0")
    rng = np.random.default_rng(repeats)
    m, lens = 16_384 + 700, [0, 1, 2, 3, 4, 5, 7, 8, 63, 64, 65, 255, 256, 257, 259, 1030] * 75
    if repeats > 1:
        lens = lens[:48]
    k = len(lens)
    bpos = np.concatenate([[0], np.cumsum(np.array(lens) * repeats)]).astype(np.int64)
    bcrd = np.concatenate([np.repeat(np.sort(rng.choice(m, l, replace=False)), repeats) for l in lens]).astype(np.int64)
    pick = np.array([-3.0, -1.0, -0.0, 0.0, 1.0, 2.0])
    bval = rng.choice(pick, len(bcrd))
    counts = [c for c in (1, 2, 40, 47, 63, 64, 65, 130, 1023, 1024, 1025, 1200) if c <= k] * 3
    apos = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    acrd = np.concatenate([np.sort(rng.choice(k, c, replace=False)) for c in counts])
    aval = rng.choice(pick, len(acrd))
    A, B = rt.CsrMatrix.from_arrays((len(counts), k), apos, acrd, aval), rt.CsrMatrix.from_arrays((k, m), bpos, bcrd, bval)
    want = orc.spgemm(apos, acrd, aval, bpos, bcrd, bval, m, semiring=semiring)
    for _ in range(2):
        p, c, v = rt.spgemm(A, B, semiring=semiring).to_arrays()
        assert np.array_equal(p, want[0]) and np.array_equal(c, want[1]) and np.array_equal(v, want[2])
        if semiring is None or semiring[0] == "plus":
            assert not np.any(np.signbit(v[v == 0]))          # an accumulator that starts at zero


@pytest.mark.parametrize("wide", [0, 1 << 40])
def test_spgemm_keeps_entries_whose_products_underflow(wide, monkeypatch):
    # the block kernel tells an empty accumulator by its sign: a product of no size and of either sign is an entry, +0.0
    monkeypatch.setenv("COMET_HIP_SPGEMM_WIDE", str(wide))
    rng = np.random.default_rng(3)
    n, m = 200, 20_000
    S = np.sort(np.stack([rng.choice(m, 300, replace=False) for _ in range(n)]), axis=1)
    bpos, bcrd = np.arange(0, 300 * n + 1, 300).astype(np.int64), S.ravel().astype(np.int64)
    apos = np.array([0, 1, 1 + n, 61 + n]).astype(np.int64)
    acrd = np.concatenate([[7], np.arange(n), np.arange(60)]).astype(np.int64)
    aval, bval = (rng.choice([-1e-200, 1e-200], k) for k in (len(acrd), len(bcrd)))
    A, B = rt.CsrMatrix.from_arrays((3, n), apos, acrd, aval), rt.CsrMatrix.from_arrays((n, m), bpos, bcrd, bval)
    want = orc.spgemm(apos, acrd, aval, bpos, bcrd, bval, m)
    p, c, v = rt.spgemm(A, B).to_arrays()
    assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
    assert not v.any() and not np.any(np.signbit(v))


@pytest.mark.parametrize("semiring", [None, ("min", "plus"), ("any", "second")])
@pytest.mark.parametrize("ncols", [40, 9000, 65_536])
@pytest.mark.parametrize("times,others", [(1, True), (1, False), (70, True), (70, False)])
def test_spgemm_rows_of_a_product_a_lane(times, others, ncols, semiring):
    # rows around 64 entries and 256 products, entries without products among them, columns that meet and that are stored
    # twice; few and many such rows, alone and beside rows with more products
    rng = np.random.default_rng(ncols + times)
    blens = np.array([0, 0, 1, 1, 1, 2, 3, 4, 5, 8, 17, 33] * 12)
    bcrd = np.concatenate([np.sort(rng.integers(0, ncols, l)) for l in blens]).astype(np.int64)
    bpos = np.concatenate([[0], np.cumsum(blens)]).astype(np.int64)
    k, ones = len(blens), np.flatnonzero(blens == 1)
    rows = [[], [0], [2], [11]]
    for entries in (1, 2, 15, 16, 17, 63, 64, 65, 100):
        rows.append(np.sort(rng.choice(k, entries, replace=False)))
    for products in (63, 64, 65, 127, 128, 129, 255, 256, 257):          # as few entries as make them up, and single ones
        row, left = [], products
        for r in np.argsort(-blens, kind="stable"):
            if 0 < blens[r] <= left and blens[r] > 1:
                row.append(r)
                left -= blens[r]
        rows.append(np.sort(np.concatenate([row, ones[:left]]).astype(np.int64)))
    rows = [r for r in rows if others or blens[np.asarray(r, int)].sum() <= 256] * times
    apos = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    acrd = np.concatenate(rows).astype(np.int64)
    pick = np.array([-3.0, -1.0, 0.5, 1.0, 2.0])
    aval, bval = rng.choice(pick, len(acrd)), rng.choice(pick, len(bcrd))
    A, B = rt.CsrMatrix.from_arrays((len(rows), k), apos, acrd, aval), rt.CsrMatrix.from_arrays((k, ncols), bpos, bcrd, bval)
    want = orc.spgemm(apos, acrd, aval, bpos, bcrd, bval, ncols, semiring=semiring)
    p, c, v = rt.spgemm(A, B, semiring=semiring).to_arrays()
    assert np.array_equal(p, want[0]) and np.array_equal(c, want[1])
    assert np.array_equal(v, want[2])          # quarters of whole numbers: sums are exact


@pytest.mark.parametrize("semiring", [None, ("min", "plus"), ("max", "times"), ("any", "pair")])
def test_spgemm_of_one_entry_and_a_row_with_repeated_columns(semiring, monkeypatch):
    # a row of A with one entry copies its row of B where that is right: columns stored more than once are added up
    monkeypatch.setenv("COMET_HIP_SPGEMM_WIDE", str(1 << 40))
    rng = np.random.default_rng(5)
    m, lens, repeats = 40_000, [600, 9000, 2500, 5000], [16, 1, 2, 1]
    rows = [np.sort(rng.choice(m, l, replace=False)) for l in lens]
    bcrd = np.concatenate([np.repeat(c, r) for c, r in zip(rows, repeats)]).astype(np.int64)
    bpos = np.concatenate([[0], np.cumsum(np.multiply(lens, repeats))]).astype(np.int64)
    apos, acrd = np.array([0, 1, 2, 3, 4, 6, 7]).astype(np.int64), np.array([0, 1, 2, 3, 0, 3, 0]).astype(np.int64)
    pick = np.array([-3.0, -1.0, -0.0, 0.0, 1.0, 2.0])
    aval, bval = rng.choice(pick, len(acrd)), rng.choice(pick, len(bcrd))
    A, B = rt.CsrMatrix.from_arrays((6, 4), apos, acrd, aval), rt.CsrMatrix.from_arrays((4, m), bpos, bcrd, bval)
    want = orc.spgemm(apos, acrd, aval, bpos, bcrd, bval, m, semiring=semiring)
    p, c, v = rt.spgemm(A, B, semiring=semiring).to_arrays()
    assert np.array_equal(p, want[0]) and np.array_equal(c, want[1]) and np.array_equal(v, want[2])


@pytest.mark.parametrize("medium", [False, True])
@pytest.mark.parametrize("K,ldb,ldc,shift,accumulate", [(63, 63, 63, 0, False), (63, 63, 63, 0, True), (17, 53, 40, 0, True),
                                                        (64, 64, 64, 1, False), (64, 65, 67, 0, True), (99, 99, 100, 1, False)])
def test_spmm_sweep_of_rows_that_are_no_multiple_of_16_bytes(K, ldb, ldc, shift, accumulate, medium, monkeypatch):
    # odd widths, odd leading dimensions and addresses 8 bytes off, where B is large enough for the sweep; the last column
    # is a lane's own and its neighbour's; nothing outside C's columns is written, B's last row is the end of its array
    monkeypatch.setenv("COMET_HIP_SPMM_NO_COLUMNS", "1")
    if medium:
        monkeypatch.setenv("COMET_HIP_SPMM_MEDIUM", "1")
    n = 60_000
    pos, crd, val = gen.zipf_csr(n=n, mean=16.0, cap=4096, seed=7)
    crd[-1] = n - 1 if pos[-1] > pos[-2] else crd[-1]
    assert len(crd) >= 1 << 19 and n * ldb * 8 >= 24 << 20
    rng = np.random.default_rng(K)
    B, C0 = rng.uniform(-1, 1, (n, K)), rng.uniform(-1, 1, (n, K))
    flatB, flatC = np.full(shift + (n - 1) * ldb + K, 5.0), np.full(shift + n * ldc, 7.0)
    view = lambda flat, ld: np.lib.stride_tricks.as_strided(flat[shift:], (n, K), (8 * ld, 8))
    view(flatB, ldb)[:] = B
    view(flatC, ldc)[:] = C0
    dB, dC = rt.DeviceArray.from_numpy(flatB), rt.DeviceArray.from_numpy(flatC)
    A = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    rt.profile_reset()
    rt.profile_enable(True)
    for _ in range(1 if accumulate else 2):
        rt._check(rt.lib().comet_hip_spmm_csr_f64(A.handle, K, dB.ptr + 8 * shift, ldb, dC.ptr + 8 * shift, ldc, int(accumulate)), "spmm")
    rt.sync()
    assert "spmm_heavy_sweep" in rt.profile_report()
    rt.profile_enable(False)
    want = orc.spmm(pos, crd, val, B, C0 if accumulate else None)
    bound = orc.spmm(pos, crd, np.abs(val), np.abs(B), np.abs(C0) if accumulate else None)
    out = dC.to_numpy()
    got = view(out, ldc).copy()
    assert np.all(np.abs(got - want) <= 1e-12 * bound)
    assert np.array_equal(got[np.diff(pos) <= 1], want[np.diff(pos) <= 1])
    view(out, ldc)[:] = 7.0
    assert np.all(out == 7.0)


@pytest.mark.parametrize("mean,widths", [(4.0, {17: False, 33: False, 63: False, 64: True}), (8.0, {17: False, 33: True, 63: True, 64: True}),
                                         (16.0, {17: True, 63: True, 64: True})])
def test_spmm_sweeps_odd_widths_where_long_rows_hold_the_matrix(mean, widths, monkeypatch):
    # the plan of a matrix is made by the first call it is right for, whatever calls came before
    monkeypatch.setenv("COMET_HIP_SPMM_NO_COLUMNS", "1")
    n = 200_000
    pos, crd, val = gen.zipf_csr(n=n, mean=mean, cap=4096, seed=7)
    A = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    rng = np.random.default_rng(int(mean))
    for K, swept in widths.items():
        B = rng.uniform(-1, 1, (n, K))
        dB, dC = rt.DeviceArray.from_numpy(B), rt.DeviceArray((n, K))
        rt.profile_reset()
        rt.profile_enable(True)
        rt.spmm(A, dB, dC, accumulate=False)
        rt.sync()
        assert ("spmm_heavy_sweep" in rt.profile_report()) == swept, K
        rt.profile_enable(False)
        bound = orc.spmm(pos, crd, np.abs(val), np.abs(B))
        assert np.all(np.abs(dC.to_numpy() - orc.spmm(pos, crd, val, B)) <= 1e-12 * bound)


def _edges(kind, rng):
    """Pairs of vertices (u > v) and the number of vertices."""
    if kind == "complete":
        n = 70
        u, v = np.tril_indices(n, -1)
    elif kind == "dense":               # rows of more words than a wavefront's table takes
        n = 3400
        u, v = np.tril_indices(n, -1)
        keep = rng.random(len(u)) < 0.9
        u, v = u[keep], v[keep]
    elif kind == "star":                # no triangles, one vertex with all edges
        n = 5000
        u, v = np.arange(1, n), np.zeros(n - 1, np.int64)
    elif kind == "wheel":               # its rim closes one triangle for every vertex
        n = 40_000
        u = np.concatenate([np.arange(1, n), np.arange(2, n), [n - 1]])
        v = np.concatenate([np.zeros(n - 1, np.int64), np.arange(1, n - 1), [1]])
    else:
        n, m, hubs = (*kind, 1)[:3]          # hubs > 1: vertices with many edges, rows much longer than the mean
        u, v = (n * rng.random((2, m)) ** hubs).astype(np.int64) if m else np.zeros((2, 0), np.int64)
        u, v = np.maximum(u, v)[u != v], np.minimum(u, v)[u != v]
    key = np.unique(np.asarray(u, np.int64) * n + v)
    return n, key // n, key % n


@pytest.mark.parametrize("only", [None, "workgroup", "wavefront"])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("kind", ["complete", "dense", "star", "wheel", (1, 0), (2, 1), (15, 60), (16, 90), (17, 100), (33, 300),
                                  (4097, 60_000), (100_003, 900_000), (1 << 20, 2_000_000), ((1 << 20) + 1, 500_000),
                                  (511, 4000, 4), (1025, 30_000, 3), (20_001, 300_000, 4), (1 << 20, 2_000_000, 3)])
def test_triangle_counts_of_every_kind_of_graph(kind, upper, only, monkeypatch):
    # both triangles of the matrix, rows through either kernel, numbers of vertices around a word's and the most that are
    # named in 16 + 4 bits; counts of one handle walk the vertices by their number of edges, a mask of its own walks L as it is
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    if only:
        monkeypatch.setenv("COMET_HIP_MASKED_SUM_ONLY", only)
    rng = np.random.default_rng(7)
    n, u, v = _edges(kind, rng)
    shuffle = rng.permutation(n)
    u, v = np.maximum(shuffle[u], shuffle[v]), np.minimum(shuffle[u], shuffle[v])
    if upper:
        u, v = v, u
    order = np.lexsort((v, u))
    u, v = u[order], v[order]
    pos = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int64)
    L = rt.CsrMatrix.from_arrays((n, n), pos, v.astype(np.int64), np.full(len(u), 0.5))
    if kind == "dense":
        D = np.zeros((n, n))
        D[u, v] = 1.0
        want = float(((D @ D) * D).sum())
    else:
        want = orc.tricount_masked(pos, v.astype(np.int64), np.ones(len(u)))
    assert [rt.triangle_count(L) for _ in range(3)] == [0.25 * want] * 3
    mask = rt.CsrMatrix.from_arrays((n, n), pos, v.astype(np.int64), np.full(len(u), 2.0))
    assert [rt.spgemm_masked_sum(L, L, mask) for _ in range(2)] == [0.25 * want] * 2


@pytest.mark.parametrize("only", [None, "workgroup", "wavefront"])
def test_sums_of_hits_of_any_number_of_workgroups(only, monkeypatch):
    # bands of three: from no workgroup over fewer than eight and remainders to those of a full chip and more rows than that
    if only:
        monkeypatch.setenv("COMET_HIP_MASKED_SUM_ONLY", only)
    for n in [2, 3, 4, 7, 9, 10, 11, 30, 33, 66, 257, 1030, 2051, 9000]:
        u = np.repeat(np.arange(n), 2)
        v = u - np.tile([2, 1], n)
        u, v = u[v >= 0], v[v >= 0]
        pos = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int64)
        L, M = (rt.CsrMatrix.from_arrays((n, n), pos, v.astype(np.int64), np.full(len(u), x)) for x in (0.5, 2.0))
        assert [rt.triangle_count(L), rt.spgemm_masked_sum(L, L, M), rt.triangle_count(L)] == [0.25 * (n - 2)] * 3, n


def test_the_plan_of_triangle_counts_is_made_once_and_where_it_serves(monkeypatch):
    # at the first count and never again, for matrices that are strictly on one side and hold no column twice - the last
    # column of a row and the first of the next may be the same -; the others' sums take the pairs as they are
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    rng = np.random.default_rng(11)
    for what in ("lower", "upper", "star", "diagonal", "both sides", "twice", "last row twice"):
        n, u, v = (700, np.arange(1, 700), np.zeros(699, np.int64)) if what == "star" else _edges((700, 9000), rng)
        if what == "upper":
            u, v = v, u
        extra = {"diagonal": ([5], [5]), "both sides": (v[:1], u[:1]), "twice": (u[100:101], v[100:101]),
                 "last row twice": (u[-1:], v[-1:])}.get(what, ([], []))
        u, v = np.concatenate([u, extra[0]]).astype(np.int64), np.concatenate([v, extra[1]]).astype(np.int64)
        order = np.lexsort((v, u))
        u, v = u[order], v[order]
        pos = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int64)
        L = rt.CsrMatrix.from_arrays((n, n), pos, v, np.ones(len(u)))
        D = np.zeros((n, n))
        np.add.at(D, (u, v), 1.0)
        want = float(((D @ D) * (D > 0)).sum())
        plans = []
        for _ in range(2):
            rt.profile_reset()
            rt.profile_enable(True)
            assert rt.triangle_count(L) == want
            report = rt.profile_report()
            rt.profile_enable(False)
            plans.append([k for k in ("triangle_plan", "spgemm_pair_plan") if k in report])
        renumbered = what in ("lower", "upper", "star")
        assert plans == [["triangle_plan" if renumbered else "spgemm_pair_plan"], []], what


def test_sums_that_are_no_triangle_count_stay_as_they_are():
    # one handle three times, but with a diagonal, with entries on both sides, with a column twice, with more columns than
    # rows of other vertices; and values that change under the handle
    rng = np.random.default_rng(3)
    n, u, v = _edges((300, 6000), rng)
    csr = lambda a, b, val: (np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int64), b.astype(np.int64), val)
    diagonal = np.arange(n)
    for a, b in ((np.concatenate([u, diagonal]), np.concatenate([v, diagonal])), (np.concatenate([u, v]), np.concatenate([v, u])),
                 (np.concatenate([u, u[:50]]), np.concatenate([v, v[:50]]))):
        order = np.lexsort((b, a))
        pos, crd, val = csr(a[order], b[order], np.ones(len(a)))
        L = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
        rows = np.repeat(np.arange(n), np.diff(pos))
        D = np.zeros((n, n))
        np.add.at(D, (rows, crd), 1.0)
        want = float(((D @ D) * (D > 0)).sum())
        assert rt.triangle_count(L) == rt.triangle_count(L) == want
    pos, crd, val = csr(u, v, np.ones(len(u)))
    D = np.zeros((n, n))
    D[u, v] = 1.0
    L = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    count = float(((D @ D) * D).sum())
    assert rt.triangle_count(L) == rt.triangle_count(L) == count
    val = rng.integers(1, 4, len(u)).astype(np.float64)
    rt._check(rt.lib().comet_hip_memcpy(L.device_arrays()[2], rt._vptr(val), val.nbytes, 0))
    rt._check(rt.lib().comet_hip_csr_invalidate(L.handle), "invalidate")
    W = np.zeros((n, n))
    W[u, v] = val
    assert rt.triangle_count(L) == rt.triangle_count(L) == float(((W @ W) * D).sum())


def _refusing(k, call):
    """call() with its k-th request for device memory refused."""
    rt.lib().comet_hip_debug_fail_allocations(k, 1)
    try:
        return call()
    finally:
        rt.lib().comet_hip_debug_fail_allocations(0, 0)


def test_a_refused_request_fails_its_own_call_only():
    pos, crd, val = gen.poisson_csr(n=3000, mean=4.0, seed=5)
    A = rt.CsrMatrix.from_arrays((3000, 3000), pos, crd, val)
    for k in range(4):
        with pytest.raises(rt.CometHipError):
            rt.lib().comet_hip_debug_fail_allocations(k, 100)
            try:
                rt.spgemm(A, A)
            finally:
                rt.lib().comet_hip_debug_fail_allocations(0, 0)
        B = rt.CsrMatrix.from_arrays((3000, 3000), pos, crd, val)          # copies and launches look at what failed before
        assert np.array_equal(B.to_arrays()[2], val)
    assert rt.spgemm(A, A).nnz == rt.spgemm(B, A).nnz > 0


@pytest.mark.parametrize("op,K", [("spmm", 64), ("spmm", 81), ("sweep", 64), ("sweep", 81), ("spmv", 1), ("sddmm", 40)])
def test_a_plan_without_memory_is_done_without(op, K, monkeypatch):
    # the second call on a handle makes its plan; where that finds no memory the call goes the way of the first
    monkeypatch.delenv("COMET_HIP_PLAN_AT_ONCE")
    if op == "sweep":                     # the long rows' lists in place of the chunks by columns
        monkeypatch.setenv("COMET_HIP_SPMM_NO_COLUMNS", "1")
        op = "spmm"
    n = 700_001 if op == "spmv" else 40_001
    pos, crd, val = (gen.poisson_csr(n=n, mean=3.0, seed=5) if op == "spmv" else gen.zipf_csr(n=n, mean=16.0, cap=4096, seed=7))
    rng = np.random.default_rng(2)
    x = rng.uniform(-1, 1, n) if op == "spmv" else rng.uniform(-1, 1, (n, K))
    dx = rt.DeviceArray.from_numpy(x)
    dt = rt.DeviceArray.from_numpy(np.ascontiguousarray(x.T)) if op == "sddmm" else None
    out = rt.DeviceArray(len(crd) if op == "sddmm" else x.shape)

    def call(A):
        if op == "spmv":
            rt.spmv(A, dx, out, accumulate=False)
        elif op == "spmm":
            rt.spmm(A, dx, out, accumulate=False)
        else:
            rt.sddmm(A, dx, dt, out_values=out)
        return out.to_numpy()

    def plans():
        A = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
        return A, call(A)

    A, want = plans()
    planned = call(A)                       # what the library keeps for all matrices is there
    bound = {"spmv": lambda: orc.spmv(pos, crd, np.abs(val), np.abs(x)), "spmm": lambda: orc.spmm(pos, crd, np.abs(val), np.abs(x)),
             "sddmm": lambda: np.abs(want)}[op]()
    assert np.all(np.abs(planned - want) <= 1e-12 * bound)
    for k in range(24):
        A, first = plans()
        assert np.array_equal(first, want)
        got = _refusing(k, lambda: call(A))
        assert np.all(np.abs(got - want) <= 1e-12 * bound), k
        assert np.all(np.abs(call(A) - want) <= 1e-12 * bound), k


def test_a_sweep_without_room_for_its_sums_is_done_without(monkeypatch):
    # a planned matrix meets a wider B than any before: scratch for the sums, and for the chunk kernel, is refused in turn
    monkeypatch.setenv("COMET_HIP_SPMM_NO_COLUMNS", "1")          # the first product plans the sweep
    n = 40_001
    pos, crd, val = gen.zipf_csr(n=n, mean=16.0, cap=4096, seed=7)
    A = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    rng = np.random.default_rng(2)
    rt.spmm(A, rt.DeviceArray.from_numpy(rng.uniform(-1, 1, (n, 16))))
    for k, K in ((0, 2040), (1, 2046), (0, 2048)):
        few = rng.integers(0, K, 8)
        x = np.zeros((n, K))
        x[:, few] = rng.uniform(-1, 1, (n, len(few)))
        dx, out = rt.DeviceArray.from_numpy(x), rt.DeviceArray((n, K))
        _refusing(k, lambda: rt.spmm(A, dx, out, accumulate=False))
        got = out.to_numpy()
        bound = orc.spmm(pos, crd, np.abs(val), np.abs(x[:, few]))
        assert np.all(np.abs(got[:, few] - orc.spmm(pos, crd, val, x[:, few])) <= 1e-12 * bound)
        got[:, few] = 0.0
        assert not got.any()


def test_an_sddmm_without_room_for_whole_lines_takes_its_rows_packed():
    m, n, K = 50, 5_000_000, 9          # D turned over in lines of 128 bytes: 640 MB, packed 360
    rng = np.random.default_rng(4)
    crd = np.sort(rng.choice(n, (m, 40), replace=False), axis=1).ravel().astype(np.int64)
    pos = np.arange(0, 40 * m + 1, 40).astype(np.int64)
    val = rng.uniform(-1, 1, len(crd))
    C0, D = rng.uniform(-1, 1, (m, K)), rng.uniform(-1, 1, (K, n))
    S = rt.CsrMatrix.from_arrays((m, n), pos, crd, val)
    dC, dD, out = rt.DeviceArray.from_numpy(C0), rt.DeviceArray.from_numpy(D), rt.DeviceArray(len(crd))
    _refusing(0, lambda: rt.sddmm(S, dC, dD, out_values=out))
    rows = np.repeat(np.arange(m), 40)
    want = np.zeros(len(crd))
    for k in range(K):
        want += C0[rows, k] * D[k, crd]
    got = out.to_numpy()
    assert np.all(np.abs(got - val * want) <= 1e-14 * K)


def test_a_plan_without_memory_is_done_without_triangle_count():
    n, u, v = _edges((60_001, 900_000), np.random.default_rng(5))
    pos = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int64)
    new = lambda: rt.CsrMatrix.from_arrays((n, n), pos, v, np.ones(len(u)))
    want = orc.tricount_masked(pos, v, np.ones(len(u)))
    assert rt.triangle_count(new()) == want          # what the library keeps for all matrices is there
    for k in range(20):
        L = new()
        assert _refusing(k, lambda: [rt.triangle_count(L) for _ in range(3)]) == [want] * 3, k


def test_parts_by_stretches_are_done_without_where_they_find_no_memory():
    # of what the plan of a masked product asks for, the parts by stretches (lists of more than 14 MiB) are no condition of it
    n = 4000
    rng = np.random.default_rng(5)
    crd = np.sort(rng.random((n, n)).argsort(1)[:, :330], axis=1).astype(np.int32).ravel()
    pos, val = np.arange(n + 1, dtype=np.int64) * 330, rng.integers(1, 9, n * 330).astype(float)
    assert len(crd) * 12 > 14 << 20
    new = lambda: rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
    mask = np.arange(0, n + 1, dtype=np.int64) * 40, np.tile(np.arange(0, n, 100, dtype=np.int32), n), np.ones(40 * n)
    M = rt.CsrMatrix.from_arrays((n, n), *mask)
    want = orc.spgemm(pos, crd, val, pos, crd, val, n, mask=mask[:2])
    rt.spgemm(new(), new(), M)          # what the library keeps for all matrices is there
    served = []
    for k in range(40):
        A, B = new(), new()
        try:
            got = _refusing(k, lambda: rt.spgemm(A, B, M)).to_arrays()
            served.append(True)
            assert all(np.array_equal(g, w) for g, w in zip(got, want)), k
        except rt.CometHipError:
            served.append(False)
    last = max(k for k in range(40) if not served[k])
    assert last < 39 and 1 <= sum(served[:last]) <= 2, served          # one for each side of the plan that has such parts


@pytest.mark.parametrize("long_rows", [0, 3])
def test_what_a_structure_keeps_is_for_rows_that_are_long(long_rows):
    # bitmaps of rows with a 64th of the columns: for as many as there are, and nothing for a matrix without
    n = 20_000
    rng = np.random.default_rng(1)
    lengths = rng.integers(60, 100, n)
    lengths[:long_rows] = n // 64 + 1
    crd = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lengths]).astype(np.int64)
    pos = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    val = np.ones(len(crd))

    def free():
        rt.sync()
        rt.release_memory()
        got = [C.c_int64(), C.c_int64()]
        rt._check(rt.lib().comet_hip_mem_info(*map(C.byref, got)))
        return got[0].value

    kept = []
    for _ in range(2):              # the first of them brings up what the library keeps for all matrices
        A = rt.CsrMatrix.from_arrays((n, n), pos, crd, val)
        before = free()
        dpos, nnz = rt.spgemm_symbolic(A, A)
        counts = np.diff(dpos.to_numpy())
        dpos.free()
        kept.append(before - free())
    assert kept[1] < len(crd), kept
    import scipy.sparse as sp
    S = sp.csr_matrix((val, crd, pos), shape=(n, n))
    want = (S[:200] @ S).astype(bool)
    assert np.array_equal(counts[:200], np.diff(want.indptr))
