"""Conversions at the edges of their kernels' tiles (64 rows, 256 threads, 2048
entries, 32 slots a batch), bit-exact against the CPU oracle: entry counts and
row counts around the tiles, long runs of empty rows, repeated and unsorted
entries, diagonals in any order and repeated, sizes that leave phantom slots."""
import ctypes as C

import numpy as np
import pytest

import oracle
from morpheus_amd import capi, device
from morpheus_amd.formats import (COO_FORMAT, CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HDC_FORMAT,
                                  HYB_FORMAT, Coo, Dia)
from tests.helpers import same_container
from tests.test_convert_gpu import gpu_convert, round_values

pytestmark = pytest.mark.gpu

COO_TARGETS = [CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HYB_FORMAT, HDC_FORMAT]


def _check(A, fmt, dtype="f64"):
    A = round_values(A, dtype)
    try:
        ref = oracle.from_coo(A, fmt) if isinstance(A, Coo) else oracle.convert(A, fmt)
    except oracle.FormatConversion:
        return
    assert same_container(gpu_convert(A, fmt, dtype), ref), fmt


def _entries(nrows, ncols, nnz, seed, band=None):
    """nnz distinct entries in (row, column) order, values 1, 2, ..."""
    rng = np.random.default_rng(seed)
    if band is None:
        key = np.sort(rng.choice(nrows * ncols, size=nnz, replace=False))
    else:
        r, o = rng.integers(0, nrows, 4 * nnz), rng.integers(-band, band + 1, 4 * nnz)
        ok = (r + o >= 0) & (r + o < ncols)
        key = np.unique(r[ok] * ncols + r[ok] + o[ok])[:nnz]
    return Coo(nrows, ncols, key // ncols, key % ncols, 1.0 + np.arange(key.size))


@pytest.mark.parametrize("nnz", [1, 2, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 4097])
@pytest.mark.parametrize("fmt", COO_TARGETS)
def test_entry_counts(gpu, nnz, fmt):
    _check(_entries(120, 120, nnz, nnz), fmt)
    A = _entries(120, 120, nnz, nnz)
    back = oracle.convert(oracle.from_coo(A, CSR_FORMAT), fmt)
    assert same_container(gpu_convert(oracle.from_coo(A, CSR_FORMAT), fmt), back)
    assert same_container(gpu_convert(back, CSR_FORMAT), oracle.convert(back, CSR_FORMAT))


@pytest.mark.parametrize("nrows", [1, 63, 64, 65, 127, 129, 255, 257, 1000])
@pytest.mark.parametrize("band", [1, 15, 16, 40])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_row_counts_and_slots(gpu, nrows, band, dtype):
    A = _entries(nrows, nrows, max(1, min(nrows * 3, nrows * nrows // 2)), nrows + band, band)
    A.values = (A.values % 200) + 1.0  # exact in BF16
    for fmt in COO_TARGETS:
        _check(A, fmt, dtype)
        try:
            B = oracle.from_coo(A, fmt)
        except oracle.FormatConversion:
            continue
        got = gpu_convert(B, COO_FORMAT, dtype)
        assert same_container(got, oracle.to_coo(B)), fmt


@pytest.mark.parametrize("where", ["first", "middle", "last", "spread"])
def test_long_runs_of_empty_rows(gpu, where):
    n = 90000
    rows = {"first": np.arange(10), "last": n - 1 - np.arange(10)[::-1],
            "middle": np.r_[0, 1, 2, n - 3, n - 2, n - 1],
            "spread": np.arange(0, n, 2500)}[where]
    rows = np.repeat(rows, 3)
    cols = np.tile([0, 5, 9], rows.size // 3)
    A = Coo(n, 12, rows, cols, 1.0 + np.arange(rows.size))
    csr = oracle.from_coo(A, CSR_FORMAT)
    _check(A, CSR_FORMAT)
    assert same_container(gpu_convert(csr, COO_FORMAT), oracle.to_coo(csr))


@pytest.mark.parametrize("order", ["repeated", "unsorted columns", "unsorted rows"])
@pytest.mark.parametrize("fmt", COO_TARGETS)
def test_repeated_and_unsorted_entries(gpu, order, fmt):
    A = _entries(300, 300, 2100, 7, 4)
    rng = np.random.default_rng(3)
    at = np.arange(A.nnz)
    if order == "repeated":
        at = np.sort(np.r_[at, rng.integers(0, A.nnz, 200)])
    elif order == "unsorted columns":
        at = np.lexsort((rng.random(A.nnz), A.row_indices))
    else:
        at = rng.permutation(A.nnz)
    B = Coo(300, 300, A.row_indices[at], A.column_indices[at], 1.0 + np.arange(at.size))
    _check(B, fmt)


@pytest.mark.parametrize("offsets", [[5, -3, 0, 2, -70], [0, 0, 1], [-1, 2, -1, 0, 2],
                                     list(range(20, -21, -1))])
@pytest.mark.parametrize("extra", [0, 3])
def test_dia_in_any_order(gpu, offsets, extra):
    """Diagonals unsorted or repeated; nnz above the stored non-zeros leaves
    phantom entries."""
    n, pitch = 130, 160
    rng = np.random.default_rng(9)
    v = rng.integers(-2, 3, size=(len(offsets), pitch)).astype(float)
    v[:, ::7] = -0.0
    v[:, n:] = 0.0
    off = np.array(offsets, dtype=np.int32)
    inside = (np.arange(pitch)[None, :] + off[:, None] >= 0) & \
        (np.arange(pitch)[None, :] + off[:, None] < n)
    nnz = int(np.count_nonzero(v * inside)) + extra
    A = Dia(n, n, nnz, off, v.reshape(-1), pitch)
    assert same_container(gpu_convert(A, COO_FORMAT), oracle.to_coo(A))


@pytest.mark.parametrize("nnz", [2, 64, 511, 513, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("nrows,ncols", [(1, 1), (2, 300), (257, 255), (70000, 3), (3, 1 << 24),
                                         (1 << 22, 1 << 23)])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_sort_tiles_and_key_widths(gpu, nnz, nrows, ncols, dtype):
    """The COO sort around its tiles of 4096 and over 0 to 45 key bits; equal
    keys keep their order."""
    import ctypes as C
    import torch
    from morpheus_amd import capi, device
    rng = np.random.default_rng(nnz + nrows)
    r = rng.integers(0, nrows, nnz).astype(np.int32)
    c = rng.integers(0, ncols, nnz).astype(np.int32)
    v = (np.arange(nnz) % 251).astype(float)
    ref = oracle.sort_by_row_and_column(Coo(nrows, ncols, r, c, v))
    tr, tc = torch.from_numpy(r).cuda(), torch.from_numpy(c).cuda()
    tv = torch.from_numpy(v).cuda().to(device.DTYPES[dtype][0])
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    capi.call("mph_coo_sort_by_row_and_column", nnz, p(tr), p(tc), p(tv),
              capi.VALUE_TYPES[dtype], device.stream_handle())
    assert np.array_equal(tr.cpu().numpy(), ref.row_indices)
    assert np.array_equal(tc.cpu().numpy(), ref.column_indices)
    assert np.array_equal(tv.double().cpu().numpy(), ref.values)


@pytest.mark.parametrize("nnz", [3, 4096, 5000])
def test_unsorted_coo_to_csr_in_place(gpu, nnz):
    """ci_out / v_out may be the input's: rows not in order are sorted in place."""
    import ctypes as C
    import torch
    from morpheus_amd import capi, device
    rng = np.random.default_rng(nnz)
    A = Coo(400, 700, rng.integers(0, 400, nnz), rng.integers(0, 700, nnz), 1.0 + np.arange(nnz))
    ref = oracle.from_coo(A, CSR_FORMAT)
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    ri, ci, v = i32(A.row_indices), i32(A.column_indices), torch.from_numpy(A.values).cuda()
    ro = torch.empty(401, dtype=torch.int32, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    capi.call("mph_convert_coo_to_csr", 400, nnz, p(ri), p(ci), p(v), capi.F64, p(ro), p(ci),
              p(v), device.stream_handle())
    assert np.array_equal(ro.cpu().numpy(), ref.row_offsets)
    assert np.array_equal(ci.cpu().numpy(), ref.column_indices)
    assert np.array_equal(v.cpu().numpy(), ref.values)


@pytest.mark.parametrize("nnz", [0, 1])
def test_is_sorted_reads_no_pair(gpu, nnz):
    """One entry is sorted; its arrays are not looked at."""
    out = C.c_int(-1)
    capi.call("mph_coo_is_sorted", nnz, None, None, C.byref(out), device.stream_handle())
    assert out.value == 1


@pytest.mark.parametrize("nrows", [4096 * 2048 - 1, 4096 * 2048, 4096 * 2048 + 1,
                                   3 * 4096 * 2048 + 7])
def test_long_scans(gpu, nrows):
    """Row positions about the longest prefix sum that takes two launches
    (4096 tiles of 2048 counts), and well past it."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(nrows)
    ci = torch.randint(-1, 3, (nrows,), dtype=torch.int32, device="cuda", generator=g)
    ci[-1] = 1
    v = torch.rand(nrows, device="cuda", generator=g)
    rows = torch.nonzero(ci >= 0).reshape(-1)
    ri, co = (torch.empty(rows.numel(), dtype=torch.int32, device="cuda") for _ in range(2))
    vo = torch.empty(rows.numel(), device="cuda")
    capi.call("mph_convert_ell_to_coo", nrows, rows.numel(), 1, nrows, ci.data_ptr(), v.data_ptr(),
              capi.F32, ri.data_ptr(), co.data_ptr(), vo.data_ptr(), device.stream_handle())
    assert torch.equal(ri, rows.int()) and torch.equal(co, ci[rows]) and torch.equal(vo, v[rows])


@pytest.mark.parametrize("gap", [31, 32, 33, 95, 1023, 1024, 1025, 2048, 7000])
@pytest.mark.parametrize("where", ["first", "middle", "last", "all"])
@pytest.mark.parametrize("fmt", [CSR_FORMAT, HYB_FORMAT, HDC_FORMAT])
def test_gaps_between_rows(gpu, gap, where, fmt):
    """Rows without entries about the lengths up to which the scan of the
    entries fills their offsets by lanes (32) and by waves (1024 rows), and of
    the tiles that are filled afterwards (2048)."""
    lead, mid, tail = (gap if where in (w, "all") else 0 for w in ("first", "middle", "last"))
    a = lead + np.arange(300)
    rows = np.r_[a, a[-1] + 1 + mid + np.arange(40)]
    n = rows[-1] + 1 + tail
    rows = np.repeat(rows, 1 + np.arange(rows.size) % 4 // 3)
    cols = (np.arange(rows.size) * 37) % n
    A = Coo(n, n, rows, cols, 1.0 + np.arange(rows.size))
    at = np.lexsort((A.column_indices, A.row_indices))
    A = Coo(n, n, rows[at], cols[at], A.values[at])
    _check(A, fmt)
    perm = np.random.default_rng(gap).permutation(rows.size)
    _check(Coo(n, n, A.row_indices[perm], A.column_indices[perm], A.values[perm]), fmt)


@pytest.mark.parametrize("order", ["shuffled", "runs", "ends"])
def test_offsets_take_time_by_entries_and_rows(gpu, order):
    """Rows in no order, in many ascending runs, and at both ends of a long
    matrix: a scan that fills the rows between an entry and the one before it
    took 8 to 240 ms."""
    import torch
    n, nnz = 4_000_000, 2_000_000
    g = torch.Generator(device="cuda").manual_seed(1)
    ri = torch.randint(0, n, (nnz,), dtype=torch.int32, device="cuda", generator=g).sort().values
    if order == "shuffled":
        ri = ri[torch.randperm(nnz, device="cuda", generator=g)]
    elif order == "runs":
        ri = ri.reshape(-1, 64).t().reshape(-1).contiguous()
    else:
        ri = torch.cat([ri[:500] % 500, n - 1 - ri[:500] % 500]).sort().values
    A = device.DeviceMatrix(COO_FORMAT, n, n, ri.numel(), "f64",
                            dict(ri=ri, ci=ri.clone(), v=ri.double()), {})
    ms = []
    for _ in range(4):
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        t[0].record()
        B = device.from_coo(A, CSR_FORMAT)
        t[1].record()
        t[1].synchronize()
        ms.append(t[0].elapsed_time(t[1]))
    ro = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ro[1:] = torch.cumsum(torch.bincount(ri.long(), minlength=n), 0)
    assert torch.equal(B.arrays["ro"], ro.int())
    assert torch.equal(B.arrays["v"], ri.sort(stable=True).values.double())
    assert min(ms) < (1.2 if order == "ends" else 4)


def _wide(nrows, per, ncols, seed):
    """`per` distinct columns a row (fewer in every third row), in order."""
    rng = np.random.default_rng(seed)
    lens = [per - (per // 2 if r % 3 == 1 else 0) for r in range(nrows)]
    cols = [np.sort(rng.choice(ncols, n, replace=False)) for n in lens]
    rows = np.repeat(np.arange(nrows), lens)
    return Coo(nrows, ncols, rows, np.concatenate(cols), 1.0 + np.arange(rows.size) % 200)


@pytest.mark.parametrize("nrows", [1, 2, 7, 63, 64, 65, 130])
@pytest.mark.parametrize("per", [224, 256, 257, 480, 513, 1100])
@pytest.mark.parametrize("dtype", ["f64", "bf16"])
def test_long_rows(gpu, nrows, per, dtype):
    """Few rows of many slots and diagonals: segments of 256, their ends, rows
    fewer than a wave's lanes and more."""
    A = _wide(nrows, per, 1300, nrows + per)
    for fmt in COO_TARGETS:
        try:
            B = oracle.from_coo(round_values(A, dtype), fmt)
        except oracle.OracleError:  # (HDC's midpoint on some shapes that are not square)
            continue
        _check(A, fmt, dtype)
        _check(B, COO_FORMAT, dtype)


@pytest.mark.parametrize("nrows", [3, 70])
def test_long_rows_with_holes(gpu, nrows):
    """ELL slots left empty before, inside and after a segment's start, and
    columns that step back where the empty slots hide the one before."""
    import torch
    rng = np.random.default_rng(nrows)
    width = 900
    ci = np.sort(rng.choice(5000, (nrows, width)), axis=1).astype(np.int32)
    ci[0, 100:400] = -1
    ci[1, 250:260] = -1
    ci[2, 256:] = -1
    ci[nrows - 1, 300] = 4999
    v = 1.0 + np.arange(nrows * width).reshape(nrows, width)
    keep = ci.ravel() >= 0
    rows = np.repeat(np.arange(nrows), width)[keep]
    cols, vals = ci.ravel()[keep], v.ravel()[keep]
    at = np.lexsort((cols, rows))  # stable
    e = [torch.from_numpy(np.ascontiguousarray(a.T.ravel())).cuda() for a in (ci, v)]
    out = [torch.empty(rows.size, dtype=t, device="cuda")
           for t in (torch.int32, torch.int32, torch.float64)]
    capi.call("mph_convert_ell_to_coo", nrows, rows.size, width, nrows, e[0].data_ptr(),
              e[1].data_ptr(), capi.F64, *(t.data_ptr() for t in out), device.stream_handle())
    for got, want in zip(out, (rows[at], cols[at], vals[at])):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("order", ["ascending", "descending", "repeated"])
@pytest.mark.parametrize("ndiag", [255, 256, 257, 512, 513, 9000])
def test_many_diagonals(gpu, ndiag, order):
    """Offsets whose order is looked at on the host and on the device."""
    n = 20
    off = np.arange(ndiag) - 10
    if order == "descending":
        off = off[::-1]
    elif order == "repeated":
        off = np.sort(off // 2)
        off[[5, 9]] = off[[9, 5]]
    pitch = 32
    val = np.zeros(pitch * ndiag)
    for r in range(n):
        d = np.arange(r, ndiag, 3)
        d = d[(r + off[d] >= 0) & (r + off[d] < ndiag)]
        val[d * pitch + r] = 1.0 + (d * 7 + r) % 250
    D = Dia(n, ndiag, int(np.count_nonzero(val)), off.astype(np.int32), val, pitch)
    _check(D, COO_FORMAT)


@pytest.mark.parametrize("nrows,ncols", [(1, 2_000_000), (4, 500_000), (100, 20_000)])
def test_long_rows_take_time_by_entries(gpu, nrows, ncols):
    """A full matrix of a few long rows: a lane, thread or workgroup for each
    took 1.5 to 500 ms a conversion."""
    import torch
    nnz = nrows * ncols
    at = torch.arange(nnz, device="cuda")
    A = device.DeviceMatrix(COO_FORMAT, nrows, ncols, nnz, "f64",
                            dict(ri=(at // ncols).int(), ci=(at % ncols).int(),
                                 v=1.0 + (at % 1000).double()), {})
    for fmt in (DIA_FORMAT, ELL_FORMAT, HYB_FORMAT):
        try:
            B = device.from_coo(A, fmt)
        except capi.FormatConversionException:
            continue
        for f in (lambda: device.from_coo(A, fmt), lambda: device.to_coo(B)):
            ms = []
            for _ in range(4):
                t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                t[0].record()
                C2 = f()
                t[1].record()
                t[1].synchronize()
                ms.append(t[0].elapsed_time(t[1]))
            limit = 6 if fmt == DIA_FORMAT else 1.2
            assert min(ms) < limit, (fmt, ms)
        assert all(torch.equal(C2.arrays[k], A.arrays[k]) for k in ("ri", "ci", "v"))
