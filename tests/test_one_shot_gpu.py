"""The one-shot products over raw arrays, whose plan (row blocks, their
records and lane counts) is made and checked on the device: row counts and
row lengths around the blocks' limits (512 rows, 1024 / 2048 entries a chunk,
1024 entries of a compensated FP32 row), against the oracle, and against the
kept handle without the x-tiled pass bit for bit; malformed input refused."""
import ctypes as C

import numpy as np
import pytest

import oracle
from morpheus_amd import capi, device
from morpheus_amd.formats import COO_FORMAT, Csr
from tests.helpers import fp64_bound, plain_fp32_bound

pytestmark = pytest.mark.gpu


def _matrix(lengths, ncols, seed):
    rng = np.random.default_rng(seed)
    cols = [np.sort(rng.choice(ncols, n, replace=False)) for n in lengths]
    ro = np.r_[0, np.cumsum(lengths)]
    ci = np.concatenate(cols) if ro[-1] else np.zeros(0, dtype=np.int64)
    return Csr(len(lengths), ncols, ro, ci, rng.standard_normal(int(ro[-1])))


SHAPES = {
    "one row": [3],
    "empty rows": [0] * 600,
    "511": [2] * 511, "512": [2] * 512, "513": [2] * 513,
    "around a chunk": [1, 1023, 1024, 1025, 0, 2047, 2048, 2049, 7, 4096, 5000, 1, 1],
    "long first": [3000] + [1] * 700, "long last": [1] * 700 + [3000],
    "mixed": [(7 * i * i) % 61 for i in range(3000)],
    "long and empty": ([0] * 40 + [1500]) * 9,
}


def _p(t):
    return C.c_void_p(t.data_ptr()) if t.numel() else None


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("fmt", ["csr", "coo"])
def test_one_shot(gpu, shape, dtype, fmt):
    import torch
    A = _matrix(SHAPES[shape], 6000, len(shape))
    x = np.random.default_rng(1).uniform(-1, 1, A.ncols)
    D = device.to_device(A, dtype)
    if fmt == "coo":
        D = device.convert(D, COO_FORMAT)
    a = D.arrays
    xt = torch.from_numpy(x).cuda().to(device.vector_dtype(dtype))
    y = torch.full((A.nrows,), float("nan"), dtype=xt.dtype, device="cuda")
    first = a["ri"] if fmt == "coo" else a["ro"]
    name = "mph_coo_multiply" if fmt == "coo" else "mph_csr_multiply"
    capi.call(name, A.nrows, A.ncols, A.nnz, _p(first), _p(a["ci"]), _p(a["v"]), D.vt, _p(xt),
              _p(y), 1, device.stream_handle())
    kept = torch.empty_like(y)
    D.set_tuning(xtile=1)
    D.multiply(xt, kept)
    torch.cuda.synchronize()
    assert torch.equal(y, kept)
    stored = Csr(A.nrows, A.ncols, A.row_offsets, A.column_indices, a["v"].double().cpu().numpy())
    xs = xt.double().cpu().numpy()
    ref = oracle.spmv(stored, xs)
    bound = (fp64_bound if dtype == "f64" else plain_fp32_bound)(
        np.diff(stored.row_offsets), oracle.absrow(stored, xs))
    assert np.all(np.abs(y.double().cpu().numpy() - ref) <= bound)


@pytest.mark.parametrize("fault", ["decreasing offsets", "first offset", "last offset",
                                   "column", "negative column"])
def test_malformed_csr_is_refused(gpu, fault):
    import torch
    A = _matrix([4] * 2000, 3000, 2)
    ro, ci = A.row_offsets.astype(np.int32).copy(), A.column_indices.astype(np.int32).copy()
    if fault == "decreasing offsets":
        ro[1000] = ro[1001] + 1
    elif fault == "first offset":
        ro[0] = 1
    elif fault == "last offset":
        ro[-1] -= 1
    else:
        ci[7777] = 3000 if fault == "column" else -1
    t = [torch.from_numpy(v).cuda() for v in (ro, ci, A.values)]
    x = torch.zeros(3000, dtype=torch.float64, device="cuda")
    y = torch.zeros(2000, dtype=torch.float64, device="cuda")
    with pytest.raises(capi.InvalidInputException):
        capi.call("mph_csr_multiply", 2000, 3000, A.nnz, _p(t[0]), _p(t[1]), _p(t[2]), capi.F64,
                  _p(x), _p(y), 1, device.stream_handle())


@pytest.mark.parametrize("nnz", [8001, 2 ** 30])
def test_columns_are_not_read_past_the_offsets(gpu, nnz):
    """An nnz that the row offsets do not end at is refused by them, before a
    column is read: the arrays hold 8000."""
    import torch
    A = _matrix([4] * 2000, 3000, 2)
    ro, ci, v = (torch.from_numpy(a).cuda() for a in (
        A.row_offsets.astype(np.int32), A.column_indices.astype(np.int32), A.values))
    x = torch.zeros(3000, dtype=torch.float64, device="cuda")
    y = torch.zeros(2000, dtype=torch.float64, device="cuda")
    with pytest.raises(capi.InvalidInputException, match="row_offsets"):
        capi.call("mph_csr_multiply", 2000, 3000, nnz, _p(ro), _p(ci), _p(v), capi.F64, _p(x),
                  _p(y), 1, device.stream_handle())
