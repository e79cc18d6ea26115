"""SpMM with a number of columns that is not a power of two: the columns left
after the groups of 16 and 8 take one pass.  Every format against the oracle
per column, over matrices with short rows, rows past a chunk and x-tiled rows,
with and without accumulation."""
import numpy as np
import pytest

import oracle
from morpheus_amd import device
from morpheus_amd import generators as gen
from morpheus_amd.formats import (COO_FORMAT, CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HDC_FORMAT,
                                  HYB_FORMAT)
from tests.helpers import fp64_bound, plain_fp32_bound

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mats():
    return {"grid": gen.stencil3d_7(13), "band": gen.banded(3001, 5, 0.02, seed=3),
            "power law": gen.powerlaw_rows(5003, 5003, 1.5, 12.0, 4000, seed=4)}


CASES = [("grid", f) for f in (CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HYB_FORMAT, HDC_FORMAT)] + \
    [("band", f) for f in (CSR_FORMAT, ELL_FORMAT, HDC_FORMAT)] + \
    [("power law", f) for f in (CSR_FORMAT, COO_FORMAT, HYB_FORMAT)]


@pytest.mark.parametrize("name,fmt", CASES)
@pytest.mark.parametrize("k", [3, 5, 6, 7, 11, 15, 23])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("xtile", [0, 2])
def test_columns(gpu, mats, name, fmt, k, dtype, xtile):
    import torch
    A = mats[name]
    D = device.convert(device.to_device(A, dtype), fmt) if fmt != CSR_FORMAT \
        else device.to_device(A, dtype)
    if xtile:
        if fmt in (DIA_FORMAT, ELL_FORMAT):
            pytest.skip("no x-tiled pass")
        D.set_tuning(xtile=xtile)
    rng = np.random.default_rng(k)
    X = torch.from_numpy(rng.uniform(-1, 1, (A.ncols, k))).cuda().to(device.vector_dtype(dtype))
    Y0 = torch.from_numpy(rng.uniform(-1, 1, (A.nrows, k))).cuda().to(X.dtype)
    Y, Ya = torch.full_like(Y0, float("nan")), Y0.clone()
    D.multiply_multi(X, Y)
    D.multiply_multi(X, Ya, init=False)
    torch.cuda.synchronize()
    vals = torch.from_numpy(A.values).to(device.DTYPES[dtype][0]).double().numpy()
    S = type(A)(A.nrows, A.ncols, A.row_offsets, A.column_indices, vals)
    bound = fp64_bound if dtype == "f64" else plain_fp32_bound
    nrow = np.diff(A.row_offsets)
    Xh, Yh, Yah, Y0h = (t.double().cpu().numpy() for t in (X, Y, Ya, Y0))
    for j in range(k):
        x = np.ascontiguousarray(Xh[:, j])
        ref, scale = oracle.spmv(S, x), oracle.absrow(S, x)
        assert np.all(np.abs(Yh[:, j] - ref) <= bound(nrow, scale)), j
        assert np.all(np.abs(Yah[:, j] - (Y0h[:, j] + ref)) <= bound(nrow + 1, scale + np.abs(Y0h[:, j]))), j
