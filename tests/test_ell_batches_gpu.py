"""ELL products where the slots a row visits end inside, at or just past a
batch of 4 or 8, at row counts around a workgroup and at even and odd pitches:
against the oracle, and one row per thread against two."""
import numpy as np
import pytest

import oracle
from morpheus_amd import device
from morpheus_amd.formats import ELL_FORMAT, Csr
from tests.helpers import fp64_bound, plain_fp32_bound

pytestmark = pytest.mark.gpu


def ragged(n, width, seed):
    """Rows of 0..width entries, at least one row of each extreme."""
    rng = np.random.default_rng(seed)
    cols = max(width, 40)
    lens = rng.integers(0, width + 1, n)
    lens[0] = width
    if n > 1:
        lens[-1] = 0
    ro = np.concatenate([[0], np.cumsum(lens)])
    ci = np.concatenate([np.sort(rng.choice(cols, m, replace=False)) for m in lens])
    return Csr(n, cols, ro.astype(np.int32), ci.astype(np.int32), rng.uniform(-1, 1, ro[-1]))


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 512, 513])
@pytest.mark.parametrize("width", [1, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_batches(gpu, n, width, dtype):
    import torch
    A = ragged(n, width, 100 * n + width)
    D = device.convert(device.to_device(A, dtype), ELL_FORMAT)
    vals = torch.from_numpy(A.values).to(device.DTYPES[dtype][0]).double().numpy()
    S = Csr(A.nrows, A.ncols, A.row_offsets, A.column_indices, vals)
    bound = fp64_bound if dtype == "f64" else plain_fp32_bound
    nrow = np.diff(A.row_offsets)
    rng = np.random.default_rng(width)
    for k in (1, 3):
        X = torch.from_numpy(rng.uniform(-1, 1, (A.ncols, k))).cuda().to(device.vector_dtype(dtype))
        Y0 = torch.from_numpy(rng.uniform(-1, 1, (n, k))).cuda().to(X.dtype)
        if k == 1:
            X, Y0 = X.reshape(-1), Y0.reshape(-1)
        out = []
        for rows in (0, 2):
            D.set_tuning(rows_per_thread=rows)
            Y, Ya = torch.full_like(Y0, float("nan")), Y0.clone()
            mult = D.multiply if k == 1 else D.multiply_multi
            mult(X, Y)
            mult(X, Ya, init=False)
            torch.cuda.synchronize()
            out.append((Y, Ya))
        assert all(torch.equal(p, q) for p, q in zip(*out))
        Xh, Yh, Yah, Y0h = (t.double().cpu().numpy().reshape(-1, k) for t in (X, *out[0], Y0))
        for j in range(k):
            x = np.ascontiguousarray(Xh[:, j])
            ref, scale = oracle.spmv(S, x), oracle.absrow(S, x)
            assert np.all(np.abs(Yh[:, j] - ref) <= bound(nrow, scale))
            assert np.all(np.abs(Yah[:, j] - (Y0h[:, j] + ref))
                          <= bound(nrow + 1, scale + np.abs(Y0h[:, j])))


@pytest.mark.parametrize("n,pitch", [(524_288, 524_288), (524_289, 524_290), (600_001, 600_001),
                                     (917_503, 917_504), (917_505, 917_506)])
@pytest.mark.parametrize("width", [1, 3, 4, 5])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_row_pairs_of_few_slots(gpu, n, pitch, width, dtype):
    """Row counts about the line to the row pairs (2048 workgroups of 256
    rows; 3584 with 4 or 5 slots), even and odd, against two rows per thread."""
    import torch
    rng = torch.Generator(device="cuda").manual_seed(n + width)
    ci = torch.randint(-1, n, (width, pitch), dtype=torch.int32, device="cuda", generator=rng)
    ci[-1, n - 1] = n - 1  # the last row's last slot is filled
    v = torch.rand((width, pitch), device="cuda", generator=rng).to(device.DTYPES[dtype][0])
    D = device.DeviceMatrix(ELL_FORMAT, n, n, width * n, dtype,
                            dict(ci=ci.reshape(-1), v=v.reshape(-1)),
                            dict(K=width, width=width, pitch=pitch))
    x = torch.rand(n, device="cuda", generator=rng)
    y0 = torch.rand(n, device="cuda", generator=rng)
    out = []
    for rows in (0, 2):
        D.set_tuning(rows_per_thread=rows)
        y, ya = torch.full_like(y0, float("nan")), y0.clone()
        D.multiply(x, y)
        D.multiply(x, ya, init=False)
        out.append((y, ya))
    assert all(torch.equal(p, q) for p, q in zip(*out))
    at = ci[:, :n].long()
    ref = torch.where(at >= 0, v[:, :n].double() * x.double()[at.clamp_min(0)], 0.0).sum(0)
    # at most 5 products, rounded once each in FP32
    assert torch.all((out[0][0].double() - ref).abs() <= 2 * 5 * 2.0 ** -24 * ref.abs() + 1e-30)
