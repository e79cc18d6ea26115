"""The 16-byte loads of dot and the CG iteration: sizes around their batches
(256 threads, 4 pieces of 16 bytes) and arrays that do not start on 16 bytes,
which take the element loads: the same sums and the same iterates."""
import numpy as np
import pytest

import oracle
from morpheus_amd import device
from morpheus_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 2047, 2049, 4097, 1024 * 2048 + 5])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shift", [0, 1])
def test_dot(gpu, n, dtype, shift):
    import torch
    vd = device.vector_dtype(dtype)
    rng = np.random.default_rng(n)
    x, y = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    xt, yt = (torch.zeros(n + shift, dtype=vd, device="cuda") for _ in range(2))
    xt[shift:] = torch.from_numpy(x).cuda().to(vd)
    yt[shift:] = torch.from_numpy(y).cuda().to(vd)
    xs, ys = xt[shift:].double().cpu().numpy(), yt[shift:].double().cpu().numpy()
    got = device.dot(xt[shift:], yt[shift:])
    # n products summed in FP64 in any order
    assert abs(got - oracle.dot(xs, ys)) <= 2 * n * 2.0 ** -53 * np.abs(xs * ys).sum()


@pytest.mark.parametrize("g", [3, 11, 23])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_cg_unaligned_x(gpu, g, dtype):
    import torch
    A = device.to_device(gen.stencil3d_7(g), dtype)
    n = A.nrows
    vd = device.vector_dtype(dtype)
    b = torch.from_numpy(gen.random_vector(n, g)).cuda().to(vd)
    out = []
    for shift in (0, 1):
        buf = torch.zeros(n + shift, dtype=vd, device="cuda")
        x = buf[shift:]
        cg = device.CG(A)
        cg.start(b, x)
        cg.iterate(x, 2)
        cg.iterate(x, 3)
        out.append((x.clone(), cg.residual()))
    assert torch.equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    x = out[0][0].double().cpu().numpy()
    r = b.double().cpu().numpy() - oracle.spmv(gen.stencil3d_7(g), x)
    # the updated residual drifts from b - A x by a few roundings an iteration
    u = 2.0 ** -53 if dtype == "f64" else 2.0 ** -24
    scale = 12.0 * np.linalg.norm(x) + np.linalg.norm(b.double().cpu().numpy())
    assert abs(np.sqrt(out[0][1]) - np.linalg.norm(r)) <= 40 * u * scale
