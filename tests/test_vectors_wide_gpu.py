"""The 16-byte loads of dot and the CG iteration.  A block's chunk is loaded in
batches of 256 threads x 4 pieces of 16 bytes (2048 elements in FP64, 4096 in
FP32), what is left of it one element at a time: small sizes, all of them by
elements, then chunks of 4 elements less than a batch, a batch, 4 more, and
two batches and a rest, in both types, with arrays that start on 16 bytes and
arrays that do not: the same bits."""
import numpy as np
import pytest

import oracle
from morpheus_amd import device
from morpheus_amd import generators as gen
from morpheus_amd.formats import DIA_FORMAT

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


BATCH = {"f64": 2048, "f32": 4096}


def _chunk(n):
    """A block's elements, as the library cuts a vector of n."""
    parts = max(1, min(1024, -(-n // 2048)))
    return -(-(-(-n // parts)) // 4) * 4


def _size(dtype, chunk):
    """A vector whose blocks take `chunk` elements, the last one fewer."""
    n = 1024 * chunk - 5 if chunk >= 2048 else 500_000
    assert _chunk(n) == chunk
    return n


CHUNKS = [(dt, c) for dt, b in BATCH.items() for c in (b - 4, b, b + 4, 2 * b + 12)]


@pytest.mark.parametrize("dtype,chunk", CHUNKS)
def test_dot_batches(gpu, dtype, chunk):
    import torch
    n = _size(dtype, chunk)
    vd = device.vector_dtype(dtype)
    g = torch.Generator(device="cuda").manual_seed(chunk)
    x, y = (torch.rand(n, dtype=torch.float64, device="cuda", generator=g).mul_(2).sub_(1).to(vd)
            for _ in range(2))
    got = []
    for at in ((0, 0), (1, 0), (1, 1), (3, 2)):
        bufs = [torch.zeros(n + 4, dtype=vd, device="cuda") for _ in at]
        for t, buf, k in zip((x, y), bufs, at):
            buf[k:k + n] = t
        got.append(device.dot(*(buf[k:k + n] for buf, k in zip(bufs, at))))
    assert len(set(got)) == 1
    xs, ys = x.double().cpu().numpy(), y.double().cpu().numpy()
    # n products summed in FP64 in any order
    assert abs(got[0] - oracle.dot(xs, ys)) <= 2 * n * 2.0 ** -53 * np.abs(xs * ys).sum()


@pytest.mark.parametrize("dtype,chunk", CHUNKS)
def test_cg_batches(gpu, dtype, chunk):
    """Three iterations on a tridiagonal matrix (4 and -1) against the same
    recurrence in 64 bits, and x on 16 bytes against x off them."""
    import torch
    n = _size(dtype, chunk)
    vd = device.vector_dtype(dtype)
    off = torch.tensor([-1, 0, 1], dtype=torch.int32, device="cuda")
    pitch = -(-n // 32) * 32
    v = torch.tensor([-1.0, 4.0, -1.0], dtype=vd, device="cuda").repeat_interleave(pitch)
    A = device.DeviceMatrix(DIA_FORMAT, n, n, 3 * n - 2, dtype, dict(off=off, v=v),
                            dict(ndiag=3, pitch=pitch))
    g = torch.Generator(device="cuda").manual_seed(chunk)
    b = torch.rand(n, dtype=torch.float64, device="cuda", generator=g).mul_(2).sub_(1).to(vd)
    out = []
    for shift in (0, 1):
        x = torch.zeros(n + shift, dtype=vd, device="cuda")[shift:]
        cg = device.CG(A)
        cg.start(b, x)
        cg.iterate(x, 3)
        out.append((x, cg.residual()))
    assert torch.equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]

    def product(p):
        q = 4 * p
        q[1:] -= p[:-1]
        q[:-1] -= p[1:]
        return q

    r = b.double()
    x, p, rr = torch.zeros_like(r), r.clone(), r.dot(r)
    for _ in range(3):
        q = product(p)
        alpha = rr / p.dot(q)
        x += alpha * p
        r -= alpha * q
        beta = r.dot(r) / rr
        rr = r.dot(r)
        p = r + beta * p
    # an iteration rounds an element about ten times (three products and sums
    # of q, two of r, x and p each, alpha and beta), values up to max |p| / 3
    # each; the condition number of 3 carries them on
    u = 2.0 ** -53 if dtype == "f64" else 2.0 ** -24
    assert (out[0][0].double() - x).abs().max() <= 3 * 10 * 3 * u * b.abs().max()
    assert abs(out[0][1] - rr) <= 3 * 10 * 3 * u * b.double().dot(b.double())
