"""Columns below 0 that are not the ELL padding: the conversions to COO carry
such entries through their sort (no entry loses its indices), in the order of
the row and then of the column's low bits, as many as the largest column has,
rounded up to a multiple of 4; a list already in order stays as it is."""
import ctypes as C

import numpy as np
import pytest

from morpheus_amd import capi, device

pytestmark = pytest.mark.gpu


def _p(t):
    return C.c_void_p(t.data_ptr()) if t.numel() else None


def _dev(a, dtype):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)).cuda()


def _sorted(ri, ci, v):
    """What the sort makes of the entries ri, ci, v."""
    order = list(zip(ri.tolist(), ci.tolist()))
    if order == sorted(order):
        return ri, ci, v
    bits = -(-int(max(ci.max(), 0)).bit_length() // 4) * 4
    at = np.lexsort((ci & ((1 << bits) - 1), ri))  # stable
    return ri[at], ci[at], v[at]


def _expect(got, ri, ci, v):
    for g, e in zip(got, _sorted(ri, ci, v)):
        np.testing.assert_array_equal(g.cpu().numpy(), e)


def _out(nnz):
    return [_dev(np.full(nnz, 77), t) for t in (np.int32, np.int32, np.float64)]


def _rows(nrows, width, ncols, stray, seed):
    """width columns a row, ascending, and the columns of `stray` put in."""
    rng = np.random.default_rng(seed)
    ci = np.sort(rng.choice(ncols, (nrows, width)), axis=1)
    for r, s, c in stray:
        ci[r, s] = c
    return ci


STRAY = {
    "first slot, in order": [(3, 0, -5)],
    "a later slot": [(3, 2, -5)],
    "several": [(3, 2, -5), (3, 3, -2), (70, 1, -2147483648), (199, 3, -77)],
}


@pytest.mark.parametrize("stray", list(STRAY))
@pytest.mark.parametrize("ncols", [3, 100, 5000])
def test_ell(gpu, stray, ncols):
    nrows, width = 200, 4
    ci = _rows(nrows, width, ncols, STRAY[stray], 1)
    v = 1.0 + np.arange(nrows * width).reshape(nrows, width)
    out = _out(ci.size)
    e = [_dev(ci.T.ravel(), np.int32), _dev(v.T.ravel(), np.float64)]
    capi.call("mph_convert_ell_to_coo", nrows, ci.size, width, nrows, _p(e[0]), _p(e[1]), capi.F64,
              *map(_p, out), device.stream_handle())
    _expect(out, np.repeat(np.arange(nrows), width), ci.ravel(), v.ravel())


@pytest.mark.parametrize("stray", list(STRAY))
def test_hyb_tail(gpu, stray):
    """The ELL part's first two slots, the rest in the COO part."""
    nrows, width = 200, 4
    ci = _rows(nrows, width, 100, STRAY[stray], 2)
    v = 1.0 + np.arange(nrows * width).reshape(nrows, width)
    rows = np.repeat(np.arange(nrows), 2)
    out = _out(ci.size)
    e = [_dev(ci[:, :2].T.ravel(), np.int32), _dev(v[:, :2].T.ravel(), np.float64)]
    t = [_dev(rows, np.int32), _dev(ci[:, 2:].ravel(), np.int32),
         _dev(v[:, 2:].ravel(), np.float64)]
    capi.call("mph_convert_hyb_to_coo", nrows, ci.size, 2, nrows, _p(e[0]), _p(e[1]), rows.size,
              *map(_p, t), capi.F64, *map(_p, out), device.stream_handle())
    _expect(out, np.repeat(np.arange(nrows), width), ci.ravel(), v.ravel())


@pytest.mark.parametrize("stray", list(STRAY))
@pytest.mark.parametrize("diagonal", [False, True])
def test_hdc_csr_part(gpu, stray, diagonal):
    nrows, width = 200, 4
    ci = _rows(nrows, width, nrows, STRAY[stray], 3)
    v = 1.0 + np.arange(nrows * width).reshape(nrows, width)
    ro = _dev(np.arange(nrows + 1) * width, np.int32)
    c = [_dev(ci.ravel(), np.int32), _dev(v.ravel(), np.float64)]
    d = [_dev([0], np.int32), _dev(-1.0 - np.arange(nrows), np.float64)]
    nd = nrows if diagonal else 0
    out = _out(ci.size + nd)
    capi.call("mph_convert_hdc_to_coo", nrows, nrows, ci.size + nd, 1 if diagonal else 0, nrows,
              _p(d[0]), _p(d[1]), ci.size, _p(ro), _p(c[0]), _p(c[1]), capi.F64, *map(_p, out),
              device.stream_handle())
    # the DIA part's entries, then the CSR part's
    diag = np.arange(nd)
    _expect(out, np.r_[diag, np.repeat(np.arange(nrows), width)], np.r_[diag, ci.ravel()],
            np.r_[-1.0 - diag, v.ravel()])
