"""The staged DIA kernels that request their first values before the x stage
is stored: row counts around the workgroups (256 / 512 rows), diagonals around
a batch (8 / 12), windows around what a thread stages ahead (1024 entries),
bit for bit against the plain kernels."""
import numpy as np
import pytest

from morpheus_amd import generators as gen
from tests.test_dia_staged_gpu import _dia, _product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrows", [1, 2, 255, 257, 511, 512, 513, 1025, 5001])
@pytest.mark.parametrize("ndiag,span", [(8, 7), (9, 512), (12, 30), (13, 511), (25, 48), (40, 500)])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_ahead_equals_plain(gpu, nrows, ndiag, span, dtype):
    offsets = np.unique(np.linspace(-(span // 2), span - span // 2, ndiag).round().astype(int))
    two = np.r_[offsets, offsets + 1500] if ndiag == 9 else offsets  # and two clusters
    D = _dia(nrows, nrows + 40, two, nrows + ndiag)
    x, y0 = gen.random_vector(D.ncols, 1), gen.random_vector(D.nrows, 2)
    for init in (True, False):
        ys = _product(D, x, y0, init, plain=False, dtype=dtype)
        assert np.array_equal(ys, _product(D, x, y0, init, plain=True, dtype=dtype))


@pytest.mark.parametrize("nrows", [1, 511, 513, 5001])
@pytest.mark.parametrize("ndiag", [16, 17, 20, 21])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_ahead_in_two_batches(gpu, nrows, ndiag, dtype):
    """Diagonals about those that take two batches of 12."""
    D = _dia(nrows, nrows + 40, np.arange(-(ndiag // 2), ndiag - ndiag // 2), nrows + ndiag)
    x, y0 = gen.random_vector(D.ncols, 1), gen.random_vector(D.nrows, 2)
    for init in (True, False):
        ys = _product(D, x, y0, init, plain=False, dtype=dtype)
        assert np.array_equal(ys, _product(D, x, y0, init, plain=True, dtype=dtype))
