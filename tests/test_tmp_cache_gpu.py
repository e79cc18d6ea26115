"""Temporaries shared by the calls of several threads and streams: the same
results as one after another; and given back by mph_finalize."""
import threading

import pytest

from morpheus_amd import capi, device
from morpheus_amd import generators as gen
from morpheus_amd.formats import CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HDC_FORMAT, HYB_FORMAT

pytestmark = pytest.mark.gpu


def test_threads_and_streams(gpu):
    import torch
    jobs = []
    for i, fmt in enumerate((DIA_FORMAT, ELL_FORMAT, HYB_FORMAT, HDC_FORMAT)):
        A = device.to_device(gen.stencil3d_7(11 + 3 * i), "f64")
        B = device.convert(A, fmt)
        jobs.append((A, fmt, {k: t.clone() for k, t in B.arrays.items()}))
    torch.cuda.synchronize()
    wrong = []

    def work(A, fmt, want):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(12):
                    B = device.convert(A, fmt, stream)
                    back = device.convert(B, CSR_FORMAT, stream)
                    stream.synchronize()
                    same = all(torch.equal(B.arrays[k], t) for k, t in want.items())
                    same = same and all(torch.equal(back.arrays[k], t)
                                        for k, t in A.arrays.items())
                    if not same:
                        wrong.append(fmt)
        except Exception as e:  # noqa: BLE001
            wrong.append(e)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_finalize_gives_back(gpu):
    import torch
    n = 4_000_000
    ri = torch.arange(n, device="cuda").flip(0).to(torch.int32)
    ci, v = ri.clone(), ri.double()
    capi.call("mph_finalize")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    capi.call("mph_coo_sort_by_row_and_column", n, ri.data_ptr(), ci.data_ptr(), v.data_ptr(),
              capi.F64, device.stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(ri, torch.arange(n, dtype=torch.int32, device="cuda"))
    del ri, ci, v
    held = free - torch.cuda.mem_get_info()[0]
    capi.call("mph_finalize")
    # keys and values twice: 32 bytes an entry
    assert held >= 32 * n and free - torch.cuda.mem_get_info()[0] < 16 * n
