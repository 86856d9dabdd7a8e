"""A copy over the link leaves the error alone that the caller's thread has pending, whatever memory it goes to."""
import ctypes

import pytest
import torch

from deserve_amd import _lib


@pytest.mark.gpu
@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("pending", [True, False])
def test_a_pending_error_stays_with_the_caller(pinned, pending):
    print("[case] swap and a pending error", pinned, pending, flush=True)
    lib, n = _lib.lib(), 1 << 20
    hip = ctypes.CDLL(lib._name)               # (finds the runtime's functions among the library's own dependencies)
    pages = torch.randint(0, 255, (2, n), dtype=torch.uint8, device="cuda")
    host = torch.zeros((2, n), dtype=torch.uint8, pin_memory=pinned)
    stream = torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()
    hip.hipGetLastError()
    if pending:
        assert hip.hipSetDevice(1 << 20) != 0  # refused by the host
    error = hip.hipPeekAtLastError()
    rc = lib.dskv_swap_slice(pages.data_ptr(), n, n, 2, host.data_ptr(), None, stream, stream)
    after = hip.hipGetLastError()
    assert rc == 0 and after == error and (error != 0) == pending
    torch.cuda.synchronize()
    assert torch.equal(host, pages.cpu())
