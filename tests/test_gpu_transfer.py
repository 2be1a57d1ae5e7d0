"""Downloads that several host threads share wait for the stream they are
given, whichever kind of stream it is."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deconwolf_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PER_THREAD = 2  # hipStreamPerThread: a handle that names another stream in each thread


@pytest.mark.parametrize("stream", [None, PER_THREAD])
def test_download_waits_for_the_callers_stream(stream):
    print("download on stream", stream, flush=True)
    L = _lib.lib()
    n = 48 << 20
    v = torch.ones(n, device=DEV)
    out = torch.zeros(n, dtype=torch.int16, device=DEV)
    torch.cuda.synchronize()
    a = np.empty(n, np.uint16)
    for k in range(1, 81):  # a few ms of queued work, the last of it what is read
        _lib.check(L.dwhip_to_u16_device(v.data_ptr(), n, float(k), _lib.U16_ROUND, out.data_ptr(), stream), "convert")
    _lib.check(L.dwhip_download(a.ctypes.data, out.data_ptr(), a.nbytes, stream), "download")
    assert a.min() == a.max() == 80
