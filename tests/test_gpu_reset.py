"""The launch that puts a stream's device state back: exactly the buffers it names, whole, and nothing
beside them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WORDS = 32


class ResetArgs(C.Structure):
    """NkResetArgs of csrc/kernel_params.h."""
    _fields_ = [("base", C.c_void_p), ("stride", C.c_ulonglong), ("z0", C.c_void_p), ("z1", C.c_void_p),
                ("st", C.c_void_p), ("nbuf", C.c_uint32), ("n", C.c_uint32), ("zn", C.c_uint32), ("words", C.c_uint32),
                ("val", C.c_int * WORDS)]


@pytest.mark.parametrize("nbuf,n,zn,words", [(24, 8 * 1024, 8 * 640, 12), (3, 257, 1, 32), (1, 1, 1000, 1), (2, 300, 0, 0),
                                             (0, 0, 5120, 24), (5, 256, 256, 0), (0, 0, 0, 32)])
def test_stream_reset_touches_its_buffers_only(gpu, nbuf, n, zn, words):
    import nemoasr

    L = nemoasr.lib()
    stride, lead = 2 * n + 40, 24  # the stream's rows lie inside larger buffers
    rng = np.random.default_rng([nbuf, n, zn, words])
    din = rng.standard_normal(lead + max(nbuf, 1) * stride).astype(np.float32)
    z0, z1 = (rng.standard_normal(zn + 2 * lead).astype(np.float32) for _ in range(2))
    st = rng.integers(-2**31, 2**31, words + 2 * lead, dtype=np.int64).astype(np.int32)
    val = rng.integers(-2**31, 2**31, WORDS, dtype=np.int64).astype(np.int32)
    d, d0, d1, ds = (gpu.put(x) for x in (din, z0, z1, st))
    a = ResetArgs(base=d.at(4 * lead), stride=stride, z0=d0.at(4 * lead) if zn else None, z1=d1.at(4 * lead) if zn else None,
                  st=ds.at(4 * lead), nbuf=nbuf, n=n, zn=zn, words=words, val=(C.c_int * WORDS)(*val.tolist()))
    f = L.nk_stream_reset
    f.restype, f.argtypes = C.c_int, [C.c_void_p, C.c_void_p]
    gpu.check(f(gpu.h, C.byref(a)))
    for l in range(nbuf):
        din[lead + l * stride:][:n] = 0
    z0[lead:lead + zn] = z1[lead:lead + zn] = 0
    st[lead:lead + words] = val[:words]
    for buf, want in ((d, din), (d0, z0), (d1, z1), (ds, st)):
        assert np.array_equal(buf.read(want.shape, want.dtype), want)
