"""SiLU and the sigmoid (GLU) over the whole range of f32, through each row-count class of the GEMM.

The activations enter as the bias of a product that is zero.  Reference: v / (1 + e^-v) and
1 / (1 + e^-v) in float64, with e^-v infinite where it leaves f32, as in the f32 formula.  Tolerance:
3e-7 relative (expf within 1 ulp, the sum and the quotient within half an ulp each: 2 x 1.2e-7), plus
one subnormal step, for the values down to v = -88.7 where e^-v reaches the end of f32.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

V = np.concatenate([
    np.linspace(-88.72, -87, 1000), np.linspace(-87, 87, 1200), [88.7, 88.8, 100, -88.73, -90, -104, -1e30, 1e30, 3.4e38, -3.4e38],
    [0.0, 1e-45, -1e-45, 1e-39, -1e-39, 2.0**-126, -(2.0**-126), 1e-10, -1e-10, np.inf, -np.inf, np.nan]]).astype(np.float32)
V = np.concatenate([V, np.zeros(2304 - len(V), np.float32)])


@pytest.mark.parametrize("M", [1, 2, 4, 8, 16, 32, 100])
@pytest.mark.parametrize("act", [1, 3])
def test_activation_range(gpu, M, act):
    import nemoasr

    L = nemoasr.lib()
    K, n = 64, len(V)
    bias = V if act == 1 else np.concatenate([np.ones(n, np.float32), V])
    N = len(bias)
    dA, dW, db = gpu.put(np.zeros((M, K), np.float32)), gpu.put(np.zeros((N, K), np.uint16)), gpu.put(bias)
    dC = gpu.alloc(M * n * 4)
    gpu.begin()
    gpu.check(L.nk_gemm(gpu.h, dA.ptr, K, dW.ptr, K, db.ptr, dC.ptr, n, M, N, K, act, 0, 1.0))
    gpu.end()
    got = dC.read((M, n))
    assert np.array_equal(got, np.broadcast_to(got[0], got.shape), equal_nan=True)
    with np.errstate(all="ignore"):
        v = V.astype(np.float64)
        e = np.exp(-v)
        e[e > np.finfo(np.float32).max] = np.inf
        ref = (v if act == 1 else 1.0) / (1.0 + e)
        assert np.array_equal(np.isnan(got[0]), np.isnan(ref))
        ok = np.isfinite(ref)
        assert np.array_equal(got[0][~ok], ref[~ok].astype(np.float32), equal_nan=True)
        err = np.abs(got[0][ok] - ref[ok])
    worst = int(np.argmax(err - 3e-7 * np.abs(ref[ok])))
    assert (err <= 3e-7 * np.abs(ref[ok]) + 1.5e-45).all(), (V[ok][worst], got[0][ok][worst], ref[ok][worst])
