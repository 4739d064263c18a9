"""Token splits of the covariance's two passes, read on the host from the
workspace its check entry asks for: per head, in rows of 128 floats, one for
each of the mean's partials, 36 tiles of 256 and a diagonal for each of the
covariance's, and the query norms.
"""
import ctypes

import pytest

from rotatek_amd import _lib

CUS = 256


def _desc(shape, dtype):
    t = _lib.RkTensor()
    t.dtype, t.ndim = dtype, len(shape)
    st = 1
    for i in reversed(range(len(shape))):
        t.shape[i], t.stride[i] = shape[i], st
        st *= shape[i]
    return t


def _rows(B, H, S, dtype):
    need = ctypes.c_size_t(0)
    k, cov = _desc((B, H, S, 128), dtype), _desc((B, H, 128, 128), _lib.RK_F32)
    assert _lib.load().rk_key_covariance_check(ctypes.byref(k), None, ctypes.byref(cov), CUS, ctypes.byref(need)) == 0
    assert need.value % (B * H * 512) == 0
    return need.value // (B * H * 512)


@pytest.mark.parametrize("B,H,S,mean", [(1, 8, 65536, 64), (1, 8, 131072, 64), (4, 4, 65536, 32), (1, 32, 30720, 32),
                                        (16, 4, 30720, 60), (32, 32, 30720, 60), (32, 32, 14000, 28),
                                        (8, 4, 12001, 24), (1, 32, 2304, 9),
                                        (1, 8, 500, 2), (1, 1, 1, 1)])
def test_mean_splits(B, H, S, mean):
    """Two workgroups per CU, or 512 tokens each while that is at most 32 (with few heads) per head."""
    assert (_rows(B, H, S, _lib.RK_BF16) - 1) % 73 == mean


@pytest.mark.parametrize("B,H,S,dtype,splits", [
    (1, 1, 131072, _lib.RK_BF16, 90), (1, 1, 1000000, _lib.RK_F16, 250), (1, 2, 1000000, _lib.RK_BF16, 128),
    (1, 4, 131072, _lib.RK_BF16, 64), (1, 1, 65536, _lib.RK_F32, 256), (1, 2, 65536, _lib.RK_F32, 128),
    (1, 4, 65536, _lib.RK_F32, 128), (1, 4, 32768, _lib.RK_F32, 64), (1, 3, 32768, _lib.RK_F32, 128),
    (1, 4, 20000, _lib.RK_F32, 64), (1, 8, 65536, _lib.RK_F32, 64), (8, 4, 12001, _lib.RK_BF16, 16),
    (10, 32, 4000, _lib.RK_F16, 3), (32, 32, 14000, _lib.RK_F16, 1), (1, 8, 500, _lib.RK_BF16, 1)])
def test_covariance_splits(B, H, S, dtype, splits):
    """Few heads with long spans fill the CUs; the others keep the split of least estimated cost."""
    bh = B * H
    two_per_cu = min(-(-2 * CUS // bh), -(-S // 256))
    mean = max(two_per_cu, min(-(-S // 512), max(32, bh), 4096))
    assert _rows(B, H, S, dtype) == mean + 73 * splits + 1
