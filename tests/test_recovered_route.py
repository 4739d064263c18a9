"""Which ThinK / SparK layers the decode takes without recovered Keys, read on
the host from the entry's check."""
import ctypes

import pytest

from rotatek_amd import _lib

CUS = 256


def _desc(shape, dtype, stride=None, data=4096):
    t = _lib.RkTensor()
    t.data, t.dtype, t.ndim = data, dtype, len(shape)
    st = 1
    for i in reversed(range(len(shape))):
        t.shape[i], t.stride[i] = shape[i], st if stride is None else stride[i]
        st *= shape[i]
    return t


def _check(method, D, Dk, dtype=_lib.RK_F16, B=2, H=3, G=2, S_v=70, S_f=9, k_pruned=None, mask=None):
    q, kf = _desc((B, H * G, D), dtype), _desc((B, H, S_f, D), dtype)
    v = _desc((B, H, S_f + S_v, D), dtype)
    kp = k_pruned or _desc((B, H, S_v, Dk), dtype)
    vs = _desc((B, H, S_v, D), dtype, (H * (S_f + S_v) * D, (S_f + S_v) * D, D, 1))
    out, need = _desc((B, H * G, D), dtype), ctypes.c_size_t(0)
    tm = sm = pm = None
    if method == "think":
        tm = mask or _desc((B, H, D), _lib.RK_U8)
    else:
        sm, pm = mask or _desc((B, H, S_v, D), _lib.RK_U8), _desc((B, H, S_v, 1), dtype)
    return _lib.load().rk_recovered_decode_check(
        _lib.ref(q), _lib.ref(tm), _lib.ref(kf), _lib.ref(v), 4, S_v, _lib.ref(sm), _lib.ref(pm), _lib.ref(kp),
        _lib.ref(vs), G, _lib.ref(out), _lib.RK_POLICY_PAPER, CUS, ctypes.byref(need))


@pytest.mark.parametrize("D,Dk,taken", [(128, 32, True), (128, 8, True), (128, 128, True), (128, 13, False),
                                        (128, 90, False), (96, 24, True), (96, 13, False), (64, 32, True),
                                        (100, 40, True), (50, 13, True), (33, 33, True), (1, 1, True)])
def test_think_compact_rows(D, Dk, taken):
    """Compact Keys that alone keep the decode from 16-byte loads are recovered first."""
    assert (_check("think", D, Dk) == 0) == taken
    wide = _desc((2, 3, 70, Dk), _lib.RK_F16, (3 * 70 * (Dk + 3), 70 * (Dk + 3), Dk + 3, 1))
    if D % 8 == 0:
        assert _check("think", D, Dk, k_pruned=wide) != 0
