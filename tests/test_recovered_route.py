"""Which ThinK / SparK layers the decode takes without recovered Keys, read on
the host from the entry's check."""
import ctypes

import pytest
import torch

from rotatek_amd import _lib
from rotatek_amd.cache import DynamicCache
from rotatek_amd.kernels import _launch

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


def _layout(method, D, Dk, dtype, kind, B=2, H=3, S_v=70):
    q, kp = torch.zeros(B, 2 * H, D, dtype=dtype), torch.zeros(B, H, S_v, Dk, dtype=dtype)
    if method == "think":
        return q, None, kp
    wide = torch.zeros(B, H, S_v, 2 * D + 16, dtype=torch.bool)
    return q, {"rows": torch.zeros(B, H, S_v, D, dtype=torch.bool), "offset": wide[..., 8:8 + D],
               "strided": wide[..., 16:16 + D], "split": wide[..., :2 * D:2]}[kind], kp


@pytest.mark.parametrize("method,kind", [("think", "rows"), ("spark", "rows"), ("spark", "offset"),
                                         ("spark", "strided"), ("spark", "split")])
def test_early_refusal_is_the_entry_refusal(method, kind):
    """What the host rule turns away, the entry refuses too, and these layouts the other way round."""
    codes = {torch.float16: _lib.RK_F16, torch.bfloat16: _lib.RK_BF16, torch.float32: _lib.RK_F32}
    for dtype, code in codes.items():
        for D in (1, 50, 64, 96, 100, 128):
            for Dk in [k for k in (0, 1, 8, 13, 32, 64, 72, 128) if k <= D]:
                q, mask, kp = _layout(method, D, Dk, dtype, kind)
                taken = _check(method, D, Dk, code, mask=_lib.desc(mask)) == 0
                assert _launch.recovered_decode_takes(q, mask, kp) == taken, (dtype, D, Dk)


@pytest.mark.parametrize("method,D,Dk,kind", [("spark", 128, 96, "rows"), ("spark", 128, 13, "rows"),
                                              ("spark", 64, 32, "rows"), ("spark", 128, 32, "offset"), ("think", 128, 13, "rows")])
def test_refused_before_anything_is_packed(monkeypatch, method, D, Dk, kind):
    q, mask, kp = _layout(method, D, Dk, torch.float16, kind)
    B, H, S_v, _ = kp.shape
    c = DynamicCache(reserve_tokens=4)
    c.store_pruned(kp, torch.zeros(B, H, 2, D).half(), torch.zeros(B, H, 3, D).half(), None,
                   torch.zeros(B, H, S_v + 5, D).half(), 0)
    c.think_mask.append(torch.zeros(B, H, D, dtype=torch.bool) if method == "think" else None)
    c.spark_mask.append(mask)
    c.spark_pruned_mean.append(torch.zeros(B, H, S_v, 1).half())

    def never(*a):
        raise AssertionError("reached the launcher")

    monkeypatch.setattr(_launch, "recovered_decode", never)
    assert c._decode_pruned(q, 0, 2) is None
