"""The paper family's decomposition where query heads share a KV head: one
unit per query head while that grid is one round of one workgroup per CU
(dense, and RotateK in fp32), else the grouped units of the gqa family.  The
line is checked on the CPU from the workspace each call asks for; on the
device both sides of it run against the float64 oracle.
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import decode as od
from rotatek_amd import _lib

CUS = 256
DTYPES = {torch.float16: _lib.RK_F16, torch.bfloat16: _lib.RK_BF16, torch.float32: _lib.RK_F32}


def _d(shape, dtype):
    t = _lib.RkTensor()
    t.dtype, t.ndim = dtype, len(shape)
    st = 1
    for i in reversed(range(len(shape))):
        t.shape[i], t.stride[i] = shape[i], st
        st *= shape[i]
    return t


def _ws(policy, B, H, G, S, dtype, vis=None):
    """Workspace bytes the dense (or, with ``vis`` = (S_v, Dk), RotateK) check asks for."""
    need = ctypes.c_size_t(0)
    q, kv = _d((B, H * G, 128), dtype), _d((B, H, S, 128), dtype)
    if vis is None:
        st = _lib.load().rk_full_channel_decode_check(ctypes.byref(q), ctypes.byref(kv), ctypes.byref(kv), G, None,
                                                      policy, CUS, ctypes.byref(need))
    else:
        S_v, Dk = vis
        R, ks, vs = _d((B, H, 128, Dk), dtype), _d((B, H, S_v, Dk), dtype), _d((B, H, S_v, 128), dtype)
        st = _lib.load().rk_rotatek_decode_check(
            ctypes.byref(q), ctypes.byref(R), None, ctypes.byref(kv), ctypes.byref(kv), None, ctypes.byref(ks),
            ctypes.byref(vs), G, None, policy, CUS, ctypes.byref(need))
    assert st == 0
    return need.value


# B, KV heads, G, full tokens, (visual tokens, kept), dtype code, one unit per query head?
LINE = [
    (1, 8, 4, 70, None, _lib.RK_BF16, True), (1, 8, 4, 2000, None, _lib.RK_BF16, True),
    (4, 8, 4, 300, None, _lib.RK_F16, True),
    (1, 8, 4, 8000, None, _lib.RK_F16, False), (4, 1, 40, 300, None, _lib.RK_F16, False),
    (32, 8, 4, 70, None, _lib.RK_F16, False),
    (1, 4, 7, 2000, None, _lib.RK_F32, True), (1, 4, 7, 8000, None, _lib.RK_F32, False),
    (1, 4, 7, 100, (1000, 32), _lib.RK_F32, True), (4, 4, 7, 100, (8000, 32), _lib.RK_F32, False),
    (1, 4, 7, 100, (1000, 32), _lib.RK_F16, False),
]


# the same past one round of one workgroup per CU, and within it
LINE += [
    (16, 16, 2, 300, None, _lib.RK_BF16, True), (4, 8, 2, 2400, None, _lib.RK_F16, True),
    (1, 16, 2, 4800, None, _lib.RK_BF16, True), (4, 8, 2, 4800, None, _lib.RK_BF16, False),
    (1, 8, 2, 9600, None, _lib.RK_BF16, False), (1, 8, 2, 4800, None, _lib.RK_BF16, False),
    (16, 4, 3, 600, None, _lib.RK_BF16, False),
    (1, 8, 7, 1200, None, _lib.RK_F32, True), (1, 8, 7, 2400, None, _lib.RK_F32, False),
    (1, 16, 4, 600, None, _lib.RK_F32, True), (1, 16, 4, 1200, None, _lib.RK_F32, False),
    (1, 1, 64, 1200, None, _lib.RK_F32, True), (1, 1, 64, 2400, None, _lib.RK_F32, False),
    (16, 1, 20, 64, None, _lib.RK_F32, True), (32, 4, 7, 64, None, _lib.RK_F32, False),
    (16, 2, 2, 600, None, _lib.RK_F32, False),
    (1, 4, 2, 100, (9600, 32), _lib.RK_F32, True), (4, 4, 2, 100, (2400, 32), _lib.RK_F32, True),
    (1, 2, 2, 100, (4800, 32), _lib.RK_F32, True), (1, 8, 2, 100, (8061, 32), _lib.RK_F32, True),
]


@pytest.mark.parametrize("case", LINE, ids=lambda c: "-".join(str(v) for v in c))
def test_paper_family_decomposition(case):
    B, H, G, S, vis, dtype, per_head = case
    esz = 4 if dtype == _lib.RK_F32 else 2
    S_v, Dk = vis or (0, 0)
    plan = _lib.plan_decode(B, H * G, H, Dk, S_v, S, esz, _lib.RK_POLICY_PAPER if per_head else _lib.RK_POLICY_GQA, CUS)
    per_block = 8 if esz == 4 else 16
    assert plan["units"] == B * H * (G if per_head else -(-G // per_block))
    assert _ws(_lib.RK_POLICY_PAPER, B, H, G, S, dtype, vis) == plan["workspace_bytes"]


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("B,H,G,S,S_v", [(1, 8, 4, 1, 0), (1, 8, 4, 2047, 0), (1, 8, 4, 2049, 0), (2, 4, 7, 257, 0),
                                         (1, 2, 20, 300, 0), (1, 4, 7, 61, 1001), (1, 8, 4, 61, 4097),
                                         (3, 4, 7, 61, 4097)])
def test_paper_family_matches_oracle(B, H, G, S, S_v, dtype):
    from rotatek_amd.kernels.fused_decode import rotatek_decode_fused
    from rotatek_amd.kernels.full_channel_flash_decoding import full_channel_decode
    print(f"[case] paper family B={B} H={H} G={G} S={S} S_v={S_v} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(17 * S + S_v)

    def rn(*s):
        return torch.randn(*s, generator=g, device="cuda").to(dtype)

    q, k, v = rn(B, H * G, 128), rn(B, H, S, 128), rn(B, H, S, 128)
    # the decode bars of test_gpu_decode.py
    tol = {torch.float16: 2e-3, torch.bfloat16: 1e-2, torch.float32: 1e-4}[dtype]
    if S_v == 0:
        got, want = full_channel_decode(q, k, v, G), od.full_channel_decode(_np(q), _np(k), _np(v), G)
    else:
        R = torch.linalg.qr(torch.randn(B, H, 128, 32, generator=torch.Generator().manual_seed(3)))[0]
        R = R.contiguous().cuda().to(dtype)
        a = dict(q_full=q, R_partial=R, delta_mu=rn(B, H, 128), k_full=k, v_full=v,
                 mask_full=torch.ones(B, S, dtype=torch.uint8, device="cuda"), k_sparse=rn(B, H, S_v, 32),
                 v_sparse=rn(B, H, S_v, 128), num_kv_groups=G)
        got = rotatek_decode_fused(**a)[0]
        want = od.rotatek_decode(**{n: (t if n == "num_kv_groups" else t.cpu().numpy() if n == "mask_full" else _np(t))
                                    for n, t in a.items()})
    # a bf16 output is held to the bar or to its own rounding (one token: |out| up to 4)
    err = np.abs(_np(got) - want)
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}[dtype]
    assert got.shape == want.shape and (err <= np.maximum(tol, np.abs(want) * ulp)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 128), (torch.float16, 96)])
@pytest.mark.parametrize("B,H,S,per_head", [(7, 11, 900, True), (3, 7, 3999, True), (32, 8, 300, True),
                                            (1, 16, 4800, True), (3, 1, 1, True),
                                            (1, 16, 1199, True), (4, 8, 4800, False)])
def test_two_heads_per_kv_head_match_oracle(B, H, S, per_head, dtype, D):
    """Dense units that share K/V rows, in the launch order and in XCD order
    (a number of workgroups that 8 does and does not divide)."""
    from rotatek_amd.kernels.full_channel_flash_decoding import full_channel_decode
    print(f"[case] two heads per KV head B={B} H={H} S={S} D={D} {dtype}", flush=True)
    plan = _lib.plan_decode(B, 2 * H, H, 0, 0, S, 2, _lib.RK_POLICY_PAPER if per_head else _lib.RK_POLICY_GQA, CUS)
    assert _ws(_lib.RK_POLICY_PAPER, B, H, 2, S, DTYPES[dtype]) == plan["workspace_bytes"]
    g = torch.Generator(device="cuda").manual_seed(S)
    shapes = ((B, 2 * H, D), (B, H, S, D), (B, H, S, D))
    q, k, v = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in shapes)
    got, want = full_channel_decode(q, k, v, 2), od.full_channel_decode(_np(q), _np(k), _np(v), 2)
    # the decode bars of test_gpu_decode.py, or the output's own rounding
    tol, ulp = {torch.float16: (2e-3, 2.0 ** -10), torch.bfloat16: (1e-2, 2.0 ** -8)}[dtype]
    assert (np.abs(_np(got) - want) <= np.maximum(tol, np.abs(want) * ulp)).all()
