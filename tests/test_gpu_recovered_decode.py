"""Decode over ThinK / SparK pruned Keys without recovering them: against the
recovery followed by the dense decode (the same products in another fp32
order) and the float64 oracle, over span edges, kept counts, groups, ragged
masks and the layouts that are recovered first.
"""
import numpy as np
import pytest
import torch

from oracle import decode as od
from rotatek_amd.cache import DynamicCache
from rotatek_amd.kernels.full_channel_flash_decoding import full_channel_decode

pytestmark = pytest.mark.gpu

TOL = {torch.float16: 2e-3, torch.bfloat16: 1e-2}


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


def _cache(method, B, H, S_v, n_p, n_t, keep, dtype, g, D=128, kept=None):
    """A cache of one layer; ``kept``: channels the mask keeps (default ``keep``)."""
    def rn(*s):
        return torch.randn(*s, generator=g, device="cuda").to(dtype)
    kept = keep if kept is None else kept
    rows = S_v if method == "spark" else 1
    r = torch.rand(B, H, rows, D, generator=g, device="cuda")
    mask = torch.zeros_like(r, dtype=torch.bool).scatter_(-1, r.topk(kept, dim=-1).indices, True)
    c = DynamicCache(reserve_tokens=5)
    c.store_pruned(rn(B, H, S_v, keep), rn(B, H, n_p, D), rn(B, H, n_t, D), None, rn(B, H, S_v + n_p + n_t, D), 0)
    c.think_mask.append(mask[:, :, 0].contiguous() if method == "think" else None)
    c.spark_mask.append(mask if method == "spark" else None)
    c.spark_pruned_mean.append(rn(B, H, S_v, 1) if method == "spark" else None)
    return c


def _staged(c, q, G):
    k = c.recovered_keys(0)
    return full_channel_decode(q, k, c._spans[0].v[:, :, :k.shape[2]], G)


def _check(c, q, G, dtype):
    want = _staged(c, q, G)
    k, v = c.recovered_keys(0).clone(), c._spans[0].v[:, :, :c.recovered_keys(0).shape[2]]
    oracle = od.full_channel_decode(_np(q), _np(k), _np(v), G)
    got = c.decode_recovered(q, 0, G)
    assert got.shape == want.shape and got.dtype == want.dtype
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -10
    for ref in (oracle, _np(want)):
        assert (np.abs(_np(got) - ref) <= np.maximum(TOL[dtype], np.abs(ref) * ulp)).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("method", ["think", "spark"])
@pytest.mark.parametrize("B,H,G,S_v,n_p,n_t,keep", [
    (1, 2, 1, 1, 1, 0, 8), (1, 4, 1, 31, 0, 1, 32), (2, 3, 1, 33, 5, 7, 16), (1, 2, 7, 257, 30, 33, 32),
    (2, 2, 4, 1000, 30, 30, 64), (1, 2, 20, 129, 3, 4, 40), (1, 32, 1, 2304, 64, 64, 32), (3, 8, 2, 4097, 30, 31, 24),
    (1, 2, 1, 300, 9, 9, 72), (1, 2, 2, 300, 9, 9, 128), (1, 2, 2, 70, 3, 3, 13)])
def test_matches_recovery_and_oracle(method, B, H, G, S_v, n_p, n_t, keep, dtype):
    print(f"[case] recovered {method} B={B} H={H} G={G} S_v={S_v} {n_p}+{n_t} keep={keep} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S_v * keep)
    c = _cache(method, B, H, S_v, n_p, n_t, keep, dtype, g)
    q = torch.randn(B, H * G, 128, generator=g, device="cuda").to(dtype)
    _check(c, q, G, dtype)
    # an appended token, then a device-only append that the host has not seen
    kn, vn = (torch.randn(B, H, 1, 128, generator=g, device="cuda").to(dtype) for _ in range(2))
    c.update(kn, vn, 0)
    _check(c, q, G, dtype)
    c.append_(0, kn, vn)
    _check(c, q, G, dtype)


@pytest.mark.parametrize("kept", [0, 3, 31, 33, 90, 128])
@pytest.mark.parametrize("method", ["think", "spark"])
def test_masks_that_keep_another_count(method, kept):
    """Rows that keep fewer channels than K_compact has columns leave the rest
    unused; past the last column, kept channels take the fill."""
    print(f"[case] recovered {method} kept={kept} of 32 columns", flush=True)
    g = torch.Generator(device="cuda").manual_seed(kept)
    c = _cache(method, 2, 3, 200, 4, 4, 32, torch.float16, g, kept=kept)
    _check(c, torch.randn(2, 6, 128, generator=g, device="cuda").half(), 2, torch.float16)


@pytest.mark.parametrize("how", ["mask255", "mask_offset", "mask_strided", "mean_strided", "heads_first", "D64"])
def test_spark_layouts(how):
    print(f"[case] recovered spark layout {how}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    D = 64 if how == "D64" else 128
    B, H, S_v = 2, 3, 150
    c = _cache("spark", B, H, S_v, 4, 4, 32, torch.float16, g, D=D)
    m, pm, kc = c.spark_mask[0], c.spark_pruned_mean[0], c.key_cache_pruned[0]
    if how == "mask255":
        c.spark_mask[0] = m.to(torch.uint8) * 255
    elif how in ("mask_offset", "mask_strided"):
        wide = torch.zeros(B, H, S_v, D + (8 if how == "mask_offset" else 16), dtype=torch.bool, device="cuda")
        o = 8 if how == "mask_offset" else 16
        wide[..., o:] = m
        c.spark_mask[0] = wide[..., o:]
    elif how == "mean_strided":
        wide = torch.zeros(B, H, S_v, 3, dtype=pm.dtype, device="cuda")
        wide[..., 1:2] = pm
        c.spark_pruned_mean[0] = wide[..., 1:2]
    elif how == "heads_first":
        c.key_cache_pruned[0] = kc.transpose(1, 2).contiguous().transpose(1, 2)
        c.spark_mask[0] = m.transpose(1, 2).contiguous().transpose(1, 2)
    _check(c, torch.randn(B, H, D, generator=g, device="cuda").half(), 1, torch.float16)


@pytest.mark.parametrize("method", ["think", "spark"])
def test_captured_in_a_graph(method):
    print(f"[case] recovered {method} graph", flush=True)
    g = torch.Generator(device="cuda").manual_seed(9)
    c = _cache(method, 2, 4, 500, 8, 8, 32, torch.bfloat16, g)
    q = torch.randn(2, 8, 128, generator=g, device="cuda").bfloat16()
    eager = c.decode_recovered(q, 0, 2)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            out = c.decode_recovered(q, 0, 2)
    for i in range(4):
        q.copy_(torch.randn(q.shape, generator=g, device="cuda").bfloat16())
        eager = c.decode_recovered(q, 0, 2)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_non_finite_queries():
    """A non-finite query entry makes its head's output NaN, as recovered Keys do, in a pruned channel too."""
    for method in ("think", "spark"):
        print(f"[case] recovered {method} non-finite", flush=True)
        g = torch.Generator(device="cuda").manual_seed(2)
        c = _cache(method, 1, 2, 100, 4, 4, 32, torch.float16, g)
        q = torch.randn(1, 2, 128, generator=g, device="cuda").half()
        m = c.think_mask[0][0, 0] if method == "think" else c.spark_mask[0][0, 0, 0]
        q[0, 0, int((~m).nonzero()[0])] = float("inf")
        got, want = c.decode_recovered(q, 0, 1), _staged(c, q, 1)
        assert torch.equal(got.isnan(), want.isnan())


def test_refused_calls_stay_refused():
    """Pruned Keys off the device and unified layers raise before any launch, as with recovered Keys."""
    print("[case] recovered refusals", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(1, 2, 128, generator=g, device="cuda").half()
    for method in ("think", "spark"):
        c = _cache(method, 1, 2, 60, 4, 4, 32, torch.float16, g)
        c.key_cache_pruned[0] = c.key_cache_pruned[0].cpu()
        with pytest.raises(RuntimeError, match="GPU tensor"):
            c.decode_recovered(q, 0, 1)
    c._spans[0].unified = True
    with pytest.raises(ValueError, match="unified"):
        c.decode_recovered(q, 0, 1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("method,keep,D", [("think", 8, 128), ("think", 32, 128), ("think", 64, 128), ("think", 96, 128),
                                           ("think", 32, 96), ("think", 20, 50), ("spark", 32, 128)])
def test_infinite_keys(method, keep, D, dtype):
    """A Key that is infinite against the query's sign drops its token, one with it makes the head NaN, as recovered."""
    print(f"[case] recovered {method} infinite Keys keep={keep} D={D} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(keep)
    c = _cache(method, 1, 3, 100, 4, 4, keep, dtype, g, D=D)
    q = torch.randn(1, 6, D, generator=g, device="cuda").to(dtype)
    row = c.think_mask[0][0] if method == "think" else c.spark_mask[0][0, :, 7]
    for h in range(3):
        q[0, 2 * h:2 * h + 2, int(row[h].nonzero()[0])] = 1.5
    c.key_cache_pruned[0][0, :2, 7, 0] = -float("inf")
    c.key_cache_pruned[0][0, 2, 7, 0] = float("inf")
    got, want = c.decode_recovered(q, 0, 2), _staged(c, q, 2)
    assert bool(torch.isfinite(want[:, :, :4]).all()) and bool(want[:, :, 4:].isnan().all())
    assert torch.equal(got.isnan(), want.isnan())
    err, ref = (_np(got) - _np(want))[:, :, :4], np.abs(_np(want))[:, :, :4]
    assert (np.abs(err) <= np.maximum(TOL[dtype], ref * 2.0 ** -8)).all()
