"""Launch forms of the covariance and the truncated Key write that the sizes
choose: one workgroup per head finishing its covariance itself, Keys larger
than the memory-side cache (streamed loads and stores), and the 16-byte
output path of the rotation.  Inputs are small integers with a mean of zero,
so every sum is exact and the results are compared bit for bit.
"""
import ctypes

import pytest
import torch

from rotatek_amd import _lib, prefill

pytestmark = pytest.mark.gpu


def _int_keys(B, H, S, D, dtype, seed):
    """[B, H, S, D] integers in [-2, 2], each row followed by its negative (an odd last row is zero)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    half = torch.randint(-2, 3, (B, H, S // 2, D), generator=g, device="cuda")
    K = torch.zeros(B, H, S, D, device="cuda")
    K[:, :, 0:2 * (S // 2):2], K[:, :, 1:2 * (S // 2):2] = half, -half
    return K.to(dtype)


def _cov_ref(K):
    """Kc^T Kc rounded to the key dtype; exact below 2^24."""
    k = K.float()
    return torch.matmul(k.transpose(-1, -2).contiguous(), k).to(K.dtype).float()


def _cov_splits(K):
    """Workgroups per head of the covariance pass, from the workspace it asks for
    (per head, in rows of 128 floats: the mean's partials, at most 72 of them
    here, 73 for each split, one)."""
    need = ctypes.c_size_t(0)
    d = [_lib.desc(t) for t in (K, torch.empty(*K.shape[:2], K.shape[3], K.shape[3], device="cuda"))]
    assert _lib.load().rk_key_covariance_check(ctypes.byref(d[0]), None, ctypes.byref(d[1]), 0, ctypes.byref(need)) == 0
    return (need.value // (K.shape[0] * K.shape[1] * 512) - 1) // 73


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,S,D", [(1, 1, 1, 128), (1, 2, 31, 128), (2, 3, 33, 128), (1, 4, 256, 64), (1, 4, 257, 128),
                                     (2, 300, 130, 128), (3, 256, 514, 128), (40, 8, 300, 96)])
def test_covariance_one_workgroup_per_head(B, H, S, D, dtype):
    print(f"[case] covariance B={B} H={H} S={S} D={D} {dtype}", flush=True)
    K = _int_keys(B, H, S, D, dtype, 11 * S + D)
    mean, cov = prefill.key_covariance(K)
    assert torch.equal(mean, torch.zeros_like(mean))
    assert torch.equal(cov, _cov_ref(K))
    Q = torch.randn(B, 2 * H, 40, D, generator=torch.Generator(device="cuda").manual_seed(S), device="cuda").to(dtype)
    mean_w, cov_w = prefill.key_covariance(K, Q, 2)
    assert torch.equal(mean_w, mean)
    assert torch.equal(cov_w, prefill.query_weight(cov, Q, 2))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [1, 33, 500])
@pytest.mark.parametrize("H", [39, 40, 63, 64, 65])
def test_finished_heads_equal_separate_ones(H, S, dtype):
    """Heads finished by their covariance workgroup (many heads) hold the bits
    of the separate finalisation (eight at a time), at a non-zero mean."""
    print(f"[case] finished heads H={H} S={S} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(H + S)
    K = (torch.randn(1, H, S, 128, generator=g, device="cuda") + 0.7).to(dtype)
    Q = torch.randn(1, 2 * H, 40, 128, generator=g, device="cuda").to(dtype)
    for q in (None, Q):
        mean, cov = prefill.key_covariance(K, q, 2)
        for h in range(0, H, 8):
            few = prefill.key_covariance(K[:, h:h + 8], None if q is None else q[:, 2 * h:2 * h + 16], 2)
            assert torch.equal(mean[:, h:h + 8], few[0]) and torch.equal(cov[:, h:h + 8], few[1])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [1030, 1031])
def test_streamed_keys(S, dtype):
    """Keys past the memory-side cache (32 batch rows that share one row's
    memory) give every row the same result as that row alone."""
    B, H, k = 40, 32, 128
    print(f"[case] streamed Keys S={S} {dtype}", flush=True)
    one = _int_keys(1, H, S, 128, dtype, S)
    K = one.expand(B, H, S, 128)
    assert K.numel() * 2 > 256 << 20
    mean, cov = prefill.key_covariance(K)
    assert torch.equal(mean, torch.zeros_like(mean))
    assert torch.equal(cov, _cov_ref(one).expand(B, -1, -1, -1))
    R = torch.randint(-2, 3, (1, H, 128, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    R = R.to(dtype)
    out = prefill.rotate_keys(K, R.expand(B, -1, -1, -1))
    assert out.numel() * 2 > 256 << 20
    want = torch.matmul(one.float(), R.float()).to(dtype)
    assert torch.equal(out, want.expand(B, -1, -1, -1))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,S,splits", [(16, 4, 30722, 8), (9, 32, 4098, 3), (40, 32, 1030, 1)])
def test_streamed_keys_weighted_and_split(B, H, S, splits, dtype):
    """Streamed Keys of mean one, in one and in several workgroups per head,
    plain and query-weighted (batch rows share one row's memory)."""
    print(f"[case] streamed and split B={B} H={H} S={S} {dtype}", flush=True)
    one = _int_keys(1, H, S, 128, dtype, S)
    cov_one = _cov_ref(one)
    K = (one + 1).expand(B, H, S, 128)
    assert K.numel() * 2 > 256 << 20
    Q = torch.randn(1, 2 * H, 40, 128, generator=torch.Generator(device="cuda").manual_seed(S), device="cuda").to(dtype)
    Q = Q.expand(B, 2 * H, 40, 128)
    mean, cov = prefill.key_covariance(K)
    assert _cov_splits(K) == splits
    # the centre is the mean in the key dtype, exactly one
    assert float((mean - 1).abs().max()) < 1e-6
    assert torch.equal(cov, cov_one.expand(B, -1, -1, -1))
    mean_w, cov_w = prefill.key_covariance(K, Q, 2)
    assert torch.equal(mean_w, mean) and torch.equal(cov_w, prefill.query_weight(cov, Q, 2))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [8, 16, 24, 32, 40, 64, 72, 96, 128])
@pytest.mark.parametrize("S", [1, 15, 33, 127, 129, 1500])
def test_rotation_output_paths(S, k, dtype):
    """Aligned rows (16-byte stores), rows at an odd offset and a strided R
    (element paths) hold the same values."""
    B, H = 2, 3
    print(f"[case] rotate S={S} k={k} {dtype}", flush=True)
    K = _int_keys(B, H, S, 128, dtype, S + k)
    g = torch.Generator(device="cuda").manual_seed(k)
    R = torch.randint(-2, 3, (B, H, 128, k), generator=g, device="cuda").to(dtype)
    want = torch.matmul(K.float(), R.float()).to(dtype)
    wide = torch.full((B, H, S, k + 8), 9.0, dtype=dtype, device="cuda")
    odd = torch.full((B, H, S, k + 3), 9.0, dtype=dtype, device="cuda")
    strided = torch.zeros(B, H, 128, 2 * k, dtype=dtype, device="cuda")
    strided[..., ::2] = R
    prefill.rotate_keys(K, R, out=wide[..., :k])
    prefill.rotate_keys(K, R, out=odd[..., 1:k + 1])
    assert torch.equal(prefill.rotate_keys(K, R), want)
    assert torch.equal(prefill.rotate_keys(K, strided[..., ::2]), want)
    assert torch.equal(prefill.rotate_keys(K, R.float()), want)
    assert torch.equal(wide[..., :k], want) and bool((wide[..., k:] == 9).all())
    assert torch.equal(odd[..., 1:k + 1], want) and bool((odd[..., k + 1:] == 9).all()) and bool((odd[..., 0] == 9).all())


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,k", [(128, 1), (128, 31), (128, 32), (128, 96), (128, 128), (64, 17), (33, 33), (1, 1)])
def test_leading_rotation_is_gather_of_the_first_columns(D, k, out_dtype):
    """The first k columns and their mask in one launch: what the gather with
    idx = 0..k-1 gives, from a basis with more columns and from a strided one."""
    print(f"[case] leading rotation D={D} k={k} {out_dtype}", flush=True)
    B, H = 2, 3
    g = torch.Generator(device="cuda").manual_seed(D * k)
    full = torch.randn(B, H, D, D, generator=g, device="cuda")
    mean = torch.randn(B, H, D, generator=g, device="cuda")
    idx = torch.arange(k, device="cuda").expand(B, H, k)
    for basis in (full, full[..., :k].contiguous(), full.transpose(-1, -2)):
        Rp, dmu, mask = prefill.leading_rotation(basis, k, mean, out_dtype)
        want_R, want_dmu = prefill.gather_rotation(basis, idx, mean, out_dtype)
        assert torch.equal(Rp, want_R) and torch.equal(Rp, basis[..., :k].to(out_dtype))
        assert torch.equal(dmu, want_dmu)
        m = mean.double().unsqueeze(-1)
        r = Rp.double()
        exact = (m - r @ (r.transpose(-1, -2).contiguous() @ m)).squeeze(-1)
        # fp32 sums of D and k products, then the output's rounding
        scale = float(exact.abs().max()) + float((r.abs() @ (r.abs().transpose(-1, -2).contiguous() @ m.abs())).max())
        ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 0.0}[out_dtype]
        assert float((dmu.double() - exact).abs().max()) <= scale * 1e-5 + ulp * float(exact.abs().max())
        assert mask.dtype == torch.bool and torch.equal(mask, (torch.arange(D, device="cuda") < k).expand(B, H, D))


def test_failed_factorisation_raises_from_update_rotatek():
    """Keys whose fp16 covariance overflows fail the first pivot: the call
    raises and leaves the pruner's state as it was."""
    from rotatek_amd.pruning import ChannelPruner
    print("[case] update_rotatek with a failed pivot", flush=True)
    g = torch.Generator(device="cuda").manual_seed(0)
    K = (torch.randn(1, 2, 3000, 128, generator=g, device="cuda") * 40).half()
    p = ChannelPruner(0.75, 10, 10, solver="power_iter")
    for _ in range(3):
        with pytest.raises(torch.linalg.LinAlgError):
            p.update_rotatek(K, K, K, None, 1)
        assert not hasattr(p, "current_rotatek_R_partial")
    out = p.update_rotatek(K / 40, K / 40, K, None, 1)
    assert bool(torch.isfinite(out[0]).all())
