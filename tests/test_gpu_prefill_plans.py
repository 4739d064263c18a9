"""Launch forms of the covariance and the truncated Key write that the sizes
choose: one workgroup per head finishing its covariance itself, Keys larger
than the memory-side cache (streamed loads and stores), and the 16-byte
output path of the rotation.  Inputs are small integers with a mean of zero,
so every sum is exact and the results are compared bit for bit.
"""
import pytest
import torch

from rotatek_amd import prefill

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
