"""Subspace iteration at the edges of its 16-column panels and tiles, on
covariances that are not symmetric (W = C V reads C's rows), with element-wise
and 16-byte loads of C, against the float64 iteration from the same start.
"""
import pytest
import torch

from rotatek_amd.rotation import power_iteration_hip

pytestmark = pytest.mark.gpu


def _iterate64(C, V, iters, eps):
    C, V = C.double().cpu(), V.double().cpu()
    eye = torch.eye(V.shape[-1], dtype=torch.float64)
    for _ in range(iters):
        V = C @ V
        G = V.transpose(-1, -2) @ V
        L = torch.linalg.cholesky(G + eps * G.diagonal(dim1=-2, dim2=-1).mean(-1)[..., None, None] * eye)
        V = torch.linalg.solve_triangular(L, V.transpose(-1, -2), upper=False).transpose(-1, -2)
    return V


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("D,k", [(128, k) for k in (1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64)]
                         + [(1, 1), (17, 17), (64, 33), (100, 64), (127, 50)])
def test_panel_edges_against_float64(D, k, strided):
    print(f"[case] power iteration D={D} k={k} strided={strided}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(100 * D + k)
    # singular values within a factor of about 3: rounding errors of an
    # iteration (128-term fp32 sums, about 1e-6) are not amplified much, and
    # five of them stay below 1e-4
    C = torch.eye(D, device="cuda") + 0.3 / D ** 0.5 * torch.randn(2, 3, D, D, generator=g, device="cuda")
    V = torch.randn(2, 3, D, k, generator=g, device="cuda")
    want = _iterate64(C, V, 5, 1e-4)
    if strided:
        big = torch.zeros(2, 3, D, 2 * D + 1, device="cuda")
        big[..., 1::2] = C
        C = big[..., 1::2]
        V = V.transpose(-1, -2).contiguous().transpose(-1, -2)
    got = power_iteration_hip(C, V, 5, 1e-4).double().cpu()
    # each column against its own length: k = D leaves columns of every size
    err = (got - want).norm(dim=-2) / want.norm(dim=-2)
    assert float(err.max()) < (1e-4 if k < D else 1e-3)


@pytest.mark.parametrize("col", [0, 15, 16, 31, 40, 63])
def test_failed_pivot_in_every_panel(col):
    """A start block with a zero column and no ridge has a zero pivot there."""
    g = torch.Generator(device="cuda").manual_seed(col)
    C = torch.eye(128, device="cuda").expand(1, 2, 128, 128).contiguous()
    V = torch.randn(1, 2, 128, 64, generator=g, device="cuda")
    V[0, 1, :, col] = 0
    with pytest.raises(torch.linalg.LinAlgError, match=r"\[1\]"):
        power_iteration_hip(C, V, 1, 0.0)
