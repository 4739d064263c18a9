"""ThinK / SparK at the edges of their 32-row query windows (shorter, longer,
not a multiple), of the 64-token compaction tiles and of Keys larger than the
memory-side cache, with queries in 16-byte rows and at odd offsets; values
m / 8, whose sums are exact, so the results equal the oracle bit for bit.
"""
import numpy as np
import pytest
import torch

from oracle import baselines as ob
from rotatek_amd.baselines import spark_prune, think_score_and_compact

pytestmark = pytest.mark.gpu

DT = {torch.float16: "float16", torch.bfloat16: "bfloat16"}


def _np(t):
    return t.detach().cpu().to(torch.float64).numpy()


def _grid(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randint(-15, 16, shape, generator=g).to(torch.float32) / 8).to(dtype).cuda()


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("W,G,S,D,prune", [(1, 1, 64, 128, 96), (31, 2, 65, 128, 64), (32, 4, 128, 128, 121),
                                           (33, 4, 63, 128, 0), (64, 8, 191, 128, 127), (70, 2, 300, 96, 40),
                                           (40, 1, 129, 50, 25)])
def test_windows_match_oracle(W, G, S, D, prune, aligned):
    dtype = torch.float16 if W % 2 else torch.bfloat16
    print(f"[case] windows W={W} G={G} S={S} D={D} prune={prune} aligned={aligned} {dtype}", flush=True)
    B, H = 2, 3
    K = _grid((B, H, S, D), dtype, W + S)
    Q = _grid((B, H * G, W, D + 3), dtype, W * G)
    Q = Q[..., :D].contiguous() if aligned else Q[..., 1:D + 1]
    Kc, mask = think_score_and_compact(K, Q, H, prune)
    Kc_o, mask_o, _ = ob.think_score_and_compact(_np(K), _np(Q), H, prune, DT[dtype])
    np.testing.assert_array_equal(_np(mask), mask_o)
    np.testing.assert_array_equal(_np(Kc), Kc_o)
    Kc, mask, pm = spark_prune(K, Q, G, prune)
    qg = ob.group_queries(_np(Q), G, DT[dtype])
    Kc_o, mask_o, pm_o, _ = ob.per_token_channel_prune(qg, _np(K), prune, DT[dtype])
    np.testing.assert_array_equal(_np(mask), mask_o)
    np.testing.assert_array_equal(_np(Kc), Kc_o)
    np.testing.assert_array_equal(_np(pm), pm_o)


@pytest.mark.parametrize("keep", [1, 7, 8, 32, 40, 128])
def test_think_streamed_keys(keep):
    """Keys past the memory-side cache (batch rows sharing one row's memory):
    every row selects and copies what that row alone does."""
    print(f"[case] ThinK streamed keep={keep}", flush=True)
    H, S, B = 8, 1025, 130
    K = _grid((1, H, S, 128), torch.float16, keep).expand(B, H, S, 128)
    Q = _grid((1, 2 * H, 32, 128), torch.float16, 5).expand(B, 2 * H, 32, 128)
    assert K.numel() * 2 > 256 << 20
    Kc, mask = think_score_and_compact(K, Q, H, 128 - keep)
    one, mask1 = think_score_and_compact(K[:1], Q[:1], H, 128 - keep)
    _, mask_o, _ = ob.think_score_and_compact(_np(K[:1]), _np(Q[:1]), H, 128 - keep, "float16")
    np.testing.assert_array_equal(_np(mask1), mask_o)
    assert torch.equal(mask, mask1.expand_as(mask)) and torch.equal(Kc, one.expand_as(Kc))
    want = K[:1][mask1.unsqueeze(2).expand(1, H, S, 128)].view(1, H, S, keep)
    assert torch.equal(one, want)
