"""Attention whose scaled scores are large: |scale * q.k| times 2^-24 is then far above the last bit of
a weight, and what the softmax rounds, and where, shows in the output.  Scores are made exact (constant q
and k), V is 1 in the first key tile and 0 behind it, so that the output of a row is the share of the
first tile in its denominator.

fp32 storage: all scores are equal to m / scale.  exp(scale s - max) is then exp of the rounding error of
m, at most 2^-24 |m| (1 in P, which is rounded to fp16), the rescaling between tiles exactly 1; a
32-element sum per lane, its partner's, and one addition per tile: (33 + tiles) 2^-24, and 8 * 2^-24 for
exp and the division."""
import numpy as np
import pytest
import torch

from oracle import gpt2_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def worst_rounding(d):
    """fp16 values a, b whose score d*a*b (exact in fp32) times 1/sqrt(d) rounds to fp32 with nearly
    half a unit in the last place, scaled score around 700."""
    scale = np.float32(1 / np.sqrt(d))
    best = None
    a = 8.0
    for b in 700 / float(scale) / d / a + np.arange(400) / 64.0:
        b = float(np.float16(b))
        exact = float(scale) * d * a * b
        err = abs(float(scale * np.float32(d * a * b)) - exact) / exact
        if best is None or err > best[0]:
            best = (err, a, b, exact)
    return best


@pytest.mark.parametrize("d", [32, 128])
@pytest.mark.parametrize("L", [64, 300, 1024])
def test_equal_scores_fp32(K, gpu_device, d, L):
    err, a, b, m = worst_rounding(d)
    print(f"fp32 attention d={d} L={L}: scaled scores {m:.1f}, product rounded by {err:.2e}", flush=True)
    q = torch.full((1, 2, L, d), a, device=gpu_device)
    k = torch.full((1, 2, L, d), b, device=gpu_device)
    v = torch.zeros((1, 2, L, d), device=gpu_device)
    v[:, :, :64] = 1.0
    got = K.flash_attention_v1(q, k, v).double().cpu()
    rows = torch.arange(L, dtype=torch.float64)
    want = (torch.clamp(rows + 1, max=64) / (rows + 1)).view(1, 1, L, 1)
    tiles = (L + 63) // 64
    bound = (m + 33 + tiles + 8) * 2.0**-24
    rel = float(((got - want).abs() / want).max())
    assert rel <= bound, f"relative error {rel:.2e}, bound {bound:.2e}"


def test_large_scores_dropout_fp16(K, gpu_device):
    """fp16 storage with dropout: the second key tile's scores are 1 above the first's, at scaled scores
    around 504000 (scale = 1/8 and the scores, whole numbers below 2^24, are exact).  What is left is the
    rounding of P / (1 - p) and of the output to fp16, half a unit each, and exp: 3 * 2^-11."""
    L, d, p = 128, 64, 0.1
    for b in (246, 247, 249, 250):
        q = np.full((1, 1, L, d), 256, np.float16)
        k = np.full((1, 1, L, d), b, np.float16)
        q[..., -1] = 1
        k[..., -1] = 0
        k[:, :, 64:, -1] = 8
        v = np.zeros((1, 1, L, d), np.float16)
        v[:, :, :64] = 1
        print(f"fp16 attention with dropout, scaled scores {256 * 63 * b / 8:.0f}", flush=True)
        got = K.flash_attention_v1(*(torch.from_numpy(t).to(gpu_device) for t in (q, k, v)), dropout_prob=p)
        want = O.flash_attention_v1(q, k, v, dropout_prob=p).astype(np.float64)
        rel = np.abs(got.cpu().numpy().astype(np.float64) - want) / np.maximum(np.abs(want), 2.0**-10)
        assert rel.max() <= 3 * 2.0**-11, f"relative error {rel.max():.2e}"
