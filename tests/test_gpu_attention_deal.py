"""How the (batch, head) pairs and query blocks of the long-sequence attention kernels are dealt to workgroups:
fewer and more than 1024 of them (one group of pairs per XCD, several), pair counts that are and are not a
multiple of 8, a last group that is not full, and sequences that end inside a query block.  Every element
against the textbook attention in fp32, in an output filled with NaN.

Bound: the weights are rounded to fp16 (2^-11 of each, so of sum_j P_j |v_j|), and so is the output; sums
and the exponential in fp32, 2e-5."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


def excess_over_bound(q, k, v, got):
    """Largest |got - textbook| beyond the bound."""
    L, scale = q.shape[2], 1 / math.sqrt(q.shape[3])
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) * scale
    mask = torch.ones((L, L), dtype=torch.bool, device=q.device).tril()
    p = torch.softmax(s.masked_fill(~mask, float("-inf")), dim=-1)
    want, spread = torch.matmul(p, v.float()), torch.matmul(p, v.float().abs())
    tol = 2.0**-11 * want.abs() + (2.0**-11 + 2e-5) * spread + 1e-6
    return float(((got.float() - want).abs() - tol).max())


# 64: 3 blocks of queries a pair; 128 and 256 likewise at 300 rows, 2 at 129
@pytest.mark.parametrize("B,N,L,d", [(1, 5, 330, 64), (1, 8, 513, 64), (7, 48, 330, 64), (1, 343, 330, 64),
                                     (8, 43, 384, 64), (4, 129, 321, 64), (1, 3, 300, 128), (1, 347, 300, 128),
                                     (3, 171, 129, 128), (2, 172, 300, 256)])
def test_every_pair_and_block(K, gpu_device, B, N, L, d):
    print(f"attention dealt to workgroups: {B * N} pairs, L={L}, d={d}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(L + N)
    q, k, v = (torch.randn(B, N, L, d, generator=g, device=gpu_device).half() for _ in range(3))
    out = torch.full((B, L, N, d), float("nan"), device=gpu_device, dtype=torch.float16)
    lib = K._lib.load()
    rc = lib.gptmi_flash_attn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, N, L, L, d,
                              1 / math.sqrt(d), 0.0, 1337, K._lib.GPTMI_O_BLND, K._lib.GPTMI_F16,
                              torch.cuda.current_stream().cuda_stream)
    K._lib.check(rc, "flash_attn")
    got = out.transpose(1, 2)
    assert not torch.isnan(got).any(), "elements never written"
    for b in range(B):
        worst = excess_over_bound(q[b:b + 1], k[b:b + 1], v[b:b + 1], got[b:b + 1])
        assert worst <= 0, f"beyond the rounding bound by {worst:.3e} in batch {b}"


# pairs tied to no XCD behind and without tied ones: fewer than 8 pairs, one pair more than 8, no whole eights
@pytest.mark.parametrize("B,N,L,d", [(1, 1, 4096, 64), (1, 9, 14600, 64), (1, 1, 2000, 128), (2, 21, 700, 256),
                                     (1, 131, 1000, 128)])
def test_pairs_of_no_xcd(K, gpu_device, B, N, L, d):
    test_every_pair_and_block(K, gpu_device, B, N, L, d)


def test_more_pairs_than_a_grid_dimension(K, gpu_device):
    """65600 pairs of 129 rows, the fewest that the wide kernel takes at d = 128."""
    test_every_pair_and_block(K, gpu_device, 41, 1600, 129, 128)


# the ring kernel, fewer and more than 1024 blocks, whole eights of pairs and not; the wide kernel likewise
@pytest.mark.parametrize("B,heads,L,d", [(3, 3, 330, 64), (43, 8, 330, 64), (49, 7, 330, 64), (5, 3, 300, 128), (87, 4, 300, 128),
                                         (2, 3, 129, 256), (174, 2, 300, 256)])
def test_blocks_of_fp32_models(K, gpu_device, B, heads, L, d):
    """The forms with the fp32 softmax, which an attention block of fp32 storage runs on its fp16 q, k, v: weights of
    one identity each make these the normalised rows and the projection the attention's output."""
    print(f"fp32 attention block dealt to workgroups: {B * heads} pairs, L={L}, d={d}", flush=True)
    h = heads * d
    g = torch.Generator(device=gpu_device).manual_seed(L + B)
    x = torch.randn(B, L, h, generator=g, device=gpu_device)
    one, zero = torch.ones(h, device=gpu_device), torch.zeros(3 * h, device=gpu_device)
    eye = torch.eye(h, device=gpu_device)
    y = K.fused_layer_norm(x, one, zero[:h])
    got = K.attention_block(x, one, zero[:h], eye.repeat(1, 3).contiguous(), zero, eye, zero[:h], heads) - x
    assert torch.isfinite(got).all()
    q = y.half().view(B, L, heads, d).transpose(1, 2).contiguous()
    got = got.view(B, L, heads, d).transpose(1, 2)
    for b in range(B):
        worst = excess_over_bound(q[b:b + 1], q[b:b + 1], q[b:b + 1], got[b:b + 1])
        assert worst <= 0, f"beyond the rounding bound by {worst:.3e} in batch {b}"
