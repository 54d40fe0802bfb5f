"""The front of an attention block of short sequences in one launch (fp16, head size 64, up to 32 rows a sequence, rows of
up to 768): the bits of the operators it stands for, at lengths from 1 to beyond its last, head counts that fill
its column blocks and k-slices unevenly, pair counts up to and beyond the number of CUs, and with what makes the
block take its launches one by one (a bias or rows that are not 16-byte aligned)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


def shifted(t):
    """A copy 8 bytes off a 16-byte boundary."""
    buf = torch.empty(t.numel() + 4, device=t.device, dtype=t.dtype)[4:].view(t.shape)
    return buf.copy_(t)


@pytest.mark.parametrize("B,L,heads", [(1, 1, 1), (1, 2, 2), (3, 16, 3), (1, 17, 5), (1, 24, 12), (2, 31, 7), (4, 32, 12),
                                       (1, 33, 12), (21, 32, 12), (22, 32, 12), (64, 8, 4), (128, 30, 2), (256, 5, 1),
                                       (257, 5, 1)])
def test_bits_of_the_operators(K, gpu_device, B, L, heads):
    print(f"attention front: {B} x {L} rows, {heads} heads", flush=True)
    h = 64 * heads
    g = torch.Generator(device=gpu_device).manual_seed(L)
    draw = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=gpu_device) * std).half()
    x, lw, lb, bq, bp = draw(B, L, h), draw(h), draw(h, std=0.1), draw(3 * h), draw(h)
    wq, wp = (K.pack_weight(draw(h, n, std=h**-0.5)) for n in (3 * h, h))

    def operators(x):
        normed = K.fused_layer_norm(x, lw, lb)
        q, k, v = K.matmul_and_split_qkv(normed, wq, bq, heads)
        y = K.flash_attention_v1(q, k, v, merged_heads_layout=True).transpose(1, 2).contiguous().view(B, L, h)
        return normed, K.fused_ffn(y, wp, bias=bp, residual=x)

    normed, want = operators(x)
    assert torch.isfinite(want).all()
    assert torch.equal(K.attention_block(x, lw, lb, wq, bq, wp, bp, heads), want)
    assert torch.equal(K.attention_block(x, lw, lb, wq, bq, wp, bp, heads, normed=normed), want)
    assert torch.equal(K.attention_block(x, lw, lb, wq, shifted(bq), wp, bp, heads), want)
    x8 = shifted(x)  # LayerNorm sums such rows in another order
    assert torch.equal(K.attention_block(x8, lw, lb, wq, bq, wp, bp, heads), operators(x8)[1])


def test_not_finite(K, gpu_device):
    """A row that is not finite spoils what it spoils in the operators, and no other sequence."""
    g = torch.Generator(device=gpu_device).manual_seed(3)
    draw = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=gpu_device) * std).half()
    x, lw, lb, bq, bp = draw(3, 20, 768), draw(768), draw(768), draw(2304), draw(768)
    wq, wp = (K.pack_weight(draw(768, n, std=768**-0.5)) for n in (2304, 768))
    clean = K.attention_block(x, lw, lb, wq, bq, wp, bp, 12)
    x[1, 7, 5] = float("inf")
    bad = K.attention_block(x, lw, lb, wq, bq, wp, bp, 12)
    q, k, v = K.matmul_and_split_qkv(K.fused_layer_norm(x, lw, lb), wq, bq, 12)
    y = K.flash_attention_v1(q, k, v, merged_heads_layout=True).transpose(1, 2).contiguous().view(x.shape)
    want = K.fused_ffn(y, wp, bias=bp, residual=x)
    assert torch.equal(bad[0], clean[0]) and torch.equal(bad[2], clean[2])
    assert torch.equal(torch.isnan(bad), torch.isnan(want)) and bool(torch.isnan(bad[1, 7:]).all())
