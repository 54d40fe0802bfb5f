"""A block's LayerNorm and the images of its two weights in one launch: blocks with plain weights against
the same blocks with images built beforehand, bit for bit, at the edges of the rule that joins the two."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


# 64, 768: 32 lanes a row; 1024, 1600, 2048: 64; fp32 1600 and fp16 2112 are more than 4 chunks a lane
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("h,rows", [(64, 1), (64, 7), (768, 9), (768, 300), (1024, 5), (1600, 3), (2048, 6),
                                    (2112, 4)])
@pytest.mark.parametrize("unaligned", ["", "x", "weight"])
def test_bits(K, gpu_device, h, rows, dtype, unaligned):
    print(f"layer norm and weight images: h={h} rows={rows} {dtype} unaligned={unaligned!r}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(h + rows)

    def draw(*shape, std=1.0, mean=0.0, shift=False):
        n = 1
        for s in shape:
            n *= s
        flat = (torch.randn(n + 1, generator=g, device=gpu_device) * std + mean).to(dtype)
        return (flat[1:] if shift else flat[:-1]).view(shape)

    x = draw(1, rows, h, std=2.0, shift=unaligned == "x")
    lw, lb = draw(h, std=0.2, mean=1.0), draw(h, std=0.1)
    std = h ** -0.5
    a1, a1b = draw(h, 3 * h, std=std, shift=unaligned == "weight"), draw(3 * h, std=0.1)
    a2, a2b = draw(h, h, std=std), draw(h, std=0.1)
    m1, m1b = draw(h, 2 * h, std=std), draw(2 * h, std=0.1)
    m2, m2b = draw(2 * h, h, std=std, shift=unaligned == "weight"), draw(h, std=0.1)
    heads = h // 64 if h % 64 == 0 else 1
    got = K.attention_block(x, lw, lb, a1, a1b, a2, a2b, heads)
    want = K.attention_block(x, lw, lb, K.pack_weight(a1), a1b, K.pack_weight(a2), a2b, heads)
    assert torch.equal(got, want)
    got = K.mlp_block(x, lw, lb, m1, m1b, m2, m2b)
    want = K.mlp_block(x, lw, lb, K.pack_weight(m1), m1b, K.pack_weight(m2), m2b)
    assert torch.equal(got, want)
