"""Attention dropout with the mask's bits at hand in the streaming kernel and, where that has the pairs and rows
for it, in the tiled one (head size 64, up to 320 rows; masked_streams in flash_attn.hip), against the tiled
kernel that draws them: the same sums in the same order, so equal bits.  Fewer and more (batch, head) pairs
than the 256 CUs, so that workgroups go on to a second pair; chunk counts from one to ten, mask rows that start
at every bit of a word."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L", [(1, 1), (1, 320), (90, 17), (90, 32), (90, 33), (90, 64), (90, 127), (90, 211),
                                 (90, 257), (90, 319), (180, 320),
                                 # streaming, one round of pairs: one to four chunks, nine and ten
                                 (30, 17), (30, 32), (85, 33), (30, 64), (85, 127), (30, 288), (43, 289), (85, 320),
                                 # streaming, more rounds: three chunks, five, ten; the tiled kernel beside them
                                 (171, 65), (171, 96), (170, 96), (171, 97), (90, 129), (90, 288), (114, 319),
                                 (113, 319), (42, 320)])
def test_bits(K, gpu_device, B, L, dtype):
    heads, h, p = 3, 192, 0.1
    print(f"attention block with a dropout mask: B={B} L={L} {dtype}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(B + L)

    def draw(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=g, device=gpu_device) * std + mean).to(dtype)

    # scores of several units, so that the running maximum moves from tile to tile
    args = (draw(B, L, h), draw(h, std=0.2, mean=1.0), draw(h, std=0.1), draw(h, 3 * h, std=2 * h ** -0.5),
            draw(3 * h, std=0.1), draw(h, h, std=h ** -0.5), draw(h, std=0.1), heads)
    keep = K.dropout_mask(max(B * L * h, L * L), p, args[0])
    got = K.attention_block(*args, dropout_prob=p, keep=keep)
    assert torch.equal(got, K.attention_block(*args, dropout_prob=p))
