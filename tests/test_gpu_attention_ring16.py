"""The ring kernel with 16 queries a wavefront (csrc/flash_attn.hip, launch_d64): few 64-row blocks take it, and its
results are those of the kernel that serves many, bit for bit.  The same pairs by themselves and among as many as
another kernel takes; lengths on both sides of a wavefront's, a block's and a tile's edge and of each line of the rule,
both output layouts, sharp and flat distributions, and the fp32 arithmetic of fp32 models (through a block call
whose products are permutations, so exact whatever their tiles)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def reference(q, k, v):
    q, k, v = (t.double() for t in (q, k, v))
    L = q.shape[2]
    s = q @ k.transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1])
    s = s.masked_fill(~torch.ones(L, L, dtype=torch.bool, device=q.device).tril(), -math.inf)
    return s.softmax(-1) @ v


# pairs that take it, pairs beyond the line, rows (256 CUs: at most 1536 blocks of one tile, 512, 640 of more than 448 rows)
CASES = [(1, 1600, 1), (3, 1600, 15), (7, 1540, 16), (5, 1540, 17), (1530, 1540, 33), (24, 1600, 64), (255, 260, 65),
         (13, 300, 100), (256, 520, 128), (12, 513, 129), (84, 200, 211), (102, 110, 289), (12, 192, 300),
         (102, 103, 320), (12, 90, 321), (73, 74, 448), (80, 81, 449), (12, 90, 511), (12, 90, 513), (39, 64, 1024),
         (2, 20, 2100)]
# the streaming kernel's lengths: either side of every 32-row chunk and 64-key tile
CASES += [(4, 1540, L) for L in (31, 32, 48, 63)]
CASES += [(4, 700, L) for L in (66, 95, 96, 97, 127, 159, 160, 161, 191, 192, 193, 223, 224, 225, 255, 256, 257, 287, 288)]


@pytest.mark.parametrize("few,many,L", CASES)
def test_same_bits_as_among_many(K, gpu_device, few, many, L):
    g = torch.Generator(device=gpu_device).manual_seed(L)
    for std, merged in ((1.0, True), (4.0, False)):
        print(f"attention, 16 queries a wavefront: pairs={few} of {many} L={L} std={std}", flush=True)
        q, k, v = (torch.randn(many, 1, L, 64, generator=g, device=gpu_device).mul_(std).half() for _ in range(3))
        all_of_them = K.flash_attention_v1(q, k, v, merged_heads_layout=merged)
        got = K.flash_attention_v1(*(t[:few].contiguous() for t in (q, k, v)), merged_heads_layout=merged)
        assert torch.equal(got, all_of_them[:few])
        n = min(few, 3)
        want = reference(q[:n], k[:n], v[:n])
        # P and the result are rounded to fp16 (2^-11 each), the weights of a row sum to 1
        bound = 3 * 2.0 ** -11 * float(v[:n].abs().max())
        assert float((got[:n].reshape(want.shape).double() - want).abs().max()) <= bound


@pytest.mark.parametrize("few,many,L", [(1, 129, 64), (2, 33, 128), (1, 43, 128), (5, 20, 200), (2, 13, 300),
                                        (12, 13, 320), (1, 9, 500), (3, 5, 1024)])
def test_same_bits_in_fp32_arithmetic(K, gpu_device, few, many, L):
    heads, h = 12, 768
    print(f"attention in fp32, 16 queries a wavefront: sequences={few} of {many} L={L}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(L)
    eye = torch.eye(h, device=gpu_device)
    w_qkv = torch.cat([eye.roll(s, 1) for s in (0, 64, 128)], 1).contiguous()
    ones, zeros = torch.ones(h, device=gpu_device), torch.zeros(3 * h, device=gpu_device)
    rows = torch.randn(many, L, h, generator=g, device=gpu_device)

    def block(n):
        x = torch.zeros(n, L, h, device=gpu_device)
        return K.attention_block(x, ones, zeros[:h], w_qkv, zeros, eye, zeros[:h], heads, normed=rows[:n].contiguous())

    got = block(few)
    assert torch.equal(got, block(many)[:few])
    r = rows[:1].half()
    q, k, v = (r.roll(s, 2).view(1, L, heads, 64).transpose(1, 2) for s in (0, 64, 128))
    want = reference(q, k, v).transpose(1, 2).reshape(1, L, h)
    assert float((got[:1].double() - want).abs().max()) <= 3 * 2.0 ** -11 * float(v.abs().max())
