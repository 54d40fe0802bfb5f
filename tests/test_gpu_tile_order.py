"""The order in which a product's tiles are dealt to the XCDs (column_group): every tile is formed once, whatever
the group's width.  Shapes on both sides of each line of the rule: 128 rows, a weight of 2^19 * 5 elements, K = N, as many
tiles as CUs, groups that do not divide the columns, the scatter.  All ones and small whole numbers, so that every sum
is exact in fp32 and in the fp16 result (at most 5 * 2^8 of them, no result beyond 2^11): the comparison is for equality."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def exact_operands(M, N, Kd, device, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.zeros(M, Kd)
    x[:, ::max(1, Kd // 256)] = torch.randint(-2, 3, (M, len(range(0, Kd, max(1, Kd // 256)))), generator=g).float()
    w = torch.randint(-1, 2, (Kd, N), generator=g).float()
    res = torch.randint(-64, 65, (M, N), generator=g).float()
    return x.to(device), w.to(device), res.to(device)


SHAPES = [(24, 768, 768), (127, 2304, 768), (128, 3072, 768), (129, 768, 3072), (129, 3072, 768), (300, 1032, 512),
          (320, 2304, 1152), (300, 3200, 832), (777, 1600, 1600), (900, 1024, 4096), (1477, 768, 768), (2000, 1288, 640),
          (3885, 1024, 1088), (4100, 4096, 640), (4352, 3840, 704)]


@pytest.mark.parametrize("M,N,Kd", SHAPES)
def test_every_tile_once(K, gpu_device, M, N, Kd):
    print(f"tile order {M} x {N} x {Kd}", flush=True)
    x, w, res = exact_operands(M, N, Kd, gpu_device, M + N)
    want = x @ w
    assert float(want.abs().max()) <= 2048 - 64
    packed = K.pack_weight(w.half())
    for weight in (w.half(), packed):
        assert torch.equal(K.fused_ffn(x.half(), weight).float(), want)
        assert torch.equal(K.fused_ffn(x.half(), weight, residual=res.half()).float(), want + res)


@pytest.mark.parametrize("B,L,heads,h", [(2, 64, 12, 768), (3, 43, 12, 768), (1, 300, 20, 1280), (5, 777, 16, 1024)])
def test_every_tile_once_scattered(K, gpu_device, B, L, heads, h):
    print(f"tile order, scatter {B} x {L} x {h}", flush=True)
    x, w, _ = exact_operands(B * L, 3 * h, h, gpu_device, B + L)
    got = K.matmul_and_split_qkv(x.half().view(B, L, h), K.pack_weight(w.half()),
                                 torch.zeros(3 * h, device=gpu_device, dtype=torch.float16), heads)
    want = (x @ w).view(B, L, 3, heads, h // heads)
    for i, t in enumerate(got):
        assert torch.equal(t.float(), want[:, :, i].transpose(1, 2))
