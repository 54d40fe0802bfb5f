"""Dropout with its mask at hand in the persistent GEMM (ffn1 of a training forward), against the launches
that draw the mask themselves, one workgroup per tile: the same sums in the same order, the same division
and the same decisions, so equal bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


# 564 tiles of 256 x 256 and more, two rounds of any launch: always the persistent kernel.  Whole row tiles
# and a last one moved up by 1 and by 255 rows; a last column tile of 64 and of 192 columns.  The first and
# the sixth: one round, sizes that the cost model gives to it.  WITH_RESIDUAL: the second product, with a
# residual, takes two rounds (the first, of 192 or 256 columns, does not matter).  test_shapes_reach_the_kernels
# of tests/test_gpu_gemm_ragged.py holds them to the cost model.
WITH_RESIDUAL = [(44031, 768, 192), (43777, 832, 256)]
SHAPES = [(4800, 768, 3072), (12032, 768, 3072), (12031, 128, 3072), (11777, 256, 3136), (12800, 192, 3008),
          (3885, 1024, 4096)] + WITH_RESIDUAL


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("p", [0.1, 0.5])
@pytest.mark.parametrize("M,h,inner", SHAPES)
def test_bits(K, gpu_device, M, h, inner, p, dtype):
    print(f"persistent GEMM with a dropout mask: M={M} h={h} inner={inner} p={p} {dtype}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(M + h)

    def draw(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=g, device=gpu_device) * std + mean).to(dtype)

    x, lw, lb = draw(M, h), draw(h, std=0.2, mean=1.0), draw(h, std=0.1)
    w1, b1 = draw(h, inner, std=h ** -0.5), draw(inner, std=0.1)
    w2, b2 = draw(inner, h, std=inner ** -0.5), draw(h, std=0.1)
    # columns whose values are zero, large, tiny and a GELU's zero (infinities: below; their products with
    # the next weights are NaN, which no equality holds for)
    w1[:, 5:9] = 0
    b1[5:9] = torch.tensor([0.0, 7.0, 1e-30, -20.0], device=gpu_device).to(dtype)
    keep = K.dropout_mask(M * max(inner, h), p, x)
    got = K.mlp_block(x, lw, lb, w1, b1, w2, b2, dropout_prob=p, keep=keep)
    assert torch.equal(got, K.mlp_block(x, lw, lb, w1, b1, w2, b2, dropout_prob=p))


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
def test_special_values(K, gpu_device, value):
    """A bias that is no number or that the division by 1 - p makes infinite: the same rows and columns."""
    print(f"persistent GEMM with a dropout mask: bias {value}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(3)
    M, h, inner, p = 12032, 64, 3072, 0.5
    x = torch.randn(M, h, generator=g, device=gpu_device)
    w1 = torch.randn(h, inner, generator=g, device=gpu_device) * 0.1
    b1 = torch.zeros(inner, device=gpu_device)
    b1[77] = value
    w2 = torch.randn(inner, h, generator=g, device=gpu_device) * 0.02
    one, zero = torch.ones(h, device=gpu_device), torch.zeros(h, device=gpu_device)
    keep = K.dropout_mask(M * inner, p, x)
    got = K.mlp_block(x, one, zero, w1, b1, w2, zero, dropout_prob=p, keep=keep)
    want = K.mlp_block(x, one, zero, w1, b1, w2, zero, dropout_prob=p)
    assert bool(((got == want) | (got.isnan() & want.isnan())).all()) and not bool(want.isfinite().all())
