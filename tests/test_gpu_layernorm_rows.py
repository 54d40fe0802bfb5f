"""LayerNorm rows (reference: fused_layer_norm_kernel, kernels.py:104-145): the row arithmetic that the
LayerNorm kernel, the embedding kernel and the GEMM prologue share, against 64 bits, and the prologue's
16-row tiles against the two launches, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


def ln64(x, w, b):
    x, w, b = x.double(), w.double(), b.double()
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * w + b, d


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("H", [8, 64, 256, 264, 768, 1024, 1280, 1600, 2048, 8192])
def test_against_64_bits(K, gpu_device, H, dtype):
    print(f"layer norm rows: H={H} {dtype}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(H)
    x = torch.randn(37, H, generator=g, device=gpu_device)
    x = (x * torch.logspace(-4, 2, 37, device=gpu_device)[:, None] + 3.0).to(dtype)
    w = (torch.randn(H, generator=g, device=gpu_device) * 0.2 + 1).to(dtype)
    b = (torch.randn(H, generator=g, device=gpu_device) * 0.1).to(dtype)
    got = K.fused_layer_norm(x, w, b).double()
    want, d = ln64(x, w, b)
    z = want - b.double()
    # u = 2^-24.  The mean: sums of up to 32 terms in a lane and 6 steps over lanes, 38 u of mean |x|,
    # which moves every element alike; then a few roundings of the element and of 1 / sigma (the sum of
    # squares, 38 u, halved by the root).  Output rounding: half an ulp of the storage type.
    u = 2.0 ** -24
    rstd = z.abs() / d.abs().clamp_min(1e-300) / w.double().abs().clamp_min(1e-300)
    bound = (38 * u * x.double().abs().mean(-1, keepdim=True) * rstd * w.double().abs() +
             (19 + 6) * u * z.abs() + 2 * u * want.abs())
    bound = bound + want.abs() * (2.0 ** -11 if dtype == torch.float16 else u) + 2.0 ** -25
    worst = ((got - want).abs() / bound).max().item()
    assert worst <= 1.0, worst


def test_special_rows(K, gpu_device):
    """What a mean, a root and a division give: a variance that overflows scales the row to 0; infinities
    and NaN make the row NaN; constant rows are the bias; neighbours are untouched."""
    w = torch.ones(768, device=gpu_device)
    b = torch.full((768,), 0.5, device=gpu_device)
    x = torch.randn(7, 768, device=gpu_device)
    plain = K.fused_layer_norm(x, w, b)
    x[1] = x[1] * 1e20          # squares overflow
    x[2, 5] = float("inf")
    x[3, 700] = float("nan")
    x[4] = 7.0                  # exact mean, variance 0
    x[5] = x[5] * 1e16          # variance 1e32, beyond 2^100
    y = K.fused_layer_norm(x, w, b)
    assert torch.equal(y[[0, 6]], plain[[0, 6]])
    assert torch.equal(y[1], b) and torch.equal(y[4], b)
    assert torch.isnan(y[2]).all() and torch.isnan(y[3]).all()
    want, _ = ln64(x[5], w, b)
    assert torch.allclose(y[5].double(), want, rtol=0, atol=1e-5)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 31, 32, 33, 48])
@pytest.mark.parametrize("H,N", [(768, 768), (768, 1192), (512, 100), (1600, 512)])
def test_prologue_of_few_rows(K, gpu_device, M, H, N):
    """Tiles of 16 rows while they run at once, of 32 beyond that: the bits of the two launches."""
    print(f"layer_norm_ffn few rows: M={M} H={H} N={N}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(M + H + N)

    def draw(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=g, device=gpu_device) * std + mean).half()

    x, lw, lb = draw(M, H, std=2.0, mean=0.3), draw(H, std=0.2, mean=1.0), draw(H, std=0.1)
    w, b = K.pack_weight(draw(H, N, std=H ** -0.5)), draw(N, std=0.1)
    z = K.layer_norm_ffn(x, lw, lb, w, bias=b, add_gelu=True)
    assert torch.equal(z, K.fused_ffn(K.fused_layer_norm(x, lw, lb), w, bias=b, add_gelu=True))
