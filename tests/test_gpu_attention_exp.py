"""The exponential of fp32 attention over its whole range: scaled scores of exact values, from 0 to far below
what fp32 holds, and keys of -inf and NaN.  q and k give every key the score -x of its own against a first key
of score 0, V is 1 behind that key and 0 at it: a row's output is sum exp(-x_j) / (1 + sum exp(-x_j)).

Bound: P rounded to fp16 (2^-11 of each weight, 2^-25 where it is smaller than fp16's smallest normal
number), relative to the denominator; everything else in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


@pytest.mark.parametrize("L", [33, 64, 300, 450])  # resident and tiled kernels, one key tile and several
@pytest.mark.parametrize("d", [32, 64, 128])
def test_weights_over_the_range(K, gpu_device, d, L):
    print(f"fp32 attention, weights from 1 to 0: d={d}, L={L}", flush=True)
    x = torch.linspace(0, 8, L, dtype=torch.float64).square() * 8  # to 512
    x[L // 2:L // 2 + 8] = 60000.0
    c = d**0.5
    k = torch.zeros(1, 2, L, d, device=gpu_device)
    k[..., 0] = -(x.to(gpu_device).float())
    k[..., 0] = k[..., 0].half().float()  # exact as a product's operand
    q = torch.zeros(1, 2, L, d, device=gpu_device)
    q[..., 0] = torch.tensor(c).half().float()
    v = torch.ones(1, 2, L, d, device=gpu_device)
    v[:, :, 0] = 0
    got = K.flash_attention_v1(q, k, v).double().cpu()[0, :, :, 0]
    s = k[0, 0, :, 0].double().cpu() * float(q[0, 0, 0, 0]) / c
    w = torch.exp(s)
    den = torch.cumsum(w, 0)
    want = (den - w[0]) / den
    below = 2.0**-25 * (s > -90).double().cumsum(0)
    tol = (2.0**-11 * (den - w[0]) + below) / den + 1e-6
    assert bool(((got - want).abs() <= tol).all()), float(((got - want).abs() - tol).max())


@pytest.mark.parametrize("L", [64, 300, 450])
def test_infinite_and_nan_keys(K, gpu_device, L):
    """Keys of -inf weigh nothing; a NaN key makes the rows that see it NaN and no others."""
    print(f"fp32 attention, infinite and NaN keys: L={L}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(L)
    q, k, v = (torch.rand(1, 3, L, 64, generator=g, device=gpu_device) + 0.1 for _ in range(3))
    gone = torch.zeros(L, dtype=torch.bool, device=gpu_device)
    gone[1::3] = True
    gone[40:60] = True
    kept = [t.half().double() for t in (q, k, v)]
    k[:, :, gone] = float("-inf")
    got = K.flash_attention_v1(q, k, v)
    s = torch.matmul(kept[0], kept[1].transpose(-1, -2).contiguous()) / 8
    mask = torch.ones((L, L), dtype=torch.bool, device=gpu_device).tril() & ~gone
    want = torch.matmul(torch.softmax(s.masked_fill(~mask, float("-inf")), dim=-1), kept[2])
    assert float(((got - want).abs() - 2.0**-11 * want).max()) <= 1e-5
    k[:, :, 50] = float("nan")
    bad = torch.isnan(K.flash_attention_v1(q, k, v))
    assert bool(bad[:, :, 50:].all()) and not bool(bad[:, :, :50].any())


@pytest.mark.parametrize("d,L", [(16, 2), (64, 2), (64, 330), (256, 40), (256, 330)])  # resident and tiled kernels
def test_the_exponential_is_the_library_s(K, gpu_device, d, L):
    """Row 1 sees scores 0 and s, exact in fp32, and values 1 and 0: its output is 1 / (1 + exp(s)) with the library's
    exponential to the last bit (operations of lower error bounds differ from it, of higher ones too).  s from
    -0.7 up, where the sum shows every other last bit of exp(s), and a tail to -16."""
    N = 2048
    print(f"fp32 attention, last bits of the exponential: d={d}, L={L}", flush=True)
    g = torch.Generator().manual_seed(d + L)
    a = (1 + torch.rand(N, generator=g)).half().double()
    s = -0.7 * torch.rand(N, generator=g, dtype=torch.float64)
    s[::8] *= 23
    b = (s / a * d**0.5).half().double()
    s = a * b / d**0.5  # 22 bits, and a power of two
    assert torch.equal(s.float().double(), s)
    q, k, v = (torch.zeros(1, N, L, d) for _ in range(3))
    q[0, :, 1, 0], k[0, :, 1, 0], v[0, :, 0] = a.float(), b.float(), 1
    got = K.flash_attention_v1(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device))[0, :, 1, 0].cpu()
    want = (1 / (1 + torch.exp(s.float().to(gpu_device)))).cpu()
    assert torch.equal(got, want), f"{int((got != want).sum())} of {N} rows"
