"""fp32 models' blocks with packed weights and few rows: their LayerNorm runs inside the product behind it (csrc/capi.cpp,
prologue_f32), with the bits of the two launches.  Rows on both sides of a row block, of the limits and of each line
between the prologue's tiles (16 x 32, 16 x 64, 32 x 32, 32 x 64), in fp16 too; widths of each way that a row is spread over
lanes (32 or 64, whole shares or not), rows with infinities, NaN and a variance beyond fp32's range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))


def operands(rows, h, device, special):
    g = torch.Generator(device=device).manual_seed(rows * 7 + h)
    x = torch.randn(1, rows, h, generator=g, device=device) * 3
    if special:
        x[0, 0, 5] = float("inf")
        x[0, rows // 2, 0] = float("nan")
        x[0, -1] *= 1e30
    ln = [torch.randn(h, generator=g, device=device) for _ in range(2)]
    return g, x, ln


SIZES = [(rows, h) for h in (64, 320, 768) for rows in (1, 16, 17, 32, 33, 48, 49, 80, 81, 112, 113, 128, 160, 161)] + [
    (rows, h) for h in (832, 1024) for rows in (1, 24, 32, 33, 64, 65)]


@pytest.mark.parametrize("rows,h", SIZES)
def test_mlp_block(K, gpu_device, rows, h):
    for special in (False, True):
        print(f"LayerNorm in the product, fp32 rows: mlp {rows} x {h} special={special}", flush=True)
        g, x, ln = operands(rows, h, gpu_device, special)
        w1 = K.pack_weight(torch.randn(h, 4 * h, generator=g, device=gpu_device) / h ** 0.5)
        w2 = K.pack_weight(torch.randn(4 * h, h, generator=g, device=gpu_device) / h ** 0.5)
        b1, b2 = (torch.randn(n, generator=g, device=gpu_device) for n in (4 * h, h))
        inner = K.fused_ffn(K.fused_layer_norm(x, *ln), w1, bias=b1, add_gelu=True)
        want = K.fused_ffn(inner, w2, bias=b2, residual=x)
        assert same(K.mlp_block(x, *ln, w1, b1, w2, b2), want)


@pytest.mark.parametrize("rows,h", SIZES)
def test_attention_block(K, gpu_device, rows, h):
    for special in (False, True):
        print(f"LayerNorm in the product, fp32 rows: attention {rows} x {h} special={special}", flush=True)
        g, x, ln = operands(rows, h, gpu_device, special)
        w_qkv = K.pack_weight(torch.randn(h, 3 * h, generator=g, device=gpu_device) / h ** 0.5)
        w_proj = K.pack_weight(torch.randn(h, h, generator=g, device=gpu_device) / h ** 0.5)
        b_qkv, b_proj = (torch.randn(n, generator=g, device=gpu_device) for n in (3 * h, h))
        args = (x, *ln, w_qkv, b_qkv, w_proj, b_proj, h // 64)
        assert same(K.attention_block(*args), K.attention_block(*args, normed=K.fused_layer_norm(x, *ln)))


@pytest.mark.parametrize("rows", [1, 31, 33, 48, 49, 80, 81, 112, 113, 160])
def test_fp16_prologue(K, gpu_device, rows):
    h = 768
    print(f"LayerNorm in the product, fp16 rows: {rows} x {h}", flush=True)
    g, x, ln = operands(rows, h, gpu_device, False)
    x, ln = x.half(), [t.half() for t in ln]
    for n, gelu in ((4 * h, True), (3 * h, False)):
        w = K.pack_weight((torch.randn(h, n, generator=g, device=gpu_device) / h ** 0.5).half())
        b = torch.randn(n, generator=g, device=gpu_device).half()
        want = K.fused_ffn(K.fused_layer_norm(x, *ln), w, bias=b, add_gelu=gelu)
        assert torch.equal(K.layer_norm_ffn(x, *ln, w, bias=b, add_gelu=gelu), want)
