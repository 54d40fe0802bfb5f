"""attention_block and mlp_block: a block's operators behind one call of the library, against the same
operators called one by one (fused_layer_norm, matmul_and_split_qkv, flash_attention_v1, fused_ffn),
with packed and plain weights, with and without dropout.

fp16 storage runs the very same launches on the same operands: equal bits.  fp32 storage hands fp16
copies of q, k, v and of the operands on, which the operators round to anyway; only the attention may
run another of its kernels, whose fp32 sums run in another order.  A last-bit difference there can turn
the fp16 rounding of a weight P or of the attention output, so each of the h products of the
projection may be off by 2^-11 of itself: |difference| <= 2^-11 * sum |attention| |W| is the bound; the
MLP has no attention in it: equal bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def params(h, dtype, device, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    rn = lambda *s, std=1.0, mean=0.0: (mean + std * torch.randn(*s, generator=g)).to(dtype).to(device)
    return dict(ln_w=rn(h, std=0.2, mean=1.0), ln_b=rn(h, std=0.1), qkv=rn(h, 3 * h, std=h**-0.5),
                qkv_b=rn(3 * h, std=0.1), proj=rn(h, h, std=h**-0.5), proj_b=rn(h, std=0.1),
                w1=rn(h, 4 * h, std=h**-0.5), b1=rn(4 * h, std=0.1), w2=rn(4 * h, h, std=0.5 * h**-0.5),
                b2=rn(h, std=0.1)), rn


CASES = [(1, 1, 64, 1), (2, 37, 128, 2), (3, 65, 192, 6), (2, 321, 128, 2), (6, 100, 768, 12),
         (70, 40, 64, 1), (2, 130, 256, 2), (1, 300, 256, 1), (4, 50, 64, 4)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("B,L,h,heads", CASES)
def test_attention_block(K, gpu_device, dtype, packed, p, B, L, h, heads):
    P, rn = params(h, dtype, gpu_device, seed=L + h)
    x = rn(B, L, h)
    print(f"attention_block {dtype} B={B} L={L} h={h} heads={heads} packed={packed} p={p}", flush=True)
    wq, wp = (K.pack_weight(P["qkv"]), K.pack_weight(P["proj"])) if packed else (P["qkv"], P["proj"])
    y = K.fused_layer_norm(x, P["ln_w"], P["ln_b"])
    q, k, v = K.matmul_and_split_qkv(y, wq, P["qkv_b"], heads)
    a = K.flash_attention_v1(q, k, v, dropout_prob=p, merged_heads_layout=True)
    a = a.transpose(1, 2).contiguous().view(x.shape)
    want = K.fused_ffn(a, wp, bias=P["proj_b"], residual=x, dropout_prob=p)
    for normed in (None, y):
        got = K.attention_block(x, P["ln_w"], P["ln_b"], wq, P["qkv_b"], wp, P["proj_b"], heads,
                                dropout_prob=p, normed=normed)
        if dtype == torch.float16:
            assert torch.equal(got, want)
        else:
            sums = a.abs().view(-1, h) @ P["proj"].abs()
            bound = 2.0**-11 * sums.view_as(want) / (1.0 - p) + 1e-5 * want.abs().max()
            assert float(((got - want).abs() - bound).max()) <= 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("M,h", [(1, 64), (33, 192), (600, 768), (2100, 256), (9000, 64)])
def test_mlp_block(K, gpu_device, dtype, packed, p, M, h):
    P, rn = params(h, dtype, gpu_device, seed=M + h)
    x = rn(M, h)
    print(f"mlp_block {dtype} M={M} h={h} packed={packed} p={p}", flush=True)
    w1, w2 = (K.pack_weight(P["w1"]), K.pack_weight(P["w2"])) if packed else (P["w1"], P["w2"])
    y = K.fused_ffn(K.fused_layer_norm(x, P["ln_w"], P["ln_b"]), w1, bias=P["b1"], add_gelu=True,
                    dropout_prob=p)
    want = K.fused_ffn(y, w2, bias=P["b2"], residual=x, dropout_prob=p)
    got = K.mlp_block(x, P["ln_w"], P["ln_b"], w1, P["b1"], w2, P["b2"], dropout_prob=p)
    assert torch.equal(got, want)


def test_attention_block_layer_norm_in_gemm(K, gpu_device):
    P, rn = params(768, torch.float16, gpu_device, seed=3)
    x = rn(2, 50, 768)
    wq, wp = K.pack_weight(P["qkv"]), K.pack_weight(P["proj"])
    got, want = (K.attention_block(x, P["ln_w"], P["ln_b"], wq, P["qkv_b"], wp, P["proj_b"], 12,
                                   layer_norm_in_gemm=flag) for flag in (True, False))
    assert torch.equal(got, want)


def test_blocks_turn_down_what_they_do_not_hold(K, gpu_device):
    P, rn = params(96, torch.float16, gpu_device, seed=4)
    x = rn(2, 5, 96)
    assert not K.block_supported(x, 96)
    with pytest.raises(NotImplementedError):
        K.mlp_block(x, P["ln_w"], P["ln_b"], P["w1"], P["b1"], P["w2"], P["b2"])
    P, rn = params(64, torch.float16, gpu_device, seed=5)
    x = rn(2, 5, 64)
    with pytest.raises(TypeError):
        K.mlp_block(x, P["ln_w"], P["ln_b"], K.pack_weight(P["w1"]), P["b1"], P["w2"], P["b2"])
    with pytest.raises(RuntimeError, match="GPU only"):
        K.mlp_block(x.cpu(), P["ln_w"], P["ln_b"], P["w1"], P["b1"], P["w2"], P["b2"])


# x (and LayerNorm(x)) on storage that is aligned to its element only: the operators take it
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,h,heads", [(2, 37, 128, 2), (3, 300, 64, 1)])
def test_blocks_on_unaligned_rows(K, gpu_device, dtype, B, L, h, heads):
    print(f"blocks, unaligned rows {dtype} B={B} L={L} h={h}", flush=True)
    P, rn = params(h, dtype, gpu_device, seed=L)
    shift = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
    x = shift(rn(B, L, h))
    assert x.data_ptr() % 16 == x.element_size()
    y = K.fused_layer_norm(x, P["ln_w"], P["ln_b"])
    q, k, v = K.matmul_and_split_qkv(y, P["qkv"], P["qkv_b"], heads)
    a = K.flash_attention_v1(q, k, v).transpose(1, 2).contiguous().view(x.shape)
    want = K.fused_ffn(a, P["proj"], bias=P["proj_b"], residual=x)
    # equal bits in fp16; in fp32 the bound at the head of this file
    sums = (a.abs().float().view(-1, h) @ P["proj"].abs().float()).view_as(want)
    bound = 0 if dtype == torch.float16 else 2.0**-11 * sums + 1e-5 * want.abs().max()
    for normed in (None, y, shift(y)):
        got = K.attention_block(x, P["ln_w"], P["ln_b"], P["qkv"], P["qkv_b"], P["proj"], P["proj_b"],
                                heads, normed=normed)
        assert float(((got - want).abs() - bound).max()) <= 0
    got = K.mlp_block(x, P["ln_w"], P["ln_b"], P["w1"], P["b1"], P["w2"], P["b2"])
    y = K.fused_ffn(y, P["w1"], bias=P["b1"], add_gelu=True)
    assert torch.equal(got, K.fused_ffn(y, P["w2"], bias=P["b2"], residual=x))


# where something else stands in a parameter's place the modules read it through the attribute, and
# follow it when it changes
@pytest.mark.parametrize("how", ["prune", "parametrize"])
def test_modules_with_replaced_parameters(K, gpu_device, how):
    from torch.nn.utils import parametrize, prune

    from gpt_triton_amd.gpt import FusedAttention, FusedMLP

    torch.manual_seed(2)
    x = torch.randn(2, 70, 128, device=gpu_device, dtype=torch.float16)
    for module, name in ((FusedAttention(128, 2), "c_attn_weight"), (FusedMLP(128), "ffn1_weight")):
        for prm in module.parameters():
            prm.data.normal_(0.0, 0.05)
        module = module.to(gpu_device).half().eval()
        want = module(x)
        if how == "prune":
            prune.identity(module, name)
            source = getattr(module, name + "_orig")
        else:
            parametrize.register_parametrization(module, name, torch.nn.Identity())
            source = getattr(module.parametrizations, name).original
        assert torch.equal(module(x), want)
        with torch.no_grad():
            source.mul_(2)
        changed = module(x)
        (prune.remove if how == "prune" else parametrize.remove_parametrizations)(module, name)
        assert torch.equal(changed, module(x)) and not torch.equal(changed, want)


# the modules in eval mode at row counts where the blocks run their LayerNorm inside the GEMM: rows or
# LayerNorm parameters aligned to their element only take the LayerNorm kernel
@pytest.mark.parametrize("which", ["x", "layer_norm_weight", "layer_norm_bias"])
def test_modules_on_unaligned_rows(K, gpu_device, which):
    from gpt_triton_amd.gpt import FusedAttention, FusedMLP

    print(f"FusedAttention, FusedMLP in eval mode, {which} unaligned", flush=True)
    P, rn = params(128, torch.float16, gpu_device, seed=6)
    shift = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
    x = rn(2, 37, 128)
    attn, mlp = FusedAttention(128, 2), FusedMLP(128)
    for module, keys in ((attn, ("ln_w", "ln_b", "qkv", "qkv_b", "proj", "proj_b")),
                         (mlp, ("ln_w", "ln_b", "w1", "b1", "w2", "b2"))):
        module.to(gpu_device).half().eval()
        for prm, key in zip(module.parameters(), keys):
            prm.data = P[key]
        if which != "x":
            getattr(module, which).data = shift(P["ln_w" if which.endswith("weight") else "ln_b"])
    if which == "x":
        x = shift(x)
    lw, lb = attn.layer_norm_weight.data, attn.layer_norm_bias.data
    y = K.fused_layer_norm(x, lw, lb)
    q, k, v = K.matmul_and_split_qkv(y, P["qkv"], P["qkv_b"], 2)
    a = K.flash_attention_v1(q, k, v).transpose(1, 2).contiguous().view(x.shape)
    assert torch.equal(attn(x), K.fused_ffn(a, P["proj"], bias=P["proj_b"], residual=x))
    y = K.fused_ffn(y, P["w1"], bias=P["b1"], add_gelu=True)
    assert torch.equal(mlp(x), K.fused_ffn(y, P["w2"], bias=P["b2"], residual=x))


# modules whose weights were exchanged for others: an inner width that is not a multiple of 64 (the
# operators take it, the block call does not), one above 4h (a forward's dropout mask is too short for
# it), rows of another width than the module was built for
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [70, 700])
@pytest.mark.parametrize("h,inner", [(128, 100), (128, 640), (96, 512), (192, 512)])
@pytest.mark.parametrize("p", [0.0, 0.1])
def test_mlp_of_other_widths(K, gpu_device, dtype, rows, h, inner, p):
    from gpt_triton_amd.gpt import FusedMLP

    print(f"FusedMLP {dtype} rows={rows} h={h} inner={inner} p={p}", flush=True)
    P, rn = params(h, dtype, gpu_device, seed=inner)
    x = rn(rows, h)
    mlp = FusedMLP(128, dropout_prob=p).to(gpu_device).to(dtype).train(p > 0)
    w1, b1, w2 = rn(h, inner, std=0.1), rn(inner), rn(inner, h, std=0.1)
    for prm, t in zip(mlp.parameters(), (P["ln_w"], P["ln_b"], w1, b1, w2, P["b2"])):
        prm.data = t
    y = K.fused_layer_norm(x, P["ln_w"], P["ln_b"])
    y = K.fused_ffn(y, w1, bias=b1, add_gelu=True, dropout_prob=p)
    want = K.fused_ffn(y, w2, bias=P["b2"], residual=x, dropout_prob=p)
    keeps = [None] if p == 0 else [None, K.dropout_mask(4 * x.numel(), p, x)]
    for keep in keeps:
        assert torch.equal(mlp(x, keep=keep), want)


@pytest.mark.parametrize("p", [0.0, 0.1])
def test_attention_of_another_width(K, gpu_device, p):
    from gpt_triton_amd.gpt import FusedAttention

    print(f"FusedAttention of 96-wide rows p={p}", flush=True)
    P, rn = params(96, torch.float16, gpu_device, seed=8)
    x = rn(2, 35, 96)
    attn = FusedAttention(192, 3, dropout_prob=p).to(gpu_device).half().train(p > 0)
    for prm, key in zip(attn.parameters(), ("ln_w", "ln_b", "qkv", "qkv_b", "proj", "proj_b")):
        prm.data = P[key]
    q, k, v = K.matmul_and_split_qkv(K.fused_layer_norm(x, P["ln_w"], P["ln_b"]), P["qkv"], P["qkv_b"], 3)
    a = K.flash_attention_v1(q, k, v, dropout_prob=p).transpose(1, 2).contiguous().view(x.shape)
    want = K.fused_ffn(a, P["proj"], bias=P["proj_b"], residual=x, dropout_prob=p)
    assert torch.equal(attn(x), want)


def test_no_rows_are_refused_as_the_operators_refuse_them(K, gpu_device):
    P, rn = params(64, torch.float16, gpu_device, seed=7)
    x = rn(0, 5, 64)
    with pytest.raises(RuntimeError, match="status -1"):
        K.fused_layer_norm(x, P["ln_w"], P["ln_b"])
    with pytest.raises(RuntimeError, match="status -1"):
        K.attention_block(x, P["ln_w"], P["ln_b"], P["qkv"], P["qkv_b"], P["proj"], P["proj_b"], 1)
    with pytest.raises(RuntimeError, match="status -1"):
        K.mlp_block(x, P["ln_w"], P["ln_b"], P["w1"], P["b1"], P["w2"], P["b2"])
