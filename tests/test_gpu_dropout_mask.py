"""dropout_mask (the generator's decisions as bits) against the oracle's generator, and the block
functions and the model reading it against the same kernels drawing the masks themselves: the same
decisions and the same arithmetic on what is kept, so equal bits."""
import numpy as np
import pytest
import torch

from oracle import gpt2_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


@pytest.mark.parametrize("bits", [1, 31, 32, 33, 8191, 8192 * 32 + 5, 1 << 20])
@pytest.mark.parametrize("p", [0.1, 0.5, 0.999])
def test_mask_bits(K, gpu_device, bits, p):
    print(f"dropout_mask {bits} p={p}", flush=True)
    like = torch.empty(1, device=gpu_device)
    words = K.dropout_mask(bits, p, like).data.cpu().numpy().view(np.uint8)
    got = np.unpackbits(words, bitorder="little")[:bits].astype(bool)
    u = O.tl_rand(1337, np.arange(bits, dtype=np.uint32))
    assert np.array_equal(got, u > np.float32(p))


def block_params(h, dtype, device, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    rn = lambda *s, std=1.0, mean=0.0: (mean + std * torch.randn(*s, generator=g)).to(dtype).to(device)
    ln = (rn(h, std=0.2, mean=1.0), rn(h, std=0.1))
    att = (rn(h, 3 * h, std=h**-0.5), rn(3 * h, std=0.1), rn(h, h, std=h**-0.5), rn(h, std=0.1))
    mlp = (rn(h, 4 * h, std=h**-0.5), rn(4 * h, std=0.1), rn(4 * h, h, std=0.5 * h**-0.5),
           rn(h, std=0.1))
    return ln, att, mlp, rn


# head sizes 16 to 256; one row, ragged tiles, sequences whose rows of the attention mask start at
# every bit of a word, and L * L beyond the matrices' offsets
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,h,heads", [(1, 1, 64, 1), (3, 65, 192, 6), (2, 37, 128, 8), (2, 321, 128, 2),
                                         (6, 100, 768, 12), (1, 300, 256, 2), (2, 130, 256, 1),
                                         (16, 300, 128, 2), (1, 1023, 64, 1)])
def test_blocks_with_the_mask(K, gpu_device, dtype, B, L, h, heads):
    print(f"blocks with a dropout mask {dtype} B={B} L={L} h={h} heads={heads}", flush=True)
    ln, att, mlp, rn = block_params(h, dtype, gpu_device, seed=L + h)
    x, p = rn(B, L, h), 0.1
    keep = K.dropout_mask(max(4 * x.numel(), L * L), p, x)
    want = K.attention_block(x, *ln, *att, heads, dropout_prob=p)
    got = K.attention_block(x, *ln, *att, heads, dropout_prob=p, keep=keep)
    assert torch.equal(got, want)
    want = K.mlp_block(x, *ln, *mlp, dropout_prob=p)
    assert torch.equal(K.mlp_block(x, *ln, *mlp, dropout_prob=p, keep=keep), want)
    with pytest.raises(ValueError):
        K.mlp_block(x, *ln, *mlp, dropout_prob=0.2, keep=keep)
    with pytest.raises(RuntimeError, match="mask"):
        K.mlp_block(x, *ln, *mlp, dropout_prob=p, keep=K.dropout_mask(4 * x.numel() - 1, p, x))


def test_training_forward_module_by_module(K, gpu_device):
    """FusedGPT draws one mask; its modules called one by one draw their own.  A module with another
    dropout probability, and another module in an MLP's place, do not take the model's mask."""
    from gpt_triton_amd.gpt import FusedGPT, GPTConfig

    cfg = GPTConfig(vocab_size=512, block_size=128, n_layer=3, n_head=2, n_embd=128, dropout=0.1)
    model = FusedGPT(cfg).init_synthetic_().to(gpu_device).half().train()
    model.blocks[1][0].dropout_prob = 0.3
    model.blocks[2][1] = torch.nn.Identity()
    seen = []
    model.blocks[0].register_forward_hook(lambda *_: seen.append(1))
    ids = torch.randint(0, 512, (3, 77), device=gpu_device)
    with torch.no_grad():
        got = model(ids)
        x = K.fused_embeddings(ids, model.wte_weight.data, model.wpe_weight.data, dropout_prob=0.1)
        for block in model.blocks:
            for module in block:
                x = module(x)
        want = K.fused_layer_norm(x, model.layer_norm_weight.data, model.layer_norm_bias.data)
    assert torch.equal(got, want) and seen == [1]


# one chunk of columns, workgroups of several rows with idle threads, exactly 256 and just past 256
# chunks, rows that are no whole chunks; fewer rows than a workgroup takes and many
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,H", [(1, 1, 8), (2, 5, 768), (3, 700, 96), (1, 9, 2048), (2, 3, 2056), (1, 7, 100),
                                   (1, 7, 1024), (1, 7, 1028)])
def test_embedding_dropout(K, gpu_device, dtype, B, L, H):
    print(f"embedding dropout {dtype} B={B} L={L} H={H}", flush=True)
    r = np.random.default_rng(H + L)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    wte, wpe = r.standard_normal((50, H)).astype(npdt), r.standard_normal((L, H)).astype(npdt)
    ids = r.integers(0, 50, (B, L))
    got = K.fused_embeddings(*(torch.from_numpy(t).to(gpu_device) for t in (ids, wte, wpe)), dropout_prob=0.1)
    assert np.array_equal(got.cpu().numpy(), O.fused_embeddings(ids, wte, wpe, dropout_prob=0.1))


# x / (1 - p) in fp32 from the smallest subnormal to the largest finite value, infinities and NaN: the
# correctly rounded quotient, as a true division gives it
@pytest.mark.parametrize("p", [0.1, 0.5, 0.9])
def test_division_over_the_whole_range(K, gpu_device, p):
    print(f"dropout of fp32 values of every magnitude, p={p}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(9)
    bits = torch.arange(0, 255 << 23, 1 << 19, dtype=torch.int64)  # 16 values an octave, subnormals too
    bits = bits + torch.randint(0, 1 << 19, bits.shape, generator=g)
    special = torch.tensor([0, 1, 2, 3, 0x7fffff, 0x800000, 0x7f7fffff, 0x7f800000, 0x7fc00000])
    bits = torch.cat([bits, special, torch.arange(0x0c000000, 0x0d000000, 0x3331)])
    x = bits.to(torch.int32).view(torch.float32)
    x = torch.cat([x, -x])
    x = torch.cat([x, x.new_zeros(-len(x) % 64)])
    N = len(x)
    with np.errstate(all="ignore"):
        want = torch.from_numpy(x.numpy() / (np.float32(1) - np.float32(p)))
    keep = torch.from_numpy(O.tl_rand(O.SEED, np.arange(N)) > np.float32(p))
    want = torch.where(keep, want, torch.zeros(()))
    same = lambda a, b: bool(((a == b) | (a.isnan() & b.isnan())).all())
    xd = x.to(gpu_device)
    got = K.fused_embeddings(torch.zeros((1, 1), dtype=torch.int64, device=gpu_device), xd[None],
                             torch.zeros((1, N), device=gpu_device), dropout_prob=p)[0, 0].cpu()
    assert same(got, want), "embedding"
    # a zero product and the values as the bias; offsets m * N + n: the columns of row 0
    z = torch.zeros((1, 64), device=gpu_device)
    got = K.fused_ffn(z, torch.zeros((64, N), device=gpu_device), bias=xd, dropout_prob=p)[0].cpu()
    assert same(got, want), "fused_ffn"
