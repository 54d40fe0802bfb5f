"""Products that read a [K, N] weight as it stands: the kernels, the division of the rows and the order of the
sums are those of the packed image, so every result is compared with the packed weight's bit for bit (which
other tests hold against the oracle).  Rows either side of what the tile shapes take, columns that end inside a
tile, 8 columns in all, one k-slice and several that the groups of a workgroup do not share evenly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


def weights(device, k, n, seed):
    g = torch.Generator(device=device).manual_seed(seed)
    draw = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=device) * std).half()
    return draw, draw(k, n, std=k**-0.5), draw(n)


SHAPES = [(1, 64, 8), (1, 768, 768), (16, 3072, 768), (17, 320, 776), (33, 768, 2304), (64, 192, 72),
          (100, 1024, 1000), (128, 768, 3072), (300, 448, 520), (511, 768, 768), (777, 1024, 1032),
          (1477, 768, 3072), (1477, 3072, 768), (2400, 1280, 1288), (3001, 768, 768), (4800, 3072, 768),
          (5000, 64, 264), (4800, 768, 3072), (3885, 1024, 4096), (8193, 128, 512), (9600, 768, 2304)]


@pytest.mark.parametrize("M,k,n", SHAPES)
def test_bits_of_the_packed_weight(K, gpu_device, M, k, n):
    print(f"weight in place: {M} x {k} x {n}", flush=True)
    draw, w, b = weights(gpu_device, k, n, M)
    x, r = draw(M, k), draw(M, n)
    image = K.pack_weight(w)
    for bias, res, gelu in ((None, None, False), (b, None, True), (b, r, False)):
        plain = K.fused_ffn(x, w, bias=bias, residual=res, add_gelu=gelu)
        packed = K.fused_ffn(x, image, bias=bias, residual=res, add_gelu=gelu)
        assert torch.isfinite(plain).all() and torch.equal(plain, packed), (bias is not None, res is not None, gelu)
    shifted = torch.empty(k * n + 4, device=gpu_device, dtype=torch.float16)[4:].view(k, n)  # 8-byte aligned: packed
    shifted.copy_(w)
    assert torch.equal(K.fused_ffn(x, shifted, bias=b), K.fused_ffn(x, image, bias=b))


@pytest.mark.parametrize("B,L,heads,d", [(1, 5, 2, 8), (2, 64, 12, 64), (3, 333, 5, 32), (7, 211, 12, 64), (16, 300, 12, 64),
                                         (5, 777, 8, 128), (9, 1000, 6, 128)])
def test_head_major_scatter(K, gpu_device, B, L, heads, d):
    k = 64 * max(1, heads * d // 64)
    print(f"weight in place, q, k, v of {heads} x {d}: {B} x {L} rows of {k}", flush=True)
    draw, w, b = weights(gpu_device, k, 3 * heads * d, L)
    x = draw(B, L, k)
    for got, want in zip(K.matmul_and_split_qkv(x, w, b, heads),
                         K.matmul_and_split_qkv(x, K.pack_weight(w), b, heads)):
        assert torch.isfinite(got).all() and torch.equal(got, want)


@pytest.mark.parametrize("B,L,h,heads", [(1, 24, 128, 2), (2, 300, 768, 12), (16, 300, 768, 12), (3, 999, 1024, 16),
                                         (56, 300, 768, 12),
                                         (5, 307, 1024, 16), (3, 512, 1024, 16), (3, 341, 1280, 20), (4, 256, 1280, 20),
                                         # either side of the rows from which a block packs both weights
                                         (6, 768, 768, 12), (6, 769, 768, 12)])
def test_training_blocks(K, gpu_device, B, L, h, heads):
    """Dropout with its mask at hand and drawn in place, both blocks, weights plain and packed."""
    print(f"weight in place, training blocks: {B} x {L} rows of {h}", flush=True)
    draw, wq, bq = weights(gpu_device, h, 3 * h, B)
    _, wp, bp = weights(gpu_device, h, h, B + 1)
    _, w1, b1 = weights(gpu_device, h, 4 * h, B + 2)
    _, w2, b2 = weights(gpu_device, 4 * h, h, B + 3)
    x, lw, lb = draw(B, L, h), draw(h), draw(h)
    masks = (None, K.dropout_mask(B * L * 4 * h, 0.1, x)) if B * L < 2000 else (K.dropout_mask(B * L * 4 * h, 0.1, x),)
    for keep in masks:
        for call, ws in ((K.attention_block, (wq, bq, wp, bp)), (K.mlp_block, (w1, b1, w2, b2))):
            images = [K.pack_weight(t) if t.dim() == 2 else t for t in ws]
            more = (heads,) if call is K.attention_block else ()
            plain = call(x, lw, lb, *ws, *more, dropout_prob=0.1, keep=keep)
            packed = call(x, lw, lb, *images, *more, dropout_prob=0.1, keep=keep)
            assert torch.isfinite(plain).all() and torch.equal(plain, packed)


@pytest.mark.parametrize("B,L,h,heads", [(1, 24, 768, 12), (3, 341, 896, 14), (1, 100, 1280, 20), (2, 777, 1600, 25),
                                         (2, 150, 2048, 32), (3, 50, 2112, 33), (1, 300, 2560, 20)])
def test_blocks_of_any_width(K, gpu_device, B, L, h, heads):
    """The second weight of a block packed in the LayerNorm's launch and, behind rows that are handed in normalised and
    rows too wide for that, read in place; a second weight that has to be packed by itself."""
    print(f"weight in place, blocks: {B} x {L} rows of {h}", flush=True)
    draw, wq, bq = weights(gpu_device, h, 3 * h, B)
    _, wp, bp = weights(gpu_device, h, h, B + 1)
    _, w1, b1 = weights(gpu_device, h, 4 * h, B + 2)
    _, w2, b2 = weights(gpu_device, 4 * h, h, B + 3)
    x, lw, lb, y = draw(B, L, h), draw(h), draw(h), draw(B, L, h)
    for call, ws, rest in ((K.attention_block, (wq, bq, wp, bp, heads), {}), (K.mlp_block, (w1, b1, w2, b2), {}),
                           (K.attention_block, (wq, bq, wp, bp, heads), {"normed": y})):
        images = [K.pack_weight(t) if torch.is_tensor(t) and t.dim() == 2 else t for t in ws]
        shifted = torch.empty(ws[2].numel() + 4, device=gpu_device, dtype=torch.float16)[4:].view(ws[2].shape)
        shifted.copy_(ws[2])  # 8-byte aligned
        want = call(x, lw, lb, *images, **rest)
        assert torch.isfinite(want).all() and torch.equal(call(x, lw, lb, *ws, **rest), want)
        assert torch.equal(call(x, lw, lb, *ws[:2], shifted, *ws[3:], **rest), want)


@pytest.mark.parametrize("M,k,n", [(100, 768, 768), (128, 768, 3072), (600, 3072, 768), (4800, 6400, 768), (4700, 6400, 768)])
def test_output_over_the_weight(K, gpu_device, M, k, n):
    """A weight that the output lies over is copied before it is multiplied, the output at its start and across its
    end, in products and as the second of a block, where it is read in place otherwise."""
    print(f"output over the weight: {M} x {k} x {n}", flush=True)
    draw, w, b = weights(gpu_device, k, n, M)
    x = draw(M, k)
    want = K.fused_ffn(x, w, bias=b)
    room = torch.empty(k * n + M * n, device=gpu_device, dtype=torch.float16)
    for at in (0, k * n - min(M, k) * n // 2 // 8 * 8):
        room[:k * n] = w.view(-1)
        out = room[at:at + M * n].view(M, n)
        K._linear(x, room[:k * n].view(k, n), b, None, out, False, 0.0, K._lib.GPTMI_W_KN, "over the weight")
        assert torch.equal(out, want)
    if n % 192 == 0:
        parts = K.matmul_and_split_qkv(x.view(1, M, k), w, b, n // 192)
        lib, ws = K._lib.load(), torch.empty(k * n * 2 + 256, device=gpu_device, dtype=torch.uint8)
        ws = ws[-ws.data_ptr() % 256:]
        room[:k * n] = w.view(-1)
        q, kk, v = room[:M * n].view(3, M * n // 3)
        rc = lib.gptmi_linear_qkv(x.data_ptr(), room.data_ptr(), b.data_ptr(), q.data_ptr(), kk.data_ptr(), v.data_ptr(),
                                  1, M, n // 192, 64, k, K._lib.GPTMI_W_KN, ws.data_ptr(), k * n * 2, K._lib.GPTMI_F16,
                                  torch.cuda.current_stream().cuda_stream)
        K._lib.check(rc, "linear_qkv")
        for got, part in zip((q, kk, v), parts):
            assert torch.equal(got, part.view(-1))


def test_block_over_its_weight(K, gpu_device):
    B, L, h, heads = 2, 150, 768, 12
    print("block's output over its second weight", flush=True)
    draw, wq, bq = weights(gpu_device, h, 3 * h, 1)
    _, wp, bp = weights(gpu_device, h, h, 2)
    x, y, lw, lb = draw(B, L, h), draw(B, L, h), draw(h), draw(h)
    want = K.attention_block(x, lw, lb, wq, bq, wp, bp, heads, normed=y)
    lib = K._lib.load()
    nbytes = lib.gptmi_attention_block_workspace_bytes(B, L, heads, h // heads, K._lib.GPTMI_W_KN)
    ws = torch.empty(nbytes + 256, device=gpu_device, dtype=torch.uint8)
    ws = ws[-ws.data_ptr() % 256:]
    rc = lib.gptmi_attention_block(x.data_ptr(), y.data_ptr(), lw.data_ptr(), lb.data_ptr(), 1e-5, wq.data_ptr(),
                                   bq.data_ptr(), wp.data_ptr(), bp.data_ptr(), wp.data_ptr(), B, L, heads, h // heads, 0.0,
                                   1337, None, 0, 0, K._lib.GPTMI_W_KN, ws.data_ptr(), nbytes, K._lib.GPTMI_F16,
                                   torch.cuda.current_stream().cuda_stream)
    K._lib.check(rc, "attention_block")
    assert torch.equal(wp.view(-1)[:B * L * h], want.view(-1))
