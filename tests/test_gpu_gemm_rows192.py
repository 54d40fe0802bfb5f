"""Tiles of 192 rows in the persistent kernel without a residual (csrc/gemm.hip): where the rule takes them, and that
every row is formed once and right: whole and ragged last row tiles, several tiles a workgroup, a last column tile of 64
columns, two k-tiles, rows left to the tile kernel, the scatter, the weight in place, the three output types.  Small whole
numbers, so that every sum is exact in fp32 and, below 2^11, in fp16: the comparison is for equality."""
import math
import os
import re

import pytest
import torch

import test_gpu_gemm_ragged as ragged
from test_gpu_tile_order import exact_operands

# M, N, K: (rows of the persistent kernel, rows of its tiles) by the rule
PLANS = [((4800, 2304, 768), (4800, 192)), ((4032, 3072, 192), (4032, 192)), ((4033, 2304, 768), (4033, 192)),
         ((9600, 2304, 768), (9600, 192)), ((383, 25600, 192), (383, 192)), ((24592, 256, 128), (24592, 192)),
         ((16337, 320, 128), (16337, 192)), ((6700, 3072, 768), None), ((8200, 3072, 1024), None),
         ((7200, 2304, 768), None), ((4800, 3072, 768), (4800, 256)), ((153600, 2304, 768), None),
         ((2900, 4096, 1024), (2900, 192)), ((1700, 4800, 1600), (1700, 192)),
         ((2064, 3200, 256), (2064, 192))]


def plan(tiles, M, N, slices, kn=False):
    """persistent_rows of gemm.hip for 256 CUs, no residual, no dropout; kn: the weight in place, if it can be."""
    with open(os.path.join(ragged.ROOT, "gpt_triton_amd", "csrc", "gemm.hip")) as f:
        source = f.read()
    assert "if (tm == 192 && (res || drop || tiles > 6 * (int64_t)cus || (kn && !stream_reads_kn(M, N)))) break;" in source
    e192 = re.sub(r"(?<=\d)f\b", "", re.search(r"if \(bm == 192\) return (.*?);", source).group(1))
    cols = -(-N // 256)
    tiles256 = -(-M // 256) * cols
    least, head, bm = (math.inf if tiles256 >= 512 else ragged.pick(tiles, M, N, slices)[0]), 0, 256
    for tm, expression in ((256, ragged.stream_terms()[1]), (192, e192)):
        if tm == 192 and (tiles256 > 6 * 256 or kn and (N % 256 != 0 or M > 32768)):
            break
        whole = -(-M // tm) * cols // 256 * 256 // cols * tm
        for rows in (M, min(whole, M)):
            if rows == 0:
                continue
            t = -(-rows // tm) * cols
            c = eval(expression, {"rounds": -(-t // 256), "fill": t / 256, "k": slices})
            if rows < M:
                c += 1.0 + ragged.pick(tiles, M - rows, N, slices)[0]
            if c < least:
                least, head, bm = c, rows, tm
    return head, bm


def test_where_the_rule_takes_them():
    tiles = ragged.cost_tables()
    for (M, N, Kd), want in PLANS:
        head, bm = plan(tiles, M, N, Kd // 64)
        print(M, N, Kd, head, bm)
        assert want is None or (head, bm) == want
    # rows left to the tile kernel behind tiles of 192
    assert plan(tiles, 6700, 3072, 12)[1] == 192 and 0 < plan(tiles, 6700, 3072, 12)[0] < 6700
    # a weight that the persistent kernel cannot read in place: the tile kernel does, as it did
    assert plan(tiles, 2064, 3200, 4) == (2064, 192) and plan(tiles, 2064, 3200, 4, kn=True) == (0, 256)
    # many rounds: tiles of 256 only
    assert plan(tiles, 153600, 2304, 12)[1] == 256
    # and every shape of the tile kernel is still reached by the sizes that the other tests take
    import test_gpu_gemm_tile

    reached = set()
    for M, N, Kd in ragged.BETWEEN + test_gpu_gemm_tile.SHAPES:
        slices = -(-Kd // 64)
        if N % 64 or M < 256 or plan(tiles, M, N, slices)[0] == 0:
            reached.add(ragged.pick(tiles, M, N, slices)[1])
    assert reached == set(range(13)), reached


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", [p[0] for p in PLANS if p[0][0] < 30000])
def test_every_row_once(K, gpu_device, M, N, Kd):
    print(f"192-row tiles {M} x {N} x {Kd}", flush=True)
    x, w, _ = exact_operands(M, N, Kd, gpu_device, M + N)
    want = x @ w
    assert float(want.abs().max()) <= 2048
    bias = torch.randint(-3, 4, (N,), device=gpu_device).float()
    assert torch.equal(K.fused_ffn(x.half(), K.pack_weight(w.half())).float(), want)
    got = K.fused_ffn(x.half(), w.half(), bias=bias.half()).float()  # in place where the columns allow it
    assert torch.equal(got, (want + bias).half().float())
    if M * N <= 20_000_000:
        assert torch.equal(K.fused_ffn(x, w, bias=bias), want + bias)


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,heads,h", [(16, 300, 12, 768), (5, 777, 16, 1024), (37, 110, 12, 768), (32, 300, 12, 768),
                                         (500, 9, 12, 768)])
def test_every_row_once_scattered(K, gpu_device, B, L, heads, h):
    assert plan(ragged.cost_tables(), B * L, 3 * h, h // 64)[1] == 192
    print(f"192-row tiles, scatter {B} x {L} x {h}", flush=True)
    x, w, _ = exact_operands(B * L, 3 * h, h, gpu_device, B + L)
    want = (x @ w).view(B, L, 3, heads, h // heads)
    bias = torch.zeros(3 * h, device=gpu_device)
    for dtype, weight in ((torch.float16, w.half()), (torch.float16, K.pack_weight(w.half())), (torch.float32, w)):
        got = K.matmul_and_split_qkv(x.to(dtype).view(B, L, h), weight, bias.to(dtype), heads)
        for i, t in enumerate(got):
            assert torch.equal(t.float(), want[:, :, i].transpose(1, 2))
