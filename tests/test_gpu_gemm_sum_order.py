"""The order of a row's sum where the persistent kernel takes tiles of 192 rows (csrc/gemm.hip): rows whose K the tile
kernel divides over two or four groups, which gives the more exact sums, keep them, and a weight and its packed image give
the same bits.  On the CPU the rule, over many sizes; on the GPU the bits, on random operands."""
import math
import os
import re

import pytest
import torch

import test_gpu_gemm_ragged as ragged
from test_gpu_gemm_in_place import weights


def split(tiles, M, N, slices):
    """Over how many sums the tile kernel divides K for M rows; none are one."""
    return tiles[ragged.pick(tiles, M, N, slices)[1]][2] if M > 0 else 1


def plan(tiles, M, N, slices, kn=False):
    """persistent_rows of gemm.hip for 256 CUs, no residual, no dropout, as (rows, rows of a tile); kn: the weight in place, if
    it can be."""
    with open(os.path.join(ragged.ROOT, "gpt_triton_amd", "csrc", "gemm.hip")) as f:
        source = f.read()
    assert ragged.two_rounds()
    assert "if (tm == 192 && (res || drop || tiles > 6 * (int64_t)cus || (kn && !stream_reads_kn(M, N)))) break;" in source
    assert "if (tm == 192 && !one_sum(*head)) break;" in source
    assert "if (c < least && (tm == 256 || stream_reads_kn(M, N) || one_sum(rows))) least = c, *head = rows, *bm = tm;" in source
    e192 = re.sub(r"(?<=\d)f\b", "", re.search(r"if \(bm == 192\) return (.*?);", source).group(1))
    cols = -(-N // 256)
    tiles256 = -(-M // 256) * cols
    least, head, bm = (math.inf if tiles256 >= 512 else ragged.pick(tiles, M, N, slices)[0]), 0, 256
    for tm, expression in ((256, ragged.stream_terms()[1]), (192, e192)):
        if tm == 192 and (tiles256 > 6 * 256 or kn and (N % 256 != 0 or M > 32768)):
            break
        if tm == 192 and split(tiles, M - head, N, slices) > 1:
            break
        whole = -(-M // tm) * cols // 256 * 256 // cols * tm
        for rows in (M, min(whole, M)):
            if rows == 0:
                continue
            t = -(-rows // tm) * cols
            c = eval(expression, {"rounds": -(-t // 256), "fill": t / 256, "k": slices})
            if rows < M:
                c += 1.0 + ragged.pick(tiles, M - rows, N, slices)[0]
            in_place = N % 256 == 0 and M <= 32768
            if c < least and (tm == 256 or in_place or split(tiles, M - rows, N, slices) == 1):
                least, head, bm = c, rows, tm
    return head, bm


def first_plan(tiles, M, N, slices):
    """Rows of the persistent kernel with tiles of 256 rows only."""
    return ragged.persistent_rows(tiles, M, N, slices, False)


SIZES = [(M, N, Kd) for N, Kd in ((2304, 768), (3072, 768), (768, 3072), (3072, 1024), (1024, 4096), (1280, 5120), (4800, 1600),
                                  (1088, 4352), (1344, 3072), (2880, 768)) for M in range(256, 26000, 177)]


def test_no_row_loses_its_split():
    tiles, taken, left = ragged.cost_tables(), 0, 0
    for M, N, Kd in SIZES:
        head, bm = plan(tiles, M, N, Kd // 64)
        if bm != 192:
            continue
        taken += 1
        assert split(tiles, M - first_plan(tiles, M, N, Kd // 64), N, Kd // 64) == 1, (M, N, Kd)
    print(f"{taken} of {len(SIZES)} sizes take tiles of 192 rows")
    assert taken > len(SIZES) // 20


def sums(tiles, M, N, slices, kn):
    """(first row, number of sums) of the rows that are formed alike; None where a weight is packed instead."""
    head, _ = plan(tiles, M, N, slices, kn)
    if kn and head and (N % 256 != 0 or M > 32768):
        return None
    groups = split(tiles, M - head, N, slices)
    return [(0, 1)] if groups == 1 else [(0, 1), (head, groups)] if head else [(0, groups)]


def test_a_weight_and_its_image_sum_alike():
    tiles, both = ragged.cost_tables(), 0
    for N, Kd in ((1088, 4352), (1152, 4608), (1344, 5376), (1728, 6912), (2624, 768), (2880, 768), (3008, 768), (2304, 768), (4800, 1600)):
        for M in list(range(256, 36000, 97)) + list(range(7000, 9000, 8)):
            plain = sums(tiles, M, N, Kd // 64, True)
            if plain is not None:
                both += 1
                assert plain == sums(tiles, M, N, Kd // 64, False), (M, N, Kd)
    assert both > 1000


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


# M, N, K; the first of the rows that the tile kernel takes, with K divided
DIVIDED = [(7200, 1088, 4352, 0), (5924, 1344, 3072, 0), (11384, 3072, 768, 10752)]


def test_the_shapes_below():
    tiles = ragged.cost_tables()
    for M, N, Kd, start in DIVIDED:
        assert plan(tiles, M, N, Kd // 64) == (start, 256) and split(tiles, M - start, N, Kd // 64) > 1


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd,start", DIVIDED)
def test_divided_sums_stay_divided(K, gpu_device, M, N, Kd, start):
    print(f"divided sums {M} x {N} x {Kd}", flush=True)
    draw, w, b = weights(gpu_device, Kd, N, M)
    x = draw(M, Kd)
    image = K.pack_weight(w)
    whole = K.fused_ffn(x, image)
    assert torch.isfinite(whole).all() and torch.equal(whole[start:], K.fused_ffn(x[start:].contiguous(), image))
    if start == 0:  # the weight in place is the tile kernel's for these columns
        assert torch.equal(whole, K.fused_ffn(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", [(7176, 1088, 4352), (7232, 1088, 4352), (8992, 2624, 768), (8200, 2880, 768), (8212, 2880, 768),
                                    (8200, 3072, 1024), (2064, 3200, 256)])
def test_a_weight_and_its_image(K, gpu_device, M, N, Kd):
    print(f"a weight and its image {M} x {N} x {Kd}", flush=True)
    draw, w, b = weights(gpu_device, Kd, N, M)
    x = draw(M, Kd)
    image = K.pack_weight(w)
    for gelu in (False, True):
        plain = K.fused_ffn(x, w, bias=b, add_gelu=gelu)
        assert torch.isfinite(plain).all() and torch.equal(plain, K.fused_ffn(x, image, bias=b, add_gelu=gelu))
    if N % 192 == 0:
        for got, want in zip(K.matmul_and_split_qkv(x.view(1, M, Kd), w, b, N // 192),
                             K.matmul_and_split_qkv(x.view(1, M, Kd), image, b, N // 192)):
            assert torch.equal(got, want)
