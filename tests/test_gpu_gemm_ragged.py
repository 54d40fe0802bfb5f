"""GEMM rows that are no multiple of a tile: the persistent 256 x 256 kernels with the last row tile moved up
(row M - 256 on, its shared rows formed twice), and the tile shapes between those of
tests/test_gpu_gemm_tile.py, each at the edges of its rows and columns.  Reference and tolerance: as there.
test_shapes_reach_the_kernels (on the CPU) holds the lists to the cost models."""
import math
import os
import re

import pytest
import torch

from test_gpu_gemm_tile import check, operands, reference

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


# (M, N, K) that the persistent kernels take whole
RAGGED = [(257, 25600, 192), (383, 25600, 192), (511, 25600, 192), (1477, 6400, 192), (2049, 4096, 192),
          (3073, 3072, 256), (4800, 2304, 192), (4800, 3072, 768)]
# (M, N, K) for the tiles between: 16x16, 48x32, 96x64, 192x64, 256x128, and for 64x32, 64x128 beside them
BETWEEN = [(1, 40, 768), (15, 768, 768), (16, 2304, 832), (17, 776, 1024), (31, 40, 1088),
           (65, 3080, 768), (96, 3080, 832), (97, 2304, 768), (257, 1032, 768), (400, 776, 768),
           (400, 3080, 256), (500, 2304, 448), (577, 2311, 320),
           (700, 3080, 256), (1000, 2312, 448), (2500, 1032, 320),
           (2500, 3080, 256), (2561, 3080, 192), (190, 2304, 768), (600, 3080, 320)]


# (B, L, heads, h) of qkv products that the persistent kernel takes whole
SCATTERED = [(3, 1295, 12, 768), (16, 300, 12, 192), (37, 105, 16, 256), (1477, 1, 33, 192)]


def cost_tables():
    source = open(os.path.join(ROOT, "gpt_triton_amd", "csrc", "gemm_tile.hip")).read()
    tables = []
    for name in ("kTiles", "kTilesBetween"):
        rows = re.search(r"TileCost %s\[\] = \{(.*?)\};" % name, source, re.S).group(1)
        tables += [[float(v.rstrip("f")) for v in row.split(",")] for row in re.findall(r"\{([^{}]*)\}", rows)]
    return tables


def stream_terms():
    """The terms of stream_cost in gemm.hip, as (coefficient, factors) with and without a residual."""
    source = open(os.path.join(ROOT, "gpt_triton_amd", "csrc", "gemm.hip")).read()
    with_res, without = re.search(r"return res \? (rounds.*?)\n\s*: (.*?);", source, re.S).groups()
    # python reads the two expressions once the float suffixes are gone
    return [re.sub(r"(?<=\d)f\b", "", e) for e in (with_res, without)]


def two_rounds():
    source = open(os.path.join(ROOT, "gpt_triton_amd", "csrc", "gemm.hip")).read()
    return "float least = tiles >= 2 * (int64_t)cus ? INFINITY : gemm_tile_cost(M, N, Kp, cus);" in source and (
        "if (rows < M) c += 1.0f + gemm_tile_cost(M - rows, N, Kp, cus);" in source)


def pick(tiles, M, N, slices):
    def cost(tile):
        bm, bn, _, launch, fixed, per_slice = tile
        return launch + -(-(-(-M // int(bm)) * -(-N // int(bn))) // 256) * (fixed + slices * per_slice)

    costs = [cost(t) for t in tiles]
    return min(costs), costs.index(min(costs))


def persistent_rows(tiles, M, N, slices, res, drop=False):
    """persistent_rows of gemm.hip for 256 CUs, no overlap; with dropout all rows or none."""
    assert two_rounds(), "the rule below is not the one of gemm.hip any more"
    cols, row_tiles = -(-N // 256), -(-M // 256)
    whole = M if drop else row_tiles * cols // 256 * 256 // cols * 256
    expression = stream_terms()[0 if res else 1]

    def stream(t):
        return eval(expression, {"rounds": -(-t // 256), "fill": t / 256, "k": slices})

    least, head = (math.inf if row_tiles * cols >= 512 else pick(tiles, M, N, slices)[0]), 0
    for rows in (M, min(whole, M)):
        if rows == 0:
            continue
        c = stream(-(-rows // 256) * cols)
        if rows < M:
            c += 1.0 + pick(tiles, M - rows, N, slices)[0]
        if c < least:
            least, head = c, rows
    return head


def test_shapes_reach_the_kernels():
    import test_gpu_gemm_dropout
    import test_gpu_gemm_tile

    tiles = cost_tables()
    assert len(tiles) == 13
    for M, N, Kd in RAGGED:
        assert M % 256 != 0
        for res in (False, True):
            assert persistent_rows(tiles, M, N, Kd // 64, res) == M
    for B, L, heads, h in SCATTERED:
        assert B * L % 256 != 0 and persistent_rows(tiles, B * L, 3 * 64 * heads, h // 64, False) == B * L
    for M, h, inner in test_gpu_gemm_dropout.SHAPES:
        first = persistent_rows(tiles, M, inner, h // 64, False, drop=True)
        second = h >= 256 and inner >= 192 and persistent_rows(tiles, M, h, inner // 64, True, drop=True)
        assert M in (first, second)
        if (M, h, inner) in test_gpu_gemm_dropout.WITH_RESIDUAL:
            assert second == M
        else:
            assert first == M
    reached = set()
    for M, N, Kd in BETWEEN + test_gpu_gemm_tile.SHAPES:
        slices = -(-Kd // 64)
        if N % 64 or M < 256 or persistent_rows(tiles, M, N, slices, False) == 0:
            reached.add(pick(tiles, M, N, slices)[1])
    assert reached == set(range(13)), reached
    # a split in four is never picked below four k-slices
    for M in (1, 8, 16, 24, 48, 64, 128, 200, 513, 1477, 4800):
        for N in (16, 40, 768, 2304, 6400):
            for slices in (1, 2, 3):
                assert tiles[pick(tiles, M, N, slices)[1]][2] < 4


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", RAGGED)
def test_ragged_rows_of_the_persistent_kernels(K, gpu_device, M, N, Kd):
    for dtype in (torch.float16, torch.float32):
        x, w, b, res = operands(M, N, Kd, dtype, gpu_device, seed=M + N + Kd)
        print(f"ragged persistent GEMM {dtype} M={M} N={N} K={Kd}", flush=True)
        for gelu, with_res in ((False, True), (True, False)):
            r = res if with_res else None
            got = K.fused_ffn(x, w, bias=b, residual=r, add_gelu=gelu)
            want, sums = reference(x, w, b, r, gelu)
            check(got, want, sums, Kd, f"gelu={gelu} residual={with_res}")
            assert torch.equal(got, K.fused_ffn(x, w, bias=b, residual=r, add_gelu=gelu))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,heads,h", SCATTERED)
def test_ragged_rows_scattered(K, gpu_device, dtype, B, L, heads, h):
    n = heads * 64
    x, w, b, _ = operands(B * L, 3 * n, h, dtype, gpu_device, seed=B + L)
    print(f"ragged persistent QKV {dtype} B={B} L={L} heads={heads} h={h}", flush=True)
    got = K.matmul_and_split_qkv(x.view(B, L, h), w, b, heads)
    want, sums = reference(x, w, b, None, False)
    for i, t in enumerate(got):
        col = slice(i * n, (i + 1) * n)
        check(t.transpose(1, 2).reshape(B * L, n), want[:, col], sums[:, col], h, "qkv"[i])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", [(2049, 4096, 192), (4800, 2304, 192)])
def test_output_over_its_residual(K, gpu_device, M, N, Kd):
    """The output in the place of the residual: no row is added to twice."""
    from gpt_triton_amd import _lib

    x, w, b, res = operands(M, N, Kd, torch.float16, gpu_device, seed=M)
    print(f"residual in place M={M} N={N} K={Kd}", flush=True)
    want, sums = reference(x, w, b, res, False)
    inout = res.clone()
    K._linear(x, K.pack_weight(w), b, inout, inout, False, 0.0, _lib.GPTMI_W_PACKED, "linear")
    check(inout, want, sums, Kd, "in place")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,Kd", BETWEEN)
def test_tiles_between(K, gpu_device, dtype, M, N, Kd):
    x, w, b, res = operands(M, N, Kd, dtype, gpu_device, seed=M + N + Kd)
    print(f"tile GEMM {dtype} M={M} N={N} K={Kd}", flush=True)
    for gelu, with_res in ((False, True), (True, False)):
        r = res if with_res else None
        got = K.fused_ffn(x, w, bias=b, residual=r, add_gelu=gelu)
        want, sums = reference(x, w, b, r, gelu)
        check(got, want, sums, Kd, f"gelu={gelu} residual={with_res}")


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", [(17, 776, 1024), (97, 2304, 768), (500, 2304, 448), (1000, 2312, 448),
                                    (2561, 3080, 192)])
def test_tiles_between_with_dropout(K, gpu_device, M, N, Kd):
    """The same products with dropout are the ones without, kept or zeroed and divided by 1 - p."""
    x, w, b, _ = operands(M, N, Kd, torch.float32, gpu_device, seed=M)
    print(f"tile GEMM with dropout M={M} N={N} K={Kd}", flush=True)
    got = K.fused_ffn(x, w, bias=b, dropout_prob=0.25)
    want, sums = reference(x, w, b, None, False)
    kept = got != 0
    assert 0.7 < kept.float().mean().item() < 0.8
    check(torch.where(kept, got, 0.0), torch.where(kept, want / 0.75, 0.0), sums / 0.75, Kd, "dropout")
