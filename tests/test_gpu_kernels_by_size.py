"""Kernels that are picked by size, each at sizes that it really gets (256 CUs): the persistent product with tiles of 256
rows and a last one that is moved up, with and without the scatter to heads, the streaming attention kernel at every
length and on the reference's own vectors, and the ring kernel with 32 queries a wavefront.  The rules are read from the sources on the CPU (`plan` of
test_gpu_gemm_sum_order.py, `attention_kernel` below), so that a size which moves to another kernel fails there.
References and tolerances: those of test_gpu_gemm_tile.py and test_gpu_attention_stream.py."""
import os
import re

import numpy as np
import pytest
import torch

import test_gpu_attention_stream as stream
import test_gpu_gemm_ragged as ragged
from oracle import gpt2_oracle as O
from test_gpu_gemm_sum_order import plan
from test_gpu_gemm_tile import check, operands, reference


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


# M, N, K: all rows in tiles of 256, the last of them moved up by 252, 57, 1, 7 and 69 rows
RAGGED = [(5380, 2304, 768), (2503, 4800, 1600), (511, 25600, 192), (4089, 3072, 768), (1979, 6400, 192)]
# B, L, heads, h of q, k, v products, the same: sequences longer than a wavefront's 128 rows, shorter, and of one row
SCATTERED = [(2, 2690, 12, 768), (5, 1103, 12, 768), (7, 283, 33, 192), (51, 107, 12, 192), (1979, 1, 33, 192), (220, 9, 33, 192)]

# lengths on both sides of each 32-row chunk and 64-key tile, up to the streaming kernel's longest
LENGTHS = [1, 2, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 191, 192, 193, 255, 256, 257, 299, 300, 319, 320]


def pairs_for(L):
    """B, N of more pairs than any other kernel takes, and no multiple of the workgroups."""
    return (67, 23) if L <= 64 else (57, 9) if L <= 192 else (23, 9)


# pairs, rows of the ring kernel: two tiles, then both sides of a 64-key tile and of a 128-query block
RING = [(512, 65), (331, 96), (300, 127), (512, 128), (103, 321), (87, 383), (87, 384), (75, 385), (81, 449), (60, 700), (39, 1025)]

GOLDEN = [("a", 3), ("c", 1)]  # 150 and 300 rows


def attention_kernel(pairs, L, acc=False):
    """launch_d64 of flash_attn.hip for 256 CUs and a positive scale."""
    with open(os.path.join(ragged.ROOT, "gpt_triton_amd", "csrc", "flash_attn.hip")) as f:
        source = f.read()
    few, acc_few, long_rows, long_few, short_few = map(int, re.search(
        r"2 \* blocks <= \(L <= BKEY \? (\d+) : ACC \? (\d+) : L > (\d+) \? (\d+) : (\d+)\) \* \(int64_t\)cus\)", source).groups())
    ring_rows, tiles, ring_pairs = map(int, re.search(
        r"const bool ring = L > (\d+) \|\| \(L <= (\d+) \* BKEY && BN <= (\d+)\);", source).groups())
    assert "const int64_t blocks = BN * ((L + kRing16Rows - 1) / kRing16Rows);" in source
    assert "constexpr int kRing16Rows = 64;" in source
    if 2 * pairs * -(-L // 64) <= (few if L <= 64 else acc_few if acc else long_few if L > long_rows else short_few) * 256:
        return "16 queries"
    return "ring" if L > ring_rows or (L <= tiles * 64 and pairs <= ring_pairs) else "streaming"


def test_sizes_reach_the_kernels():
    tiles = ragged.cost_tables()
    for M, N, Kd in RAGGED:
        assert M % 256 and plan(tiles, M, N, Kd // 64) == (M, 256), (M, N, Kd)
    for B, L, heads, h in SCATTERED:
        assert B * L % 256 and plan(tiles, B * L, 192 * heads, h // 64) == (B * L, 256), (B, L, heads, h)
    for L in LENGTHS:
        B, N = pairs_for(L)
        assert attention_kernel(B * N, L) == "streaming", L
    for L in (150, 300):
        assert attention_kernel(18 * 11, L) == "streaming"
    for pairs, L in RING:
        assert attention_kernel(pairs, L) == "ring", (pairs, L)
    assert attention_kernel(99, 150) == "16 queries" and attention_kernel(512, 100) == "ring"


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd", RAGGED)
def test_ragged_rows_in_tiles_of_256(K, gpu_device, M, N, Kd):
    for dtype in (torch.float16, torch.float32):
        x, w, b, _ = operands(M, N, Kd, dtype, gpu_device, seed=M + N + Kd)
        print(f"256-row tiles, ragged: {dtype} {M} x {N} x {Kd}", flush=True)
        image = K.pack_weight(w)
        for gelu in (False, True):
            want, sums = reference(x, w, b, None, gelu)
            for weight in (w, image):
                check(K.fused_ffn(x, weight, bias=b, add_gelu=gelu), want, sums, Kd, f"gelu={gelu}")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,heads,h", SCATTERED)
def test_ragged_rows_in_tiles_of_256_scattered(K, gpu_device, dtype, B, L, heads, h):
    n = heads * 64
    x, w, b, _ = operands(B * L, 3 * n, h, dtype, gpu_device, seed=B + L)
    print(f"256-row tiles, ragged, scattered: {dtype} B={B} L={L} heads={heads} h={h}", flush=True)
    want, sums = reference(x, w, b, None, False)
    for weight in (w, K.pack_weight(w)):
        for i, t in enumerate(K.matmul_and_split_qkv(x.view(B, L, h), weight, b, heads)):
            col = slice(i * n, (i + 1) * n)
            check(t.transpose(1, 2).reshape(B * L, n), want[:, col], sums[:, col], h, "qkv"[i])


@pytest.mark.gpu
@pytest.mark.parametrize("L", LENGTHS)
def test_streaming_attention_lengths(K, gpu_device, L):
    B, N = pairs_for(L)
    q, k, v = stream.gaussian_qkv(B, N, L, seed=2000 + L)
    print(f"streaming attention: {B} x {N} pairs L={L}", flush=True)
    z, zm = stream.both_layouts(K, q, k, v, gpu_device)
    stream.check_f16(z, O.flash_attention_v1(q, k, v), f"L={L}")
    assert np.array_equal(z, zm)
    assert np.array_equal(z[:, :, 0], v[:, :, 0])  # query 0 sees key 0 only


@pytest.mark.gpu
@pytest.mark.parametrize("pairs,L", RING)
def test_ring_attention(K, gpu_device, pairs, L):
    q, k, v = stream.gaussian_qkv(pairs, 1, L, seed=3000 + L)
    print(f"ring attention: {pairs} pairs L={L}", flush=True)
    z, zm = stream.both_layouts(K, q, k, v, gpu_device)
    stream.check_f16(z, O.flash_attention_v1(q, k, v), f"L={L}")
    assert np.array_equal(z, zm)
    assert np.array_equal(z[:, :, 0], v[:, :, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("case,heads", GOLDEN)
def test_streaming_attention_reference_vectors(K, gpu_device, case, heads):
    """The reference's own outputs (tests/golden/flash_attention_v1.npz), its pairs first, in the middle and last of 198."""
    golden = np.load(os.path.join(os.path.dirname(__file__), "golden", "flash_attention_v1.npz"))
    gq, gk, gv, gout = (golden[f"{case}_{t}"] for t in ("q", "k", "v", "out"))
    L = gq.shape[2]
    q, k, v = stream.gaussian_qkv(18, 11, L, seed=78)
    spots = [(0, 0), (9, 5), (17, 10)]
    for i, (b, n) in enumerate(spots):
        q[b, n], k[b, n], v[b, n] = gq[0, i % heads], gk[0, i % heads], gv[0, i % heads]
    print(f"streaming attention: reference's case {case} among 198 pairs, L={L}", flush=True)
    z, zm = stream.both_layouts(K, q, k, v, gpu_device)
    for i, (b, n) in enumerate(spots):
        stream.check_f16(z[b, n], gout[0, i % heads], f"case {case} at ({b},{n}) [B,N,L,d]")
        stream.check_f16(zm[b, n], gout[0, i % heads], f"case {case} at ({b},{n}) [B,L,N,d]")
