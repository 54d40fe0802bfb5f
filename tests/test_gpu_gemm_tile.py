"""The GEMM with one workgroup per output tile (gemm_tile.hip) at the sizes where it can go wrong:
fewer k-slices than groups that split K (two groups; a four-way split is never picked below four slices),
k-steps fewer than, equal to and one more than the stages, a last k-step that not every group has a slice
of, one row and one column past a tile, columns that do not fill a 16-byte chunk, and a shape each that
the cost model sends to every tile of the menu (test_host.py holds the list to that).
Reference: an fp32 product of the fp16-rounded operands (the operands of the kernel), epilogue in fp32.

Tolerance: the fp32 sums of K products differ by at most K * 2^-24 of the sum of their absolute values,
whatever the order, and the result is rounded once: half an ulp, 2^-11 of the value in fp16, 2^-24
in fp32; GELU and the residual add a few fp32 roundings, which 2^-20 of the largest value covers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels

    return kernels


def operands(M, N, Kd, dtype, device, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    rn = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(dtype).to(device)
    return rn(M, Kd), rn(Kd, N, std=Kd**-0.5), rn(N), rn(M, N)


def reference(x, w, b, res, gelu):
    xh, wh = x.half().float(), w.half().float()
    z = xh @ wh
    if b is not None:
        z = z + b.float()
    if gelu:
        z = torch.nn.functional.gelu(z, approximate="tanh")
    if res is not None:
        z = z + res.float()
    return z, xh.abs() @ wh.abs()


def check(got, want, sums, Kd, what):
    assert bool(torch.isfinite(got).all()), f"{what}: non-finite output"
    half_ulp = 2.0**-11 if got.dtype == torch.float16 else 2.0**-24
    bound = half_ulp * want.abs() + Kd * 2.0**-24 * sums + 2.0**-20 * want.abs().max()
    over = (got.float() - want).abs() - bound
    assert float(over.max()) <= 0, f"{what}: {float(over.max()):.3e} beyond the bound"


# (M, N, K): tiles 32x16 and 32x32 split K four ways with four stages of 256, 64x32 with three,
# 64x64 two ways with four of 128, 64x128 with three, the others walk 64 at a time
SHAPES = [
    (1, 16, 64), (24, 768, 64), (31, 48, 192), (32, 32, 256), (33, 40, 320),   # 1, 1, 3; 4, 5 slices
    (24, 768, 1024), (24, 768, 1088), (24, 768, 1344),   # stages full, one slice and one step more
    (128, 768, 3072), (129, 776, 448),
    (200, 3072, 128), (300, 2304, 832), (65, 6400, 576),
    (700, 768, 768), (513, 1032, 320), (1024, 768, 448),
    (1477, 768, 576), (1500, 1544, 320),
    (1024, 3072, 768), (3073, 768, 832), (2049, 2304, 256), (2500, 3080, 192),
    (37, 50, 128), (130, 33, 70), (1100, 1001, 200),     # columns and k that fill no chunk
    (127, 2311, 448), (128, 2304, 768), (127, 2312, 832),      # 64x32: 2, 3 and 4 k-steps of three stages
    (4700, 3001, 200), (4800, 3072, 768), (4801, 3080, 832),   # 128x256
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,Kd", SHAPES)
def test_fused_ffn_tiles(K, gpu_device, dtype, M, N, Kd):
    x, w, b, res = operands(M, N, Kd, dtype, gpu_device, seed=M + N + Kd)
    print(f"tile GEMM {dtype} M={M} N={N} K={Kd}", flush=True)
    for gelu, with_res in ((False, True), (True, False)):
        r = res if with_res else None
        got = K.fused_ffn(x, w, bias=b, residual=r, add_gelu=gelu)
        want, sums = reference(x, w, b, r, gelu)
        check(got, want, sums, Kd, f"gelu={gelu} residual={with_res}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,heads,d,h", [(3, 1, 2, 8, 64), (5, 7, 3, 24, 192), (2, 333, 12, 64, 768),
                                           (11, 150, 5, 16, 320), (1, 2100, 4, 64, 256)])
def test_qkv_scatter_tiles(K, gpu_device, dtype, B, L, heads, d, h):
    n = heads * d
    x, w, b, _ = operands(B * L, 3 * n, h, dtype, gpu_device, seed=B + L + d)
    print(f"tile QKV {dtype} B={B} L={L} heads={heads} d={d}", flush=True)
    got = K.matmul_and_split_qkv(x.view(B, L, h), w, b, heads)
    want, sums = reference(x, w, b, None, False)
    for i, t in enumerate(got):
        col = slice(i * n, (i + 1) * n)
        flat = t.transpose(1, 2).reshape(B * L, n)
        check(flat, want[:, col], sums[:, col], h, "qkv"[i])


def test_rows_past_32_bit_offsets(K, gpu_device):
    """K = 2^22: 32 rows of an operand span more than a lane's 32-bit byte offset reaches.  Operands of
    +-1 and +-2^-10 make every sum exact."""
    M, N, Kd = 33, 24, 1 << 22
    g = torch.Generator(device="cpu").manual_seed(4)
    sign = lambda *s: (2 * torch.randint(0, 2, s, generator=g, dtype=torch.int8) - 1).to(gpu_device).half()
    x, w = sign(M, Kd), sign(N, Kd).mul_(2.0**-10)
    print("tile GEMM, K = 2^22", flush=True)
    got = K.fused_ffn(x, w.t().contiguous())
    want = x.double() @ w.double().t()
    assert torch.equal(got, want.half())
