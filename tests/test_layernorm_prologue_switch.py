"""gpt.LN_PROLOGUE_MAX_ROWS = 0, and -1 in a block call, mean the LayerNorm in a launch of its own in both storage types,
though fp32 blocks of few rows take it into the product without being asked.  On the CPU what the modules pass on and that
the limits agree; on the GPU the launches, counted in a captured graph, and their bits."""
import ctypes
import os
import re

import pytest
import torch

from gpt_triton_amd import gpt, kernels

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_zero_rows_turn_it_off(monkeypatch):
    asked = []
    monkeypatch.setattr(gpt, "attention_block", lambda x, *a, **kw: asked.append(kw["layer_norm_in_gemm"]) or x)
    monkeypatch.setattr(gpt, "mlp_block", lambda x, *a, **kw: asked.append(kw["layer_norm_in_gemm"]) or x)
    monkeypatch.setattr(gpt, "_weights", lambda module, tensors, *names: [tensors[n].data for n in names])
    block = gpt.FusedAttention(128, 2).eval(), gpt.FusedMLP(128).eval()
    x = torch.zeros(1, 8, 128)
    for module in block:
        module(x)
    monkeypatch.setattr(gpt, "LN_PROLOGUE_MAX_ROWS", 0)
    for module in block:
        module(x)
    assert asked == [False, False, None, None]
    assert [kernels._in_gemm_code(v) for v in (False, True, None)] == [0, 1, -1]


def test_the_limits_agree():
    with open(os.path.join(ROOT, "gpt_triton_amd", "csrc", "capi.cpp")) as f:
        rule = re.search(r"h <= (\d+) && M <= \(h <= (\d+) \? (\d+) : (\d+)\) && gemm_layernorm_supported", f.read()).groups()
    assert [int(v) for v in rule] == [gpt.LN_PROLOGUE_FEW_WIDTH, gpt.LN_PROLOGUE_MAX_WIDTH, gpt.LN_PROLOGUE_MAX_ROWS,
                                      gpt.LN_PROLOGUE_FEW_ROWS]


def launches(call):
    """Nodes of the graph of a call that has run once on the capturing stream, and its output behind a replay."""
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=side):
        out = call()
    nodes, hip = ctypes.c_size_t(0), ctypes.CDLL("libamdhip64.so")
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    graph.instantiate()
    graph.replay()
    torch.cuda.synchronize()
    return nodes.value, out.clone()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("rows", [24, 128])
def test_a_launch_more_without_it(gpu_device, dtype, rows):
    h, g = 768, torch.Generator(device=gpu_device).manual_seed(rows)
    print(f"LayerNorm in the product, declined: {rows} x {h} {dtype}", flush=True)
    draw = lambda *shape: torch.randn(*shape, generator=g, device=gpu_device)
    x, ln = draw(1, rows, h).to(dtype), [draw(h).to(dtype) for _ in range(2)]
    pack = lambda k, n: kernels.pack_weight((draw(k, n) / k ** 0.5).to(dtype))
    mlp = (x, *ln, pack(h, 4 * h), draw(4 * h).to(dtype), pack(4 * h, h), draw(h).to(dtype))
    attention = (x, *ln, pack(h, 3 * h), draw(3 * h).to(dtype), pack(h, h), draw(h).to(dtype), 12)
    fused = True if dtype is torch.float16 else False
    with torch.no_grad():
        for block, args in ((kernels.mlp_block, mlp), (kernels.attention_block, attention)):
            two, want = launches(lambda: block(*args, layer_norm_in_gemm=None))
            one, got = launches(lambda: block(*args, layer_norm_in_gemm=fused))
            assert one == two - 1, (block.__name__, one, two)
            assert torch.equal(got, want)
