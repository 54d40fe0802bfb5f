"""Which attention kernel serves head size 64 in fp16 depends on length and (batch, head) pairs.  The mask is
causal, so the first rows of a longer sequence are the attention of the shorter one: the same tiles in the
same order, whichever kernel, so equal bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


@pytest.mark.parametrize("merged", [False, True])
@pytest.mark.parametrize("B,heads", [(1, 1), (3, 21), (5, 17), (2, 43), (4, 128), (27, 19)])  # 1, 63, 85, 86, 512, 513 pairs
def test_first_rows(K, gpu_device, B, heads, merged):
    g = torch.Generator(device=gpu_device).manual_seed(B)
    q, k, v = (torch.randn(B, heads, 400, 64, generator=g, device=gpu_device).half() * 2 for _ in range(3))
    whole = K.flash_attention_v1(q, k, v, merged_heads_layout=merged)  # the ring
    for L in (1, 31, 32, 33, 63, 64, 65, 128, 288, 289, 300, 312, 313, 320, 321):
        print(f"attention of the first rows: pairs={B * heads} L={L} merged={merged}", flush=True)
        part = K.flash_attention_v1(*(t[:, :, :L].contiguous() for t in (q, k, v)), merged_heads_layout=merged)
        assert torch.equal(part, whole[:, :, :L]), L
