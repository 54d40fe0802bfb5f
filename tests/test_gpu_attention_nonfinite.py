"""Rows of k and v that are not finite (an overflow, padding that was never written) behind a query: attention works through
32 queries and 32 keys at a time, and a block of keys that all of a block's queries come before does not enter, whichever
kernel the number of pairs picks.  Those queries have the bits that they have with zeros in that row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from gpt_triton_amd import kernels
    return kernels


# few pairs (16 queries a wavefront), up to 512 of two tiles, longer ones (ring) and more (streaming)
SHAPES = [(2, 3, 64), (2, 3, 72), (2, 12, 100), (8, 12, 128), (30, 12, 100), (1, 12, 200), (8, 12, 300), (16, 12, 300),
          (2, 5, 448), (16, 12, 400), (1, 3, 777)]


@pytest.mark.parametrize("B,N,L", SHAPES)
def test_hidden_keys_do_not_enter(K, gpu_device, B, N, L):
    print(f"rows that are not finite: {B} x {N} x {L}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(L)
    q, k, v = (torch.randn((B, N, L, 64), generator=g, device=gpu_device).half() for _ in range(3))
    for key in sorted({33, 40, 63, min(L, 100) - 1, L // 64 * 64 - 1, L - 1}):
        first = key // 32 * 32  # queries in front of the key's block
        for value in (float("inf"), float("nan")):
            kk, vv = k.clone(), v.clone()
            kk[:, :, key], vv[:, :, key] = 0, 0
            want = K.flash_attention_v1(q, kk, vv)[:, :, :first]
            kk[:, :, key], vv[:, :, key] = value, value
            got = K.flash_attention_v1(q, kk, vv)[:, :, :first]
            assert torch.isfinite(got).all() and torch.equal(got, want), (key, value)
