"""Layers in one call, whose attention launches have further workgroups that touch the weights behind them: the bits of
the layers called one by one, where such workgroups fill idle CUs and where they follow a full round, for each of the
attention kernels that take them.  What they touch does not show in the output: test_weights_ahead.py holds it to
the images."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# the front kernel, the ring (short, long; few and many workgroups), the streaming kernel (few pairs, one round, more)
@pytest.mark.parametrize("B,L,heads,dtype", [(2, 20, 4, "fp16"), (64, 24, 4, "fp16"), (3, 60, 4, "fp16"), (100, 50, 4, "fp16"),
                                             (2, 400, 4, "fp16"), (20, 500, 4, "fp16"), (150, 330, 4, "fp16"),
                                             (5, 200, 4, "fp16"), (60, 150, 4, "fp16"), (62, 128, 4, "fp16"),
                                             (90, 300, 4, "fp16"), (2, 100, 4, "fp32"), (80, 200, 4, "fp32"),
                                             # nothing to request; one round of pairs of layers too large for the cache
                                             (2, 40, 25, "fp16"), (15, 128, 16, "fp16")])
def test_layers_in_one_call(gpu_device, B, L, heads, dtype):
    from gpt_triton_amd import kernels as K
    print(f"prefetching layers: {B} x {L} rows, {heads} heads, {dtype}", flush=True)
    t = torch.float16 if dtype == "fp16" else torch.float32
    h, inner, n = 64 * heads, 256 * heads, 3
    g = torch.Generator(device=gpu_device).manual_seed(B)
    draw = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=gpu_device) * std).to(t)
    layers = []
    for _ in range(n):
        image = lambda k, m: K.pack_weight(draw(k, m, std=k**-0.5))
        layers.append((draw(h), draw(h), image(h, 3 * h), draw(3 * h), image(h, h), draw(h),
                       draw(h), draw(h), image(h, inner), draw(inner), image(inner, h), draw(h)))
    x = draw(B, L, h)
    want = x
    for p in layers:
        want = K.mlp_block(K.attention_block(want, *p[:6], heads), *p[6:])
    got = K.block_layers(x, [v.data_ptr() for p in layers for v in p], heads, inner)
    assert torch.isfinite(want).all() and torch.equal(got, want)
