"""Forwards below `gpt.BLOCK_MAX_ELEMENTS` and, the limit moved under them, beyond it: the blocks in calls of the library
and operator by operator give the same bits, at row counts that are and are not whole row tiles, of 256 and of 768."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,width", [(28, 300, 256), (9, 1024, 256), (131, 64, 256),  # 8400, 9216 and 8384 rows
                                       (64, 300, 768), (145, 300, 768)])  # 19200 and 43500, just below the limit
def test_same_bits(gpu_device, monkeypatch, B, L, width):
    from gpt_triton_amd import gpt
    print(f"blocks and operators: {B} x {L} tokens, {width} wide", flush=True)
    cfg = gpt.GPTConfig(vocab_size=512, block_size=1024, n_layer=2, n_head=width // 64, n_embd=width, dropout=0.0)
    model = gpt.FusedGPT(cfg).init_synthetic_(std=0.05).half().to(gpu_device).eval()
    g = torch.Generator().manual_seed(B)
    ids = torch.randint(0, 512, (B, L), generator=g).to(gpu_device)
    called = []
    whole = gpt.blocks_forward
    monkeypatch.setattr(gpt, "blocks_forward", lambda *a, **k: called.append(1) or whole(*a, **k))
    with torch.no_grad():
        model(ids)  # builds the weight images
        called.clear()
        blocks = model(ids)
        assert called
        monkeypatch.setattr(gpt, "BLOCK_MAX_ELEMENTS", B * L * width - 1)
        called.clear()
        operators = model(ids)
    assert not called
    assert torch.isfinite(blocks).all() and torch.equal(blocks, operators)
