"""Which eval-mode forwards go to the library in one call (gpt._stack), on the CPU: nothing is launched."""
import pytest
import torch

from gpt_triton_amd import gpt
from gpt_triton_amd.kernels import PackedWeight


def pack(weight):
    return PackedWeight(torch.empty(16), weight.shape, weight.dtype)


def build(layers=3):
    model = gpt.FusedGPT(gpt.GPTConfig(n_layer=layers, n_head=2, n_embd=128, vocab_size=8, block_size=16)).eval()
    for block in model.blocks:
        for module, names in ((block[0], ("c_attn_weight", "c_proj_weight")),
                              (block[1], ("ffn1_weight", "ffn2_weight"))):
            for name in names:
                module._packed.get(name, getattr(module, name), pack)
    return model, torch.zeros(1, 4, 128)


def taken(model, x):
    return gpt._stack(list(model.blocks), x) is not None


def test_untouched_blocks_are_taken():
    model, x = build()
    pointers, heads, inner, in_gemm, _ = gpt._stack(list(model.blocks), x)
    assert len(pointers) == 36 and (heads, inner, in_gemm) == (2, 512, False)
    mlp = model.blocks[2][1]
    assert pointers[-6:] == [mlp.layer_norm_weight.data_ptr(), mlp.layer_norm_bias.data_ptr(),
                             mlp._packed.held("ffn1_weight", mlp.ffn1_weight).data_ptr(), mlp.ffn1_bias.data_ptr(),
                             mlp._packed.held("ffn2_weight", mlp.ffn2_weight).data_ptr(), mlp.ffn2_bias.data_ptr()]


@pytest.mark.parametrize("name", ["__call__", "_call_impl"])
@pytest.mark.parametrize("kind", ["_Block", "FusedAttention", "FusedMLP"])
def test_a_call_of_the_class_runs(kind, name, monkeypatch):
    model, x = build()
    monkeypatch.setattr(getattr(gpt, kind), name, lambda self, *a, **k: None, raising=False)
    assert not taken(model, x)
    monkeypatch.undo()
    assert taken(model, x)


@pytest.mark.parametrize("name", ["forward", "_weights", "_call_impl", "_wrapped_call_impl"])
@pytest.mark.parametrize("which", [0, 1])
def test_what_an_instance_has_in_the_place_of_a_method_runs(name, which):
    model, x = build()
    module = model.blocks[1][which]
    setattr(module, name, lambda *a, **k: None)
    assert not taken(model, x)
    delattr(module, name)
    assert taken(model, x)


@pytest.mark.parametrize("name", ["attention_block", "mlp_block", "layer_norm_ffn", "_weights", "_tensors"])
def test_a_replaced_function_runs(name, monkeypatch):
    model, x = build()
    monkeypatch.setattr(gpt, name, lambda *a, **k: None)
    assert not taken(model, x)


def refusals():
    """(what, changed arguments, changed pointers of the last layer, status)"""
    yield "inner", {"inner": 100}, {}, -1
    yield "inner", {"inner": 1 << 27}, {}, -1
    for i in (0, 1, 2, 4, 6, 7, 8, 10):
        yield f"pointer {i}", {}, {i: None}, -1
    for i in (2, 4, 8, 10):
        yield f"image {i}", {}, {i: 256 + 8}, -1
    yield "LayerNorm in the product in fp32", {"dtype": 0, "fuse": 1}, {}, -2
    yield "LayerNorm in the product, behind rows normalised already", {"dtype": 0, "fuse": 1, "normed": 256}, {}, -2
    yield "rows beyond the attention's", {"L": (1 << 24) + 1}, {}, -2
    yield "pairs beyond the grid", {"B": 1 << 31, "L": 1, "heads": 1}, {}, -2


@pytest.mark.parametrize("what,args,pointers,status", refusals())
@pytest.mark.parametrize("layers", [1, 3])
def test_blocks_refuse_before_any_launch(what, args, pointers, status, layers):
    import ctypes

    from gpt_triton_amd import _lib
    lib = _lib.load()
    a = {"normed": None, "B": 1, "L": 8, "heads": 2, "inner": 512, "fuse": 0, "dtype": 1, **args}
    table = [256] * 12 * layers
    for i, p in pointers.items():
        table[12 * (layers - 1) + i] = p
    need = lib.gptmi_blocks_workspace_bytes(a["B"], a["L"], a["heads"], 64, a["inner"], a["dtype"])
    fake = ctypes.c_void_p(256)
    rc = lib.gptmi_blocks(fake, a["normed"], (ctypes.c_void_p * len(table))(*table), layers, 1e-5, fake, a["B"],
                          a["L"], a["heads"], 64, a["inner"], a["fuse"], fake, need, a["dtype"], None)
    assert rc == status and lib.gptmi_last_error().startswith(b"blocks:")
