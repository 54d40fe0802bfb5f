"""Which eval-mode forwards go to the library in one call (gpt._stack), on the CPU: nothing is launched."""
import pytest
import torch

from gpt_triton_amd import gpt
from gpt_triton_amd.kernels import PackedWeight


def pack(weight):
    return PackedWeight(torch.empty(16), weight.shape, weight.dtype)


def build(layers=3, rows=2048):
    model = gpt.FusedGPT(gpt.GPTConfig(n_layer=layers, n_head=2, n_embd=128, vocab_size=8, block_size=16)).eval()
    for block in model.blocks:
        for module, names in ((block[0], ("c_attn_weight", "c_proj_weight")),
                              (block[1], ("ffn1_weight", "ffn2_weight"))):
            for name in names:
                module._packed.get(name, getattr(module, name), pack)
    return model, torch.zeros(1, rows, 128)


@pytest.fixture
def through(monkeypatch):
    """(layers of each call of the library, layers left to the modules) of a forward of these blocks."""
    def run(model, x):
        calls = []

        def call(x, pointers, heads, inner, normed=None, layer_norm_in_gemm=False, out=None, workspace=None):
            assert workspace is scratch and (heads, inner, layer_norm_in_gemm) == (2, 512, False) and (normed is None) == bool(calls)
            calls.append(pointers)
            return x

        scratch = (None, 0)
        monkeypatch.setattr(gpt, "blocks_workspace", lambda x, heads, inner: scratch)
        monkeypatch.setattr(gpt, "block_layers", call)
        monkeypatch.setattr(gpt, "blocks_forward", call)
        blocks = list(model.blocks)
        stack = gpt._stack(blocks, x)
        rest = blocks if stack is None else gpt._through(stack, blocks, x, x)[1]
        assert rest == blocks[len(blocks) - len(rest):]
        assert sum(calls, []) == addresses(blocks[:len(blocks) - len(rest)])
        return [len(c) // 12 for c in calls], len(rest)
    return run


def addresses(blocks):
    found = []
    for attention, mlp in blocks:
        for module, names in ((attention, ("layer_norm_weight", "layer_norm_bias", "c_attn_weight", "c_attn_bias",
                                           "c_proj_weight", "c_proj_bias")),
                              (mlp, ("layer_norm_weight", "layer_norm_bias", "ffn1_weight", "ffn1_bias",
                                     "ffn2_weight", "ffn2_bias"))):
            for name in names:
                t = module._parameters[name]
                found.append((t if t.dim() == 1 else module._packed.held(name, t)).data_ptr())
    return found


@pytest.mark.parametrize("layers,few,many", [(1, [1], [1]), (2, [2], [1, 1]), (4, [2, 2], [1, 3]),
                                             (12, [2, 10], [1, 3, 8]), (24, [2, 10, 12], [1, 3, 9, 11])])
def test_untouched_blocks_are_taken(layers, few, many, through):
    assert through(*build(layers, 1024)) == (few, 0)
    assert through(*build(layers, 1025)) == (many, 0)


@pytest.mark.parametrize("name", ["__call__", "_call_impl"])
@pytest.mark.parametrize("kind", ["_Block", "FusedAttention", "FusedMLP"])
def test_a_call_of_the_class_runs(kind, name, through, monkeypatch):
    model, x = build()
    with monkeypatch.context() as m:
        m.setattr(getattr(gpt, kind), name, lambda self, *a, **k: None, raising=False)
        assert through(model, x) == ([], 3)
    assert through(model, x) == ([1, 2], 0)


@pytest.mark.parametrize("name", ["forward", "_weights", "_call_impl", "_wrapped_call_impl"])
@pytest.mark.parametrize("which", [0, 1])
def test_what_an_instance_has_in_the_place_of_a_method_runs(name, which, through):
    model, x = build()
    for block, want in ((0, ([], 3)), (1, ([1], 2)), (2, ([1, 1], 1))):
        module = model.blocks[block][which]
        setattr(module, name, lambda *a, **k: None)
        assert through(model, x) == want
        delattr(module, name)
    assert through(model, x) == ([1, 2], 0)


@pytest.mark.parametrize("name", ["attention_block", "mlp_block", "layer_norm_ffn", "_weights", "_tensors"])
def test_a_replaced_function_runs(name, through, monkeypatch):
    model, x = build()
    monkeypatch.setattr(gpt, name, lambda *a, **k: None)
    assert through(model, x) == ([], 3)


def test_the_layers_in_front_of_another_one_are_taken(through):
    changes = [lambda block: setattr(block[1].ffn2_weight, "data", torch.zeros(1024, 64)), lambda block: block[0].train(),
               lambda block: block.append(torch.nn.Identity()), lambda block: block.__setattr__("extra", block[0]),
               lambda block: block[0].register_forward_hook(lambda *a: None),
               lambda block: block[1].register_forward_pre_hook(lambda *a: None),
               lambda block: block.register_forward_hook(lambda *a: None),
               lambda block: setattr(block[0], "hidden_size", 64),
               lambda block: setattr(block[0].c_attn_bias, "data", block[0].c_attn_bias.data.half()),
               lambda block: setattr(block[0].c_attn_bias, "data", torch.zeros(768)[::2]),
               lambda block: setattr(block[1].layer_norm_bias, "data", torch.zeros(1, 128)),
               lambda block: block[1]._parameters.pop("ffn1_bias"),
               lambda block: block[1]._parameters.__setitem__("ffn1_bias", torch.zeros(512)),
               lambda block: block[0]._parameters.__setitem__("c_proj_weight", torch.zeros(128, 128)),
               lambda block: block[0]._packed._entries.clear() or block[0]._parameters.pop("c_proj_weight"),
               lambda block: setattr(block[0].c_attn_weight, "data", torch.zeros(384, 128).t())]
    with torch.no_grad():
        for change in changes:
            for block, want in ((0, ([], 5)), (1, ([1], 4)), (2, ([1, 1], 3)), (4, ([1, 3], 1))):
                model, x = build(5)
                change(model.blocks[block])
                if change is changes[0]:
                    model.blocks[block][1]._packed.get("ffn2_weight", model.blocks[block][1].ffn2_weight, pack)
                calls, left = through(model, x)
                assert (calls, left) == want, (changes.index(change), block)


@pytest.mark.parametrize("edit", [lambda block: block[0].c_proj_weight.add_(1), lambda block: block[1]._packed.clear(),
                                  lambda block: setattr(block[1], "ffn2_weight", torch.nn.Parameter(torch.zeros(512, 128)))])
def test_images_that_are_not_held_are_built(edit, through, monkeypatch):
    packed = []
    monkeypatch.setattr(gpt._PackedWeights.get, "__defaults__", (lambda w: packed.append(w) or pack(w),))
    with torch.no_grad():
        for block, calls in ((0, [1, 1, 3]), (1, [1, 3, 1]), (4, [1, 3, 1])):
            model, x = build(5)
            edit(model.blocks[block])
            packed.clear()
            assert through(model, x) == (calls, 0) and 1 <= len(packed) <= 2
            packed.clear()
            assert through(model, x) == ([1, 3, 1], 0) and not packed
    # none built for a module whose other weight cannot be packed
    model, x = build(2)
    model.blocks[1][0].train().eval()
    model.blocks[1][0]._parameters["c_proj_weight"] = torch.zeros(128, 128)
    assert through(model, x) == ([1], 1) and not packed


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
