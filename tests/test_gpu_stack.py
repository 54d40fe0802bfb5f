"""The blocks of an eval-mode forward in one call of the library (gptmi_blocks): the bits of the modules
called one by one, and whatever a program has put on or in the place of a module, an operator or a
parameter still runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G(gpu_device):
    from gpt_triton_amd import gpt
    return gpt


def build(G, device, dtype, layers=3, heads=4, width=256):
    torch.manual_seed(5)
    model = G.FusedGPT(G.GPTConfig(n_layer=layers, n_head=heads, n_embd=width, vocab_size=101, block_size=512))
    with torch.no_grad():
        for name, prm in model.named_parameters():
            prm.normal_(1.0 if name.endswith("layer_norm_weight") else 0.0, 0.05)
    model = model.to(device=device, dtype=dtype).eval()
    with torch.no_grad():  # the first forward builds the weight images
        model(torch.zeros((1, 8), dtype=torch.int64, device=device))
    return model


def one_by_one(G, model, ids, monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(G, "_stack", lambda blocks, x: None)
        return model(ids)


def counted(G, monkeypatch):
    calls = []
    real = G.blocks_forward
    monkeypatch.setattr(G, "blocks_forward", lambda *a, **k: calls.append(1) or real(*a, **k))
    return calls


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,layers,heads,width", [(1, 1, 1, 2, 128), (2, 64, 3, 12, 768), (3, 77, 2, 4, 256),
                                                    (1, 24, 12, 16, 1024), (5, 300, 2, 2, 512)])
def test_same_bits_as_the_modules(G, gpu_device, dtype, B, L, layers, heads, width, monkeypatch):
    print(f"stack {dtype} B={B} L={L} layers={layers} heads={heads} width={width}", flush=True)
    model = build(G, gpu_device, dtype, layers, heads, width)
    ids = torch.randint(0, 101, (B, L), device=gpu_device)
    with torch.no_grad():
        calls = counted(G, monkeypatch)
        got = model(ids)
        assert calls == [1]
        assert torch.equal(got, one_by_one(G, model, ids, monkeypatch)) and calls == [1]


def test_what_a_program_changed_still_runs(G, gpu_device, monkeypatch):
    model = build(G, gpu_device, torch.float16)
    ids = torch.randint(0, 101, (2, 40), device=gpu_device)
    calls = counted(G, monkeypatch)
    with torch.no_grad():
        plain = model(ids)
        assert calls.pop() == 1
        # hooks: on a block, on its modules, on every module
        seen = []
        for module in (model.blocks[1], model.blocks[0][0], model.blocks[2][1]):
            for register in (module.register_forward_hook, module.register_forward_pre_hook):
                handle = register(lambda *a: seen.append(1))
                assert torch.equal(model(ids), plain)
                handle.remove()
        assert len(seen) == 6 and not calls
        handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(1))
        model(ids)
        handle.remove()
        assert len(seen) > 10 and not calls
        # a forward replaced on an instance and in the class
        model.blocks[1][1].forward = lambda x: x
        changed = model(ids)
        assert not torch.equal(changed, plain) and not calls
        del model.blocks[1][1].forward
        with monkeypatch.context() as m:
            m.setattr(G.FusedMLP, "forward", lambda self, x: x)
            assert not torch.equal(model(ids), plain) and not calls
        # an operator replaced, a module exchanged or appended
        with monkeypatch.context() as m:
            m.setattr(G, "attention_block", lambda x, *a, **k: x)
            assert not torch.equal(model(ids), plain) and not calls
        model.blocks[1].append(torch.nn.Identity())
        assert torch.equal(model(ids), plain) and not calls
        del model.blocks[1][2]
        # weights edited in place, and others in the place of the parameters
        model.blocks[0][0].c_proj_weight.mul_(1.5)
        edited = model(ids)  # not whole from images at hand: one has to be built again
        assert not calls and not torch.equal(edited, plain)
        assert torch.equal(model(ids), edited) and calls.pop() == 1
        assert torch.equal(edited, one_by_one(G, model, ids, monkeypatch))
        other = {k: torch.zeros_like(p) for k, p in model.named_parameters() if k.endswith("ffn2_weight")}
        assert not torch.equal(torch.func.functional_call(model, other, (ids,)), edited) and not calls
        assert torch.equal(model(ids), edited) and calls.pop() == 1
        # one module in training mode draws its dropout
        model.blocks[2][1].train()
        assert not torch.equal(model(ids), edited) and not calls
        model.blocks[2][1].eval()
        # parameters of another type are refused as the block calls refuse them
        model.blocks[1][0].c_attn_bias.data = model.blocks[1][0].c_attn_bias.data.float()
        with pytest.raises(TypeError):
            model(ids)
    assert not calls


def test_captured_and_on_a_stream_of_its_own(G, gpu_device):
    model = build(G, gpu_device, torch.float16, 2, 12, 768)
    ids = torch.randint(0, 101, (2, 64), device=gpu_device)
    with torch.no_grad():
        want = model(ids)
        graph = G.GraphedForward(model, ids)
        for _ in range(4):
            assert torch.equal(graph(ids), want)
            assert torch.equal(model(ids), want)
            torch.cuda.synchronize()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got = model(ids)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(got, want)


@pytest.mark.parametrize("one_call", [True, False])
def test_first_forward_under_capture_keeps_no_images(G, gpu_device, one_call, monkeypatch):
    """A weight image whose packing is recorded into a graph does not exist until a replay: an eager forward
    between capture and replay builds its own."""
    ids = torch.randint(0, 101, (2, 24), device=gpu_device)
    if not one_call:
        monkeypatch.setattr(G, "_stack", lambda blocks, x: None)
    with torch.no_grad():
        want, logits = build(G, gpu_device, torch.float16)(ids, return_logits=True)
        model = build(G, gpu_device, torch.float16)  # the same weights
        model.train().eval()  # drops its images
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = model(ids, return_logits=True)
        assert not any(m._packed._entries for m in model.modules() if hasattr(m, "_packed"))
        for _ in range(3):
            got = model(ids, return_logits=True)
            assert torch.equal(got[0], want) and torch.equal(got[1], logits)
            graph.replay()
            assert torch.equal(captured[0], want) and torch.equal(captured[1], logits)
            torch.cuda.synchronize()


def test_arguments_are_refused_before_any_launch(gpu_device):
    import ctypes

    from gpt_triton_amd import _lib
    lib = _lib.load()
    fake = ctypes.c_void_p(256)
    prm = (ctypes.c_void_p * 12)(*[256] * 12)
    need = lib.gptmi_blocks_workspace_bytes(1, 8, 2, 64, 512, 1)
    assert need > 0 and lib.gptmi_blocks_workspace_bytes(1, 8, 2, 64, 512, 7) == 0
    for n, d, inner, nbytes, dtype, rc in ((0, 64, 512, need, 1, -1), (1, 64, 512, need - 1, 1, -3),
                                           (1, 48, 512, 1 << 30, 1, -2), (1, 64, 512, need, 7, -1),
                                           (1, 64, 0, need, 1, -1)):
        assert lib.gptmi_blocks(fake, None, prm, n, 1e-5, fake, 1, 8, 2, d, inner, 0, fake, nbytes, dtype,
                                None) == rc
