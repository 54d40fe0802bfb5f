"""Host-side checks that need no GPU: the C-ABI library loads and exports exactly what
include/gptmi.h declares, argument validation answers before any launch, the model helpers
reproduce the reference's known answers (test.py:136-152), and CPU tensors are refused."""
import ctypes
import os
import re

import pytest
import torch

from gpt_triton_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_lib.LIB_PATH):
        from gpt_triton_amd import build

        build.build()
    return _lib.load()


def declared_functions():
    text = open(os.path.join(ROOT, "include", "gptmi.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gptmi_[a-z_0-9]+)\s*\(", text)))


def test_header_symbols_are_exported_and_bound(lib):
    names = declared_functions()
    assert len(names) >= 11
    for name in names:
        assert hasattr(lib, name), f"{name} declared in gptmi.h but not exported"
    assert sorted(_lib.SIGNATURES) == names, "ctypes prototypes and gptmi.h disagree"


def test_version_and_error_string(lib):
    assert lib.gptmi_version() == 102
    assert isinstance(lib.gptmi_last_error(), bytes)


def test_invalid_arguments_are_rejected_before_any_launch(lib):
    # NULL pointers / bad sizes -> GPTMI_ERR_INVALID (-1); none of these touches the GPU
    assert lib.gptmi_embed(None, None, None, None, 1, 1, 1, 1, 1, 0.0, 0, 1, None) == -1
    assert lib.gptmi_layernorm(None, None, None, None, 4, 4, 1e-5, 1, None) == -1
    assert lib.gptmi_softmax(None, None, 4, 4, 0, None) == -1
    assert lib.gptmi_linear(None, None, None, None, None, 1, 1, 1, 0, 0.0, 0, 0, None, 0, 1, None) == -1
    assert lib.gptmi_flash_attn(None, None, None, None, 1, 1, 1, 1, 64, 0.125, 0.0, 0, 0, 1, None) == -1
    fake = ctypes.c_void_p(256)  # never dereferenced: validation fails first
    assert lib.gptmi_layernorm(fake, fake, fake, fake, 4, 4, 1e-5, 7, None) == -1       # bad dtype
    assert lib.gptmi_layernorm(fake, fake, fake, fake, 4, 10000, 1e-5, 1, None) == -2   # H too large
    assert b"8192" in lib.gptmi_last_error()
    assert lib.gptmi_embed(fake, fake, fake, fake, 1, 8, 4, 4, 8, 0.0, 0, 1, None) == -1  # L > P
    assert lib.gptmi_embed(fake, fake, fake, fake, 1, 4, 4, 4, 8, 1.0, 0, 1, None) == -1  # p >= 1
    assert lib.gptmi_flash_attn(fake, fake, fake, fake, 1, 1, 8, 8, 64, 0.125, -0.1, 0, 0, 1,
                                None) == -1                                             # p < 0
    assert lib.gptmi_flash_attn(fake, fake, fake, fake, 1, 1, 8, 9, 48, 0.125, 0.0, 0, 0, 1,
                                None) == -2                                             # head size
    # output rows wider than the epilogues' 32-bit lane offsets can address: refused, not wrapped
    wide = (1 << 26) + 8
    assert lib.gptmi_linear(fake, fake, None, None, fake, 4, wide, 64, 0, 0.0, 0, 2, None, 0, 1,
                            None) == -2
    assert b"N=" in lib.gptmi_last_error()
    assert lib.gptmi_linear_static(fake, fake, None, None, fake, 4, wide, 64, 0, 0.0, 0, 2, 1,
                                   None) == -2
    assert lib.gptmi_linear_qkv(fake, fake, None, fake, fake, fake, 1, 4, 1 << 20, 64, 64, 2,
                                None, 0, 1, None) == -2                    # N = 3 * 2^26
    assert lib.gptmi_linear(fake, fake, None, None, fake, 4, 4, 4, 0, 0.0, 0, 0, None, 0, 1,
                            None) == -3                                                 # workspace


def test_workspace_sizes(lib):
    # fp16, K multiple of 64, [K][N] weight: only the packed weight (N * K * 2 bytes)
    assert lib.gptmi_linear_workspace_bytes(153600, 3072, 768, 1, 0) == 3072 * 768 * 2
    # already [N][K] fp16: nothing to pack
    assert lib.gptmi_linear_workspace_bytes(153600, 50257, 768, 1, 1) == 0
    assert lib.gptmi_linear_workspace_bytes(153600, 3072, 768, 1, 2) == 0
    # fp32 storage: weight and activations are both repacked to fp16
    assert lib.gptmi_linear_workspace_bytes(128, 64, 64, 0, 0) == 64 * 64 * 2 + 128 * 64 * 2
    # K = 23 pads to 64
    assert lib.gptmi_packed_weight_bytes(31, 23) == 31 * 64 * 2 + (256 - 31 * 64 * 2 % 256) % 256


def test_flops_known_answers():
    # test.py:136-144
    from gpt_triton_amd.gpt import FusedGPT, GPTConfig, get_num_parameters

    model = FusedGPT(GPTConfig()).eval()
    fwd = model.get_fwd_flops(1024)
    n = get_num_parameters(model)
    assert fwd == 253997088768 and n == 124082688
    assert (fwd * 3) / (6 * n * 1024) >= 0.9995


def test_estimate_days_known_answer():
    # test.py:147-152
    from gpt_triton_amd.gpt import compute_mfu, estimate_days

    flops = 6 * (405 * 10**9) * (15 * 10**12)
    assert estimate_days(flops, mfu=0.45, gpu="h100", num_gpus=16_000) == 59.24544994944388
    assert compute_mfu(2 * 124 * 10**6 * 512 * 512 / 0.273, gpu="h100") == pytest.approx(0.2407, abs=2e-4)
    assert compute_mfu(1.0e15, gpu="mi355x") == pytest.approx(0.4)


def test_state_dict_keys_match_the_reference_layout():
    from gpt_triton_amd.gpt import FusedGPT, GPTConfig

    keys = set(FusedGPT(GPTConfig(n_layer=2)).state_dict())
    want = {"wte_weight", "wpe_weight", "layer_norm_weight", "layer_norm_bias"}
    for i in range(2):
        for k in ("layer_norm_weight", "layer_norm_bias", "c_attn_weight", "c_attn_bias",
                  "c_proj_weight", "c_proj_bias"):
            want.add(f"blocks.{i}.0.{k}")
        for k in ("layer_norm_weight", "layer_norm_bias", "ffn1_weight", "ffn1_bias", "ffn2_weight",
                  "ffn2_bias"):
            want.add(f"blocks.{i}.1.{k}")
    assert keys == want


def test_hf_key_conversion():
    from types import SimpleNamespace

    from gpt_triton_amd.gpt import FusedGPT, convert_huggingface_to_triton

    cfg = SimpleNamespace(vocab_size=11, n_positions=8, n_layer=1, n_head=2, n_embd=4)
    h = 4
    hf = {"wte.weight": torch.zeros(11, h), "wpe.weight": torch.zeros(8, h),
          "ln_f.weight": torch.ones(h), "ln_f.bias": torch.zeros(h),
          "h.0.ln_1.weight": torch.ones(h), "h.0.ln_1.bias": torch.zeros(h),
          "h.0.attn.bias": torch.ones(1, 1, 8, 8),
          "h.0.attn.c_attn.weight": torch.zeros(h, 3 * h), "h.0.attn.c_attn.bias": torch.zeros(3 * h),
          "h.0.attn.c_proj.weight": torch.zeros(h, h), "h.0.attn.c_proj.bias": torch.zeros(h),
          "h.0.ln_2.weight": torch.ones(h), "h.0.ln_2.bias": torch.zeros(h),
          "h.0.mlp.c_fc.weight": torch.zeros(h, 4 * h), "h.0.mlp.c_fc.bias": torch.zeros(4 * h),
          "h.0.mlp.c_proj.weight": torch.zeros(4 * h, h), "h.0.mlp.c_proj.bias": torch.zeros(h)}
    sd, config = convert_huggingface_to_triton(hf, cfg)
    assert config.block_size == 8 and config.n_head == 2
    FusedGPT(config).load_state_dict(sd)  # every key present, none extra


def test_cpu_tensors_are_refused_not_emulated(lib):
    from gpt_triton_amd import kernels as K

    x = torch.zeros(4, 64)
    w = torch.zeros(64, 64)
    with pytest.raises(RuntimeError, match="GPU only"):
        K.fused_ffn(x, w)
    with pytest.raises(RuntimeError, match="GPU only"):
        K.fused_layer_norm(x, torch.ones(64), torch.zeros(64))
    with pytest.raises(RuntimeError, match="GPU only"):
        K.fused_embeddings(torch.zeros(2, 3, dtype=torch.long), w, w)
    q = torch.zeros(1, 1, 8, 64)
    with pytest.raises(RuntimeError, match="GPU only"):
        K.flash_attention_v1(q, q, q)


@pytest.mark.parametrize("name", ["layer_norm_weight", "layer_norm_bias", "c_attn_bias", "c_proj_bias",
                                  "ffn1_bias", "ffn2_bias"])
def test_blocks_check_the_sizes_of_their_vectors(lib, name):
    """A vector shorter than the kernels read is refused as by the single operators, before the
    library is called."""
    from gpt_triton_amd import kernels

    h = 64
    vec = {"layer_norm_weight": h, "layer_norm_bias": h, "c_attn_bias": 3 * h, "c_proj_bias": h,
           "ffn1_bias": 4 * h, "ffn2_bias": h}
    vec = {k: torch.zeros(n - 1 if k == name else n) for k, n in vec.items()}
    x, ln = torch.zeros(1, 2, h), (vec["layer_norm_weight"], vec["layer_norm_bias"])
    attention = lambda: kernels.attention_block(x, *ln, torch.zeros(h, 3 * h), vec["c_attn_bias"],
                                                torch.zeros(h, h), vec["c_proj_bias"], 1)
    mlp = lambda: kernels.mlp_block(x, *ln, torch.zeros(h, 4 * h), vec["ffn1_bias"],
                                    torch.zeros(4 * h, h), vec["ffn2_bias"])
    for block, takes in ((attention, not name.startswith("ffn")), (mlp, not name.startswith("c_"))):
        with pytest.raises(AssertionError if takes else RuntimeError):
            block()


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys

    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True)
    assert r.returncode != 0 and "--gpus must be 1" in r.stderr


def test_replaced_forwards_are_called_with_x_alone(monkeypatch):
    # a forward wrapped to time or record it takes what nn.Sequential hands it, with dropout too
    from gpt_triton_amd import gpt

    monkeypatch.setattr(gpt, "fused_embeddings", lambda ids, *a, **k: torch.zeros(*ids.shape, 64))
    monkeypatch.setattr(gpt, "fused_layer_norm", lambda x, w, b: x)
    monkeypatch.setattr(gpt, "dropout_mask", lambda bits, p, like: "mask")
    ids = torch.zeros((1, 4), dtype=torch.int64)
    # on the instances of a block's two modules, on the block, on the class
    model = gpt.FusedGPT(gpt.GPTConfig(n_layer=2, n_head=1, n_embd=64)).train()
    for block in model.blocks:
        block[0].forward = lambda x: x + 1
        block[1].forward = lambda x: x * 2
    assert torch.equal(model(ids), torch.full((1, 4, 64), 6.0))
    model.blocks[1].forward = lambda x: x - 1
    assert torch.equal(model(ids), torch.full((1, 4, 64), 1.0))
    model = gpt.FusedGPT(gpt.GPTConfig(n_layer=2, n_head=1, n_embd=64)).train()
    monkeypatch.setattr(gpt.FusedAttention, "forward", lambda self, x: x + 1)
    monkeypatch.setattr(gpt.FusedMLP, "forward", lambda self, x: x * 2)
    assert torch.equal(model(ids), torch.full((1, 4, 64), 6.0))
    # what takes the mask gets it, in a subclass too
    class Attention(gpt.FusedAttention):
        pass

    monkeypatch.undo()
    seen = []
    monkeypatch.setattr(gpt, "attention_block", lambda x, *a, keep=None, **k: seen.append(keep))

    class Mask:
        serves = staticmethod(lambda x, bits, p: True)

    gpt._Block(Attention(64, 1, dropout_prob=0.1), torch.nn.Identity()).train()(torch.zeros(1, 4, 64), keep=Mask)
    assert seen == [Mask]


def test_weight_images_are_kept_for_parameters_only(monkeypatch):
    # torch.func.functional_call puts plain tensors in the place of the parameters: another tensor on
    # every call, whose address and version say nothing about its values
    from torch.func import functional_call

    from gpt_triton_amd import gpt

    class Probe(torch.nn.Module):
        def __init__(self, module, names):
            super().__init__()
            self.module, self.names = module, names

        def forward(self):
            if self.names == [None]:
                return [self.module._lm_head_weight()]
            return self.module._weights(self.module._parameters)

    model = gpt.FusedGPT(gpt.GPTConfig(n_layer=1, n_head=1, n_embd=64, vocab_size=64)).eval()
    for module, names in ((gpt.FusedAttention(64, 1).eval(), ["c_attn_weight", "c_proj_weight"]),
                          (gpt.FusedMLP(64).eval(), ["ffn1_weight", "ffn2_weight"]), (model, [None])):
        kept = []
        module._packed.get = lambda name, prm, pack=None: kept.append(name)
        probe = Probe(module, names)
        probe()
        assert kept == [n or "lm_head" for n in names]
        kept.clear()
        plain = {n: p.detach().clone() for n, p in probe.named_parameters()}
        got = functional_call(probe, plain)
        assert not kept
        for n, t in zip(names, got):
            assert t.data_ptr() == plain[f"module.{n or 'wte_weight'}"].data_ptr()
        # one of the two replaced: the block calls take both weights packed or neither
        name = f"module.{names[0] or 'wte_weight'}"
        functional_call(probe, {name: plain[name]})
        assert not kept


def test_attention_block_checks_the_head_size_before_any_launch(lib):
    fake = ctypes.c_void_p(256)
    for heads, d in ((16, 4), (8, 24), (2, 96), (1, 512)):
        need = lib.gptmi_attention_block_workspace_bytes(1, 8, heads, d, 2)
        rc = lib.gptmi_attention_block(fake, None, fake, fake, 1e-5, fake, fake, fake, fake, fake, 1, 8, heads, d,
                                       0.0, 1337, None, 0, 0, 2, fake, need, 1, None)
        assert rc == -2 and b"head size" in lib.gptmi_last_error()


def test_the_tile_gemm_cases_reach_every_tile():
    # the cost model of gemm_tile.hip, its numbers read from there, on 256 CUs
    import test_gpu_gemm_tile

    source = open(os.path.join(ROOT, "gpt_triton_amd", "csrc", "gemm_tile.hip")).read()
    menu = re.search(r"TileCost kTiles\[\] = \{(.*?)\};", source, re.S).group(1)
    tiles = [[float(v.rstrip("f")) for v in row.split(",")] for row in re.findall(r"\{([^{}]*)\}", menu)]
    assert len(tiles) == 8

    def pick(M, N, slices):
        def cost(tile):
            bm, bn, _, launch, fixed, per_slice = tile
            rounds = -(-(-(-M // int(bm)) * -(-N // int(bn))) // 256)
            return launch + rounds * (fixed + slices * per_slice)
        return min(range(len(tiles)), key=lambda i: cost(tiles[i]))

    picked = {(pick(M, N, -(-K // 64)), -(-K // 64)) for M, N, K in test_gpu_gemm_tile.SHAPES}
    assert {i for i, _ in picked} == set(range(len(tiles)))
    # k-slices: fewer than the groups; as many and more, with groups that have none in the last k-step
    groups = [int(tile[2]) for tile in tiles]
    assert any(slices < groups[i] for i, slices in picked)
    for i in range(3):  # the four-way splits
        assert groups[i] == 4 and {s % 4 == 0 for j, s in picked if j == i} == {True, False}
    sizes = [(M, N) for M in (1, 8, 24, 64, 128, 200, 513, 1477, 4800) for N in (16, 40, 768, 2304, 6400)]
    assert all(groups[pick(M, N, slices)] < 4 for M, N in sizes for slices in (1, 2, 3))


@pytest.mark.parametrize("B,L,heads", [(1, (1 << 24) + 1, 1), (1 << 31, 1, 1)])
def test_attention_block_checks_the_grid_before_any_launch(lib, B, L, heads):
    fake = ctypes.c_void_p(256)
    need = lib.gptmi_attention_block_workspace_bytes(B, L, heads, 64, 2)
    rc = lib.gptmi_attention_block(fake, None, fake, fake, 1e-5, fake, fake, fake, fake, fake, B, L, heads, 64,
                                   0.0, 1337, None, 0, 0, 2, fake, need, 1, None)
    assert rc == -2 and lib.gptmi_last_error().startswith(b"attention_block:")
