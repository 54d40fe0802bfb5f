"""Model layer: GPTConfig / FusedGPT / FusedAttention / FusedMLP and the FLOP helpers, with the
class names, constructor arguments and state_dict keys of the reference's gpt.py so that a
checkpoint or calling code written for it works unchanged:

    FusedAttention(hidden_size, num_heads, dropout_prob=0.0)     gpt.py:21-67
    FusedMLP(hidden_size, dropout_prob=0.0)                      gpt.py:70-119
    GPTConfig                                                    gpt.py:122-129
    FusedGPT(config)                                             gpt.py:132-196
    convert_huggingface_to_triton(hf_sd, hf_config)              gpt.py:199-237
    estimate_days / get_num_parameters / compute_mfu             gpt.py:250-263

Differences, all additive: GPU_TO_FLOPS knows "mi355x"; FusedGPT.forward takes
`return_logits=True` for the tied LM head the reference leaves commented out
(gpt.py:159-161, 172-179); `init_synthetic_` draws the N(0, 0.02) benchmark weights;
`FusedGPT.forward` reads `config.dropout` (the reference reads a `dropout_prob` attribute the
dataclass does not have, gpt.py:165, and so only works in eval mode).
"""
import re
import weakref
from dataclasses import dataclass

import torch
import torch.nn as nn
from torch.multiprocessing.reductions import StorageWeakRef

from .kernels import (HEAD_SIZES, PackedWeight, attention_block, block_layers, block_supported, blocks_forward,
                      blocks_workspace, dropout_mask, flash_attention_v1, fused_embeddings,
                      fused_embeddings_layer_norm, fused_ffn,
                      fused_layer_norm, layer_norm_ffn, layer_norm_linear_supported,
                      layer_norm_matmul_and_split_qkv, lm_head, matmul_and_split_qkv, mlp_block,
                      pack_lm_head, pack_weight)

# Up to this many token rows of up to this width the blocks run their LayerNorm inside the following
# GEMM (same bits, a launch less).  The fused form normalises a row block once per column tile, in front
# of its first product, and one of its workgroups fills a CU.  So it pays while all column tiles run at
# once and while normalising 16 or 32 rows costs less than a launch: 160 rows up to 768, up to 1024 as many as take
# tiles of 16 rows.  LayerNorm -> ffn1 at 24 / 128 / 160 / 192 rows of 768 takes 5.4 / 7.5 / 7.6 / 12.2 us against 6.4 /
# 7.7 / 8.3 / 8.3 for the two launches, 24 of 1280 9.8 against 8.8, 24 of 1600 12.0 against 10.1.  Forwards of the
# 1024-wide model, two launches / one, us: 1 x 8 tokens replayed 636 / 622, eager 778 / 632, 1 x 24 651 / 630 and 781 /
# 651, 1 x 41 671 / 671 and 785 / 667, 1 x 64 689 / 675 and 793 / 670, 1 x 80 745 / 754 and 791 / 749, 2 x 64 803 / 805 and 803 /
# 807 (eager ones of few rows wait for the host).  fp32 models' blocks do it without being asked, up to the same limits in the
# library (prologue_f32 in csrc/capi.cpp); LN_PROLOGUE_MAX_ROWS = 0 turns it off in both types.
LN_PROLOGUE_MAX_ROWS = 160
LN_PROLOGUE_MAX_WIDTH = 768
LN_PROLOGUE_FEW_ROWS = 64
LN_PROLOGUE_FEW_WIDTH = 1024

# Up to this many elements of the residual stream a block is one call of the library (attention_block,
# mlp_block) instead of one per operator.  Up to about 2000 rows of the 124M model and 1000 of the 1024-wide one
# the host sets the pace of an operator-by-operator forward (some 10 us per operator against 2 us per launch
# inside one call: 512 rows 926 against 567 us, 2048 rows 910 against 826; 1024-wide 512 rows 1777
# against 1291).  Beyond, what a block passes through fits or nearly fits the 256 MB memory-side cache where
# every layer writes it to the same places, as the calls do and a caching allocator does not: LayerNorm of 48 x
# 300 rows 7.8 us instead of 18.6 behind the MLP; operators / blocks: 64 x 300 tokens of 124M 4273 / 4024, 72 x 300 4527 /
# 4255, 96 x 300 6069 / 5961, 140 x 300 8367 / 8229; 1024 wide 9 x 1024 8062 / 7363, 31 x 1024 21426 / 21112; 1600 wide 16 x
# 1024 51342 / 51149; 6144 wide 8 x 700 14180 / 14210.  Up to the limit (43690 rows of 768) a block holds seven matrices of
# the stream and the MLP's inner one at once; the operators, which give each intermediate matrix back
# before they take the next, need a quarter to a third less (140 x 300: 492 MB instead of 677) and stay beyond, where
# the two are equal.  fp32 models take the block calls at every size: their
# intermediate matrices are fp16 there (see gptmi_attention_block).
BLOCK_MAX_ELEMENTS = 1 << 25


def _ln_in_gemm(x, weight):
    width = x.shape[-1]
    few = width > LN_PROLOGUE_MAX_WIDTH
    rows = min(LN_PROLOGUE_MAX_ROWS, LN_PROLOGUE_FEW_ROWS) if few else LN_PROLOGUE_MAX_ROWS
    if LN_PROLOGUE_MAX_ROWS == 0:
        return None
    return (width <= LN_PROLOGUE_FEW_WIDTH and x.numel() // width <= rows and
            layer_norm_linear_supported(x, weight))


def _as_block(x, keep=None):
    width = x.shape[-1]
    return ((keep is not None or x.dtype == torch.float32 or x.numel() <= BLOCK_MAX_ELEMENTS) and
            block_supported(x, width))


# dense fp16/bf16 tensor throughput, FLOP/s
GPU_TO_FLOPS = {
    "v100": 130 * 10**12,
    "a100": 312 * 10**12,
    "h100": 989 * 10**12,
    "mi355x": 2500 * 10**12,
}


def _keep_mask(x, width, layers, heads, p):
    """The dropout mask of a training forward's blocks, or None where the kernels draw their own: sizes
    the block calls do not take, and more offsets than the generator has.  The reference draws the
    masks of all layers from one seed at offsets that count from 0, so they are all parts of the mask
    of the widest matrix ([tokens, 4 * width]; attention weights: the first L * L offsets).  Drawn
    once per forward instead of in every kernel that applies it: 16 x 300 tokens 124M, each of 12 ffn1
    launches 85 -> 31 us, projections and ffn2 32 -> 22, attentions 72 -> 18, for one launch of 25."""
    tokens, seqlen = x.numel() // width, x.shape[1]
    bits = max(tokens * 4 * width, seqlen * seqlen)
    if (layers == 0 or bits > 1 << 32 or not block_supported(x, width) or width % heads != 0 or
            width // heads not in HEAD_SIZES):
        return None
    return dropout_mask(bits, p, x)


class _Block(nn.Sequential):
    """nn.Sequential(FusedAttention, FusedMLP) whose two modules may be handed a dropout mask.  Any
    other module put in their place is called as nn.Sequential calls it."""

    def forward(self, x, keep=None):
        for module in self:
            x = module(x) if keep is None else _call_with_mask(module, x, keep)
        return x


def _call_with_mask(module, x, keep):
    """module(x), with the mask where the forward that the call will run is one of this file's: one
    replaced on the instance, in its class or by a subclass takes what nn.Sequential hands it."""
    if getattr(module.forward, "__func__", None) in _TAKE_MASK:
        return module(x, keep=keep)
    return module(x)


_storage_expired = torch.UntypedStorage._expired  # of a StorageWeakRef's cdata


class _PackedWeights:
    """Per-module cache of the GEMM's packed weight images, used in eval mode only.  An entry is that of one
    Parameter object while it has the storage, address, dtype, shape and version counter that it was
    packed with (optimizer steps, load_state_dict, .to() and assignments change one of them), and is
    rebuilt otherwise.  Parameter and storage are referred to weakly: nothing is kept alive by its image,
    and an address that was freed and handed out again is not taken for the weight that lay there before.
    In-place edits made through `param.data` bypass the version counter -- call `clear()` (or
    `model.train()`) after those.  Copies and pickles of a module start without images."""

    def __init__(self):
        self._entries = {}

    def get(self, name, param, pack=pack_weight):
        hit = self.held(name, param)
        if hit is None:
            hit = pack(param.data)
            if param.is_cuda and torch.cuda.is_current_stream_capturing():
                return hit  # recorded into a graph and not there yet: this forward's alone
            storage = StorageWeakRef(param.untyped_storage())
            self._entries[name] = (weakref.ref(param), storage.cdata, param.data_ptr(), param._version,
                                   param.dtype, param.shape, hit, storage)
        return hit

    def held(self, name, param):
        """The image of this parameter as it is now, or None where there is none yet."""
        entry = self._entries.get(name)
        if entry is None:
            return None
        owner, storage, address, version, dtype, shape, hit, _ = entry
        # an address inside a storage that is still there is that storage's: no other has it
        if (owner() is not param or param._version != version or param.data_ptr() != address or
                param.dtype != dtype or param.shape != shape or not param.is_contiguous() or
                _storage_expired(storage)):
            return None
        return hit

    def clear(self):
        self._entries.clear()

    def __reduce__(self):
        return _PackedWeights, ()

    def __setstate__(self, state):  # of a pickle that holds entries
        self._entries = {}


def _linear_flops(tokens, fan_in, fan_out):
    # multiply-adds of the product plus the bias add, as gpt.py:62-67 / 113-119 count them
    return tokens * fan_out * (2 * fan_in) + tokens * fan_out


def _norm_flops(tokens, width):
    return 2 * tokens * width


def _tensors(module, names):
    """The tensors of a module by name: its dictionary of parameters where that has them all (an
    attribute of an nn.Module takes a failed lookup of its class and instance first, and a forward of
    few tokens waits for the host), else its attributes, which is where pruning, parametrisations
    and replicas put what stands in a parameter's place."""
    prm = module._parameters
    return prm if names <= prm.keys() else {name: getattr(module, name) for name in names}


def _weights(module, tensors, first, second):
    """A module's two weights as the products take them: images in eval mode, kept for parameters only,
    and for both or neither.  What stands in for one is another tensor every time, in the dictionary of
    parameters too (torch.func.functional_call puts plain tensors there)."""
    a, b = tensors[first], tensors[second]
    if (module.training or tensors is not module._parameters or not isinstance(a, nn.Parameter) or
            not isinstance(b, nn.Parameter)):
        return a.data, b.data
    return module._packed.get(first, a), module._packed.get(second, b)


class FusedAttention(nn.Module):
    """Pre-LN causal self-attention block: x + proj(attention(qkv(LN(x))))."""

    def __init__(self, hidden_size, num_heads, dropout_prob=0.0):
        super().__init__()
        self.hidden_size = hidden_size
        self.num_heads = num_heads
        self.dropout_prob = dropout_prob
        h = hidden_size
        self.layer_norm_weight = nn.Parameter(torch.ones(h))
        self.layer_norm_bias = nn.Parameter(torch.zeros(h))
        self.c_attn_weight = nn.Parameter(torch.rand(h, 3 * h))
        self.c_attn_bias = nn.Parameter(torch.rand(3 * h))
        self.c_proj_weight = nn.Parameter(torch.rand(h, h))
        self.c_proj_bias = nn.Parameter(torch.rand(h))
        self._packed = _PackedWeights()

    _NAMES = frozenset(("layer_norm_weight", "layer_norm_bias", "c_attn_weight", "c_attn_bias",
                        "c_proj_weight", "c_proj_bias"))

    def _weights(self, tensors):
        if (self.hidden_size // self.num_heads) % 8 != 0:
            return tensors["c_attn_weight"].data, tensors["c_proj_weight"].data
        return _weights(self, tensors, "c_attn_weight", "c_proj_weight")

    def train(self, mode=True):
        self._packed.clear()
        return super().train(mode)

    def forward(self, x, normed=None, keep=None):
        """`normed`: LayerNorm(x) with this block's weights, if the caller already has it (the
        first block of FusedGPT gets it from the embedding kernel).  `keep`: a `dropout_mask`, used
        if it is for this module's dropout and these sizes."""
        p = self.dropout_prob if self.training else 0.0
        if keep is not None and not (p > 0.0 and keep.serves(x, max(x.numel(), x.shape[1] ** 2), p)):
            keep = None
        prm = _tensors(self, self._NAMES)
        w_attn, w_proj = self._weights(prm)
        in_gemm = normed is None and p == 0.0 and _ln_in_gemm(x, w_attn)
        if _as_block(x, keep) and x.shape[-1] // self.num_heads in HEAD_SIZES:
            return attention_block(x, prm["layer_norm_weight"], prm["layer_norm_bias"], w_attn,
                                   prm["c_attn_bias"], w_proj, prm["c_proj_bias"], self.num_heads,
                                   dropout_prob=p, normed=normed, layer_norm_in_gemm=in_gemm,
                                   keep=keep)
        skip = x
        y = normed
        if in_gemm:
            q, k, v = layer_norm_matmul_and_split_qkv(x, prm["layer_norm_weight"].data,
                                                      prm["layer_norm_bias"].data, w_attn,
                                                      prm["c_attn_bias"].data, self.num_heads)
        else:
            if y is None:
                y = fused_layer_norm(x, prm["layer_norm_weight"].data, prm["layer_norm_bias"].data)
            q, k, v = matmul_and_split_qkv(y, w_attn, prm["c_attn_bias"].data, self.num_heads)
        # [B, N, L, d] values in a [B, L, N, d] buffer: the head merge below copies nothing
        y = flash_attention_v1(q, k, v, dropout_prob=p, merged_heads_layout=True)
        y = y.transpose(1, 2).contiguous().view(skip.shape)
        return fused_ffn(y, w_proj, bias=prm["c_proj_bias"].data, residual=skip, add_gelu=False,
                         dropout_prob=p)

    def get_fwd_flops(self, num_tokens):
        h = self.hidden_size
        return (_norm_flops(num_tokens, h) + _linear_flops(num_tokens, h, 3 * h) +
                _linear_flops(num_tokens, h, h))


class FusedMLP(nn.Module):
    """Pre-LN feed-forward block: x + ffn2(gelu(ffn1(LN(x)))), inner width 4h."""

    def __init__(self, hidden_size, dropout_prob=0.0):
        super().__init__()
        self.hidden_size = hidden_size
        self.intermediate_size = 4 * hidden_size
        self.dropout_prob = dropout_prob
        h, mid = hidden_size, self.intermediate_size
        self.layer_norm_weight = nn.Parameter(torch.ones((h,)))
        self.layer_norm_bias = nn.Parameter(torch.zeros((h,)))
        self.ffn1_weight = nn.Parameter(torch.rand(h, mid))
        self.ffn1_bias = nn.Parameter(torch.rand(mid))
        self.ffn2_weight = nn.Parameter(torch.rand(mid, h))
        self.ffn2_bias = nn.Parameter(torch.rand(h))
        self._packed = _PackedWeights()

    _NAMES = frozenset(("layer_norm_weight", "layer_norm_bias", "ffn1_weight", "ffn1_bias",
                        "ffn2_weight", "ffn2_bias"))

    def _weights(self, tensors):
        return _weights(self, tensors, "ffn1_weight", "ffn2_weight")

    def train(self, mode=True):
        self._packed.clear()
        return super().train(mode)

    def forward(self, x, keep=None):
        """`keep`: as in FusedAttention.forward."""
        p = self.dropout_prob if self.training else 0.0
        prm = _tensors(self, self._NAMES)
        w1, w2 = self._weights(prm)
        # the weights, and x with them, may have other widths than h and 4h (pruned, exchanged)
        width, inner = w1.shape
        if keep is not None and not (
                p > 0.0 and keep.serves(x, x.numel() // width * max(inner, width), p)):
            keep = None
        as_block = inner % 64 == 0
        in_gemm = as_block and p == 0.0 and _ln_in_gemm(x, w1)
        if in_gemm:
            return layer_norm_ffn(x, prm["layer_norm_weight"], prm["layer_norm_bias"], w1,
                                  bias=prm["ffn1_bias"], add_gelu=True, then=(w2, prm["ffn2_bias"]))
        if as_block and _as_block(x, keep):
            return mlp_block(x, prm["layer_norm_weight"], prm["layer_norm_bias"], w1,
                             prm["ffn1_bias"], w2, prm["ffn2_bias"], dropout_prob=p, layer_norm_in_gemm=in_gemm,
                             keep=keep)
        y = fused_layer_norm(x, prm["layer_norm_weight"].data, prm["layer_norm_bias"].data)
        y = fused_ffn(y, w1, bias=prm["ffn1_bias"].data, residual=None, add_gelu=True,
                      dropout_prob=p)
        return fused_ffn(y, w2, bias=prm["ffn2_bias"].data, residual=x, add_gelu=False,
                         dropout_prob=p)

    def get_fwd_flops(self, num_tokens):
        h, mid = self.hidden_size, self.intermediate_size
        return (_norm_flops(num_tokens, h) + _linear_flops(num_tokens, h, mid) +
                _linear_flops(num_tokens, mid, h))


_TAKE_MASK = (_Block.forward, FusedAttention.forward, FusedMLP.forward)


# What a forward through the modules would run: where a program has put something else in its place, or
# hooks on it, that is what runs (_stack).
def _parts():
    return (_Block.forward, FusedAttention.forward, FusedMLP.forward, FusedAttention._weights, FusedMLP._weights,
            _Block.__call__, FusedAttention.__call__, FusedMLP.__call__, _Block._call_impl,
            FusedAttention._call_impl, FusedMLP._call_impl, _tensors, _weights, attention_block, mlp_block,
            layer_norm_ffn)


_OWN = _parts()
_GLOBAL_HOOKS = tuple(getattr(nn.modules.module, name) for name in (
    "_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
    "_global_backward_pre_hooks"))


def _untouched(module, kind):
    own = module.__dict__
    return (type(module) is kind and not own["training"] and "forward" not in own and "_weights" not in own and
            "_call_impl" not in own and "_wrapped_call_impl" not in own and
            not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or
                 own["_backward_pre_hooks"]) and module._compiled_call_impl is None)


class _Layers:
    """What the layers that go to the library together have in common: the sizes, type and device of the
    first one, under x.  `pointers` gives a block's 12 device addresses for `block_layers`, or None where a
    module or a parameter is not what this file makes it, or has another size: the modules are called one
    by one from that block on.  Weight images that are not held (a first forward, a weight edited in
    place) are built there as the modules build them."""

    def __init__(self, block, x):
        attention, mlp = block
        h = x.shape[-1]
        self.h, self.heads, self.inner = h, attention.num_heads, mlp.ffn1_weight.shape[-1]
        self.dtype, self.index = x.dtype, x.get_device()
        self.alive = []  # the images, until they are launched
        self.built = 0  # blocks whose images were built
        row, wide, inner = torch.Size((h,)), torch.Size((3 * h,)), torch.Size((self.inner,))
        self.vectors = ((("layer_norm_weight", row), ("layer_norm_bias", row), ("c_attn_bias", wide),
                         ("c_proj_bias", row)),
                        (("layer_norm_weight", row), ("layer_norm_bias", row), ("ffn1_bias", inner),
                         ("ffn2_bias", row)))
        self.weights = ((("c_attn_weight", (h, 3 * h)), ("c_proj_weight", (h, h))),
                        (("ffn1_weight", (h, self.inner)), ("ffn2_weight", (self.inner, h))))

    def pointers(self, block):
        if not _untouched(block, _Block) or len(block._modules) != 2:
            return None
        attention, mlp = block._modules.values()
        if (not _untouched(attention, FusedAttention) or not _untouched(mlp, FusedMLP) or
                attention.num_heads != self.heads or attention.hidden_size != self.h):
            return None
        first = self._half(attention._parameters, attention._packed, 0)
        second = first and self._half(mlp._parameters, mlp._packed, 1)
        return second and first + second

    def _half(self, own, packed, which):
        dtype, index, kind, found = self.dtype, self.index, nn.Parameter, []
        for name, shape in self.vectors[which]:
            t = own.get(name)
            if (type(t) is not kind or t.dtype is not dtype or t.get_device() != index or t.shape != shape or
                    not t.is_contiguous()):
                return None
            found.append(t.data_ptr())
        images = []
        for name, shape in self.weights[which]:
            t = own.get(name)
            if type(t) is not kind or t.get_device() != index:
                return None
            image = packed.held(name, t)  # of these values, in this type and shape
            if image is None:
                if t.dtype is not dtype or t.shape != shape or not t.is_contiguous():
                    return None
            elif type(image) is not PackedWeight or image.dtype is not dtype or image.shape != shape:
                return None
            images.append(image)
        if None in images:  # both weights are fit to be packed: what the module would do now
            self.built += 1
            images = [image or packed.get(name, own[name]) for image, (name, _) in
                      zip(images, self.weights[which])]
        self.alive += images
        norm_w, norm_b, first, second = found
        return [norm_w, norm_b, images[0].data.data_ptr(), first, images[1].data.data_ptr(), second]


def _stack(blocks, x):
    """(the `_Layers` of an eval-mode forward, the first block's addresses) where its blocks, or the first
    of them, can go to the library together; None where the first block or an operator is not what this
    file makes it, or a size is not the block calls'."""
    h = x.shape[-1]
    if (_parts() != _OWN or any(_GLOBAL_HOOKS) or torch._C._get_tracing_state() is not None or not _as_block(x) or
            not _untouched(blocks[0], _Block) or len(blocks[0]._modules) != 2):
        return None
    attention, mlp = blocks[0]
    if type(attention) is not FusedAttention or type(mlp) is not FusedMLP:
        return None
    heads, inner = attention.num_heads, mlp._parameters.get("ffn1_weight")
    if (h % heads != 0 or h // heads not in HEAD_SIZES or inner is None or inner.dim() != 2 or
            inner.shape[1] % 64 != 0):
        return None
    layers = _Layers(blocks[0], x)
    first = layers.pointers(blocks[0])
    return None if first is None else (layers, first)


def _through(stack, blocks, x, normed):
    """(x behind the blocks that went to the library together, the blocks that are left).  Every block is
    looked over on every forward, 8 to 10 us of host work each, so they go in calls of 1, 3, 9, ... layers: the
    GPU works on those launched while the next are looked over.  Where the host sets the pace in any case, up
    to some 170 rows of 768, each call counts (5 us): 2, 10, 50, ... layers.  Microseconds of a forward that is
    waited for / of one among others, modules called one by one, all blocks looked over before one call, and
    this: 1 x 24 tokens 124M 566 / 488, 438 / 315, 420 / 307 (in calls of 1, 3, 8 407 / 315); 2 x 128 630 / 549,
    609 / 429, 520 / 400 (2, 10: 547 / 402); 7 x 211 712 / 654, 864 / 687, 716 / 655; 2 x 300 tokens of the 48-layer
    model 4114 / 4064, 4824 / 4279, 4130 / 4074.  A weight of the last layer edited in place before each
    forward of 2 x 64: 560, 680, 440."""
    layers, found = stack
    in_gemm, workspace = _ln_in_gemm(x, layers.alive[0]), blocks_workspace(x, layers.heads, layers.inner)
    sent, seen, built = 0, 1, 0
    size, growth = (2, 5) if x.numel() <= 1 << 17 else (1, 3)
    while True:
        more = found
        while more is not None and seen < min(sent + size, len(blocks)):
            more = layers.pointers(blocks[seen])
            if more is not None:
                found += more
                seen += 1
        if seen == len(blocks) and not layers.built:
            return blocks_forward(x, found, layers.heads, layers.inner, normed=normed,
                                  layer_norm_in_gemm=in_gemm, workspace=workspace), []
        if found:
            # in place behind the first call, whose x is the caller's
            x = block_layers(x, found, layers.heads, layers.inner, normed=normed, layer_norm_in_gemm=in_gemm,
                             out=x if sent else None, workspace=workspace)
        if more is None or seen == len(blocks):
            return x, blocks[seen:]
        # packing two weights takes the host as long as a layer takes the GPU
        normed, sent, size, found = None, seen, 1 if layers.built > built else growth * size, []
        built = layers.built


@dataclass
class GPTConfig:
    vocab_size: int = 50304
    block_size: int = 512
    n_layer: int = 12
    n_head: int = 12
    n_embd: int = 768
    dropout: float = 0.1


class FusedGPT(nn.Module):
    """Token + position embeddings, n_layer x (FusedAttention, FusedMLP), final LayerNorm.
    forward(x) returns the final hidden state [B, L, n_embd], like the reference."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        h = config.n_embd
        self.wte_weight = nn.Parameter(torch.rand(config.vocab_size, h))
        self.wpe_weight = nn.Parameter(torch.rand(config.block_size, h))
        self.blocks = nn.ModuleList([
            _Block(FusedAttention(h, config.n_head, dropout_prob=config.dropout),
                   FusedMLP(h, dropout_prob=config.dropout))
            for _ in range(config.n_layer)
        ])
        self.layer_norm_weight = nn.Parameter(torch.ones((h,)))
        self.layer_norm_bias = nn.Parameter(torch.zeros((h,)))
        self._packed = _PackedWeights()

    def train(self, mode=True):
        self._packed.clear()
        return super().train(mode)

    def _lm_head_weight(self):
        # In eval mode the LM head multiplies with a packed image of wte whose vocabulary is
        # zero-padded to a multiple of 64 (GPT-2's 50257 -> 50304): the logits' rows are then
        # whole 128-byte lines and the product runs on the persistent GEMM kernel, and the image
        # is built once instead of on every call; see kernels.pack_lm_head.
        w = self.wte_weight
        if self.training or not isinstance(w, nn.Parameter):
            return w.data
        return self._packed.get("lm_head", w, pack_lm_head)

    def forward(self, x, return_logits=False):
        # causal by construction; no attention or padding mask is taken
        p = self.config.dropout if self.training else 0.0
        blocks = list(self.blocks)
        if p == 0.0 and blocks:
            # eval mode: the first block's LayerNorm comes out of the embedding kernel.  The two
            # modules of blocks[0] are called one by one, so forward hooks registered on that
            # nn.Sequential container itself do not fire (hooks on its two modules do).
            first = blocks[0]
            x, y = fused_embeddings_layer_norm(x, self.wte_weight.data, self.wpe_weight.data,
                                               first[0].layer_norm_weight.data,
                                               first[0].layer_norm_bias.data)
            stack = _stack(blocks, x)
            if stack is not None:
                x, rest = _through(stack, blocks, x, y)
            else:
                x = first[1](first[0](x, normed=y))
                rest = blocks[1:]
        else:
            x = fused_embeddings(x, self.wte_weight.data, self.wpe_weight.data, dropout_prob=p)
            rest = blocks
        keep = _keep_mask(x, self.config.n_embd, len(rest), self.config.n_head, p) if p > 0.0 else None
        for block in rest:
            x = block(x) if keep is None else _call_with_mask(block, x, keep)
        x = fused_layer_norm(x, self.layer_norm_weight.data, self.layer_norm_bias.data)
        if return_logits:
            return x, lm_head(x, self._lm_head_weight())
        return x

    def get_fwd_flops(self, num_tokens):
        cfg = self.config
        # the embedding lookups are counted as if they were matmuls (gpt.py:182-196)
        lookups = num_tokens * cfg.n_embd * 2 * (cfg.vocab_size + cfg.block_size)
        body = sum(m.get_fwd_flops(num_tokens) for blk in self.blocks for m in blk)
        return body + _norm_flops(num_tokens, cfg.n_embd) + lookups

    @torch.no_grad()
    def init_synthetic_(self, seed=1337, std=0.02):
        """Benchmark initialisation: matrices N(0, std), biases 0, LayerNorm (1, 0).  The
        constructors' U[0,1) values overflow fp16 within a layer."""
        gen = torch.Generator(device="cpu").manual_seed(seed)
        for name, prm in self.named_parameters():
            if "layer_norm_weight" in name:
                prm.fill_(1.0)
            elif name.endswith("_bias"):
                prm.zero_()
            else:
                prm.copy_(torch.randn(prm.shape, generator=gen, dtype=torch.float32) * std)
        return self


_MASK_BUFFER = re.compile(r"h\.\d+\.attn\.(bias|masked_bias)")  # HF's causal-mask buffers


def convert_huggingface_to_triton(hf_sd, hf_config):
    """Renames a HuggingFace GPT2Model state dict to FusedGPT's keys.  HF's Conv1D weights are
    already [in, out], so no tensor is transposed; the causal-mask buffers are dropped."""
    n_pos = getattr(hf_config, "n_ctx", None) or hf_config.n_positions
    config = GPTConfig(vocab_size=hf_config.vocab_size, block_size=n_pos,
                       n_layer=hf_config.n_layer, n_head=hf_config.n_head,
                       n_embd=hf_config.n_embd, dropout=0.1)
    rename = {"wte.weight": "wte_weight", "wpe.weight": "wpe_weight",
              "ln_f.weight": "layer_norm_weight", "ln_f.bias": "layer_norm_bias"}
    per_layer = {
        "ln_1.weight": "0.layer_norm_weight", "ln_1.bias": "0.layer_norm_bias",
        "attn.c_attn.weight": "0.c_attn_weight", "attn.c_attn.bias": "0.c_attn_bias",
        "attn.c_proj.weight": "0.c_proj_weight", "attn.c_proj.bias": "0.c_proj_bias",
        "ln_2.weight": "1.layer_norm_weight", "ln_2.bias": "1.layer_norm_bias",
        "mlp.c_fc.weight": "1.ffn1_weight", "mlp.c_fc.bias": "1.ffn1_bias",
        "mlp.c_proj.weight": "1.ffn2_weight", "mlp.c_proj.bias": "1.ffn2_bias",
    }
    for i in range(config.n_layer):
        for src, dst in per_layer.items():
            rename[f"h.{i}.{src}"] = f"blocks.{i}.{dst}"
    sd = {}
    for key, tensor in hf_sd.items():
        if _MASK_BUFFER.fullmatch(key):
            continue
        sd[rename[key]] = tensor
    return sd, config


def convert_hf_and_load_model(model_id, device):
    """Loads HF GPT-2 weights (a hub name, or a local directory when offline) into a FusedGPT;
    returns (model, hf_model), both in eval mode on `device`."""
    from transformers import GPT2Model

    hf_model = GPT2Model.from_pretrained(model_id)
    state_dict, config = convert_huggingface_to_triton(hf_model.state_dict(), hf_model.config)
    model = FusedGPT(config)
    model.load_state_dict(state_dict)
    return model.to(device).eval(), hf_model.to(device).eval()


class GraphedForward:
    """The forward of an eval-mode FusedGPT for one input shape, captured once into a HIP graph
    and replayed per call: the 51 to 63 launches of a small forward become one graph launch and their host work
    goes (2 x 64 tokens, 124M, a pass that is waited for: 499 -> 374 us; among others 350 and 359).  Nothing in the
    library allocates or synchronises, and a captured forward has the bits of an eager one; of sequences of up to
    32 tokens with up to 32 heads in all it records two launches where an eager forward, which waits for the
    host, makes one.  The operators' output tensors come from the graph's private pool.  The result of a call is overwritten by the next call --
    clone it to keep it.  No counterpart in the reference (Triton launches kernel by kernel)."""

    def __init__(self, model, example_ids, return_logits=False, warmup=3):
        assert not model.training, "capture an eval-mode model (weights are packed once)"
        self.ids = example_ids.clone()
        side = torch.cuda.Stream(device=example_ids.device)
        side.wait_stream(torch.cuda.current_stream(example_ids.device))
        with torch.cuda.stream(side):
            for _ in range(warmup):  # packs the weights, sets kernel attributes, fills the pools
                model(self.ids, return_logits=return_logits)
        torch.cuda.current_stream(example_ids.device).wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = model(self.ids, return_logits=return_logits)

    @torch.no_grad()
    def __call__(self, ids):
        assert ids.shape == self.ids.shape and ids.dtype == self.ids.dtype
        self.ids.copy_(ids)
        self.graph.replay()
        return self.out


def estimate_days(flops, mfu=0.45, gpu="h100", num_gpus=1):
    assert gpu in GPU_TO_FLOPS
    return flops / (mfu * GPU_TO_FLOPS[gpu] * 3600 * 24 * num_gpus)


def get_num_parameters(model):
    return sum(p.numel() for p in model.parameters())


def compute_mfu(flops_per_second, gpu="h100"):
    assert gpu in GPU_TO_FLOPS
    return flops_per_second / GPU_TO_FLOPS[gpu]
