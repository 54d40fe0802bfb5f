"""Operator layer: the five public functions of the reference's kernels.py, with the same
names, argument order, defaults, assertions and return shapes, each handing raw device
pointers to one entry point of libgptmi.so (include/gptmi.h).

    fused_embeddings(x, wte, wpe, dropout_prob=0.0)              kernels.py:75-101
    fused_layer_norm(x, weight, bias)                            kernels.py:148-164
    fused_ffn(x, weight, bias=None, residual=None,
              add_gelu=False, dropout_prob=0.0)                  kernels.py:260-315
    matmul_and_split_qkv(x, weight, bias, num_heads)             kernels.py:347-367
    flash_attention_v1(q, k, v, dropout_prob=0.0)                kernels.py:477-525

plus `fused_embeddings_layer_norm` (the embedding gather and the first block's LayerNorm in one
kernel, the fusion the reference's author notes as a TODO, kernels.py:132-133), `fused_softmax(x)` (the reference only sketches a row softmax, kernels.py:318-342),
`lm_head(x, wte)` (the transposed-weight product the reference leaves as a TODO,
gpt.py:159-161) and `pack_weight(weight)`: the GEMM reads its weight as an fp16,
K-contiguous image, which `fused_ffn` / `matmul_and_split_qkv` otherwise rebuild on every call
where the kernels cannot read the weight in place (fp16, K a multiple of 64); a `PackedWeight` may be passed wherever they take `weight`.  Tensors must live on the
GPU: there is no CPU path.  dropout_prob > 0 reproduces the reference's masks: Philox-4x32-10
(Triton's tl.rand) with the kernels' default seed 1337 and the reference's offsets -- the column
for the embedding, the flat index m*N + n for fused_ffn, query*Lk + key for the attention
weights (kernels.py:31-34, 65-70, 245-251, 457-460).
"""
import array
import math
import os

import torch

from . import _lib

_DTYPES = {torch.float32: _lib.GPTMI_F32, torch.float16: _lib.GPTMI_F16}


def _dtype_code(t, what):
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError(f"{what}: dtype {t.dtype} is not supported (float32 and float16 are)")


def _on_gpu(first, *rest):
    """Index of the GPU that all the tensors (None allowed behind the first) are on."""
    index = first.get_device()  # -1 on the CPU
    if index < 0:
        raise RuntimeError("gpt_triton_amd operators run on the GPU only; got a tensor on "
                           f"{first.device} (there is no CPU fallback)")
    for t in rest:
        if t is not None and t.get_device() != index:
            raise RuntimeError(f"tensors on different devices: {first.device} and {t.device}")
    return index


def _call(index, what, fn, *args):
    """One entry point of the library on torch's current stream of GPU `index`.  A forward of a few
    tokens is bound by the host: no device guard where the GPU is the current one already, the raw
    stream from torch's own binding instead of a torch.cuda.Stream object."""
    if index == torch._C._cuda_getDevice():
        rc = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    else:
        with torch.cuda.device(index):
            rc = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    if rc != 0:
        _lib.check(rc, what)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _workspace(nbytes, like):
    return like.new_empty(nbytes, dtype=torch.uint8) if nbytes else None


class PackedWeight:
    """The fp16 [N][round_up(K, 64)] image of a [K, N] weight (see gptmi_pack_weight).  `shape`
    and `dtype` are those of the weight it was made from, so it can stand in for it."""

    __slots__ = ("data", "shape", "dtype", "device", "vocab")

    def __init__(self, data, shape, dtype, vocab=None):
        self.data, self.shape, self.dtype, self.device = data, tuple(shape), dtype, data.device
        self.vocab = vocab  # pack_lm_head: rows of wte before the zero padding

    def is_contiguous(self):
        return True

    def get_device(self):
        return self.data.get_device()

    def data_ptr(self):
        return self.data.data_ptr()


@torch.no_grad()
def pack_weight(weight):
    """Packs a contiguous [K, N] weight once; the result replaces `weight` in `fused_ffn` and
    `matmul_and_split_qkv` and must be rebuilt when the weight changes."""
    assert weight.dim() == 2 and weight.is_contiguous()
    dev = _on_gpu(weight)
    K_, N = weight.shape
    lib = _lib.load()
    buf = weight.new_empty(lib.gptmi_packed_weight_bytes(N, K_), dtype=torch.uint8)
    _call(dev, "pack_weight", lib.gptmi_pack_weight, weight.data_ptr(), buf.data_ptr(), N, K_,
          _lib.GPTMI_W_KN, _dtype_code(weight, "pack_weight"))
    return PackedWeight(buf, weight.shape, weight.dtype)


@torch.no_grad()
def pack_lm_head(wte):
    """Packs wte [V, H] once for `lm_head`, with the vocabulary padded to a multiple of 64 by zero
    rows.  GPT-2's V = 50257 is odd: rows of a dense [T, V] fp16 matrix then start on 2-byte
    boundaries and every logit is stored on its own.  With the padded image the GEMM writes
    [T, Vp] rows of whole 128-byte lines -- the shape the persistent GEMM kernel takes -- and
    `lm_head` returns the [.., :V] view of it."""
    assert wte.dim() == 2 and wte.is_contiguous()
    dev = _on_gpu(wte)
    V, H = wte.shape
    Vp = -(-V // 64) * 64
    lib = _lib.load()
    buf = wte.new_zeros(lib.gptmi_packed_weight_bytes(Vp, H), dtype=torch.uint8)
    _call(dev, "pack_lm_head", lib.gptmi_pack_weight, wte.data_ptr(), buf.data_ptr(), V, H,
          _lib.GPTMI_W_NK, _dtype_code(wte, "pack_lm_head"))
    return PackedWeight(buf, (H, Vp), wte.dtype, vocab=V)


def check_token_ids(x, vocab_size):
    """Raises IndexError if a token id lies outside [0, vocab_size).  The embedding kernels
    themselves read no memory for such an id and use a zero wte row (the reference reads out of
    bounds); this check costs a device synchronisation, so the operators run it only when the
    environment variable GPTMI_CHECK_IDS is set to 1."""
    lo, hi = int(x.min()), int(x.max())
    if lo < 0 or hi >= vocab_size:
        raise IndexError(f"token ids span [{lo}, {hi}] but the vocabulary has {vocab_size} rows")


def _maybe_check_ids(x, vocab_size):
    if os.environ.get("GPTMI_CHECK_IDS") == "1" and x.numel() > 0:
        check_token_ids(x, vocab_size)


def _wlayout(weight, default):
    return _lib.GPTMI_W_PACKED if isinstance(weight, PackedWeight) else default


def fused_embeddings(x, wte, wpe, dropout_prob=0.0):
    """dropout(wte[x] + wpe[position]) for token ids x [B, L] -> [B, L, H] in wte's dtype."""
    assert wte.shape[1] == wpe.shape[1]
    assert x.is_contiguous()
    assert wte.is_contiguous()
    assert wpe.is_contiguous()
    B, L = x.shape
    V, H = wte.shape
    P = wpe.shape[0]
    if x.dtype != torch.int64:
        raise TypeError(f"fused_embeddings: token ids must be int64, got {x.dtype}")
    if wte.dtype != wpe.dtype:
        raise TypeError("fused_embeddings: wte and wpe must share a dtype")
    dev = _on_gpu(x, wte, wpe)
    _maybe_check_ids(x, V)
    z = wte.new_empty((B, L, H))
    _call(dev, "fused_embeddings", _lib.load().gptmi_embed, x.data_ptr(), wte.data_ptr(),
          wpe.data_ptr(), z.data_ptr(), B, L, V, P, H, float(dropout_prob), 1337,
          _dtype_code(wte, "fused_embeddings"))
    return z


def fused_embeddings_layer_norm(x, wte, wpe, weight, bias):
    """(fused_embeddings(x, wte, wpe), fused_layer_norm(of that, weight, bias)) from one kernel:
    the embedding row is normalised while it is still in registers.  Both results are
    bit-identical to the two separate calls.  No dropout (eval-mode forward)."""
    assert wte.shape[1] == wpe.shape[1]
    assert x.is_contiguous()
    assert wte.is_contiguous()
    assert wpe.is_contiguous()
    assert weight.is_contiguous()
    assert bias.is_contiguous()
    assert weight.shape == bias.shape
    assert wte.shape[1] == weight.shape[0]
    B, L = x.shape
    V, H = wte.shape
    P = wpe.shape[0]
    if x.dtype != torch.int64:
        raise TypeError(f"fused_embeddings_layer_norm: token ids must be int64, got {x.dtype}")
    if not (wte.dtype == wpe.dtype == weight.dtype == bias.dtype):
        raise TypeError("fused_embeddings_layer_norm: wte, wpe, weight and bias must share a dtype")
    dev = _on_gpu(x, wte, wpe, weight, bias)
    _maybe_check_ids(x, V)
    emb = wte.new_empty((B, L, H))
    out = wte.new_empty((B, L, H))
    _call(dev, "fused_embeddings_layer_norm", _lib.load().gptmi_embed_layernorm, x.data_ptr(),
          wte.data_ptr(), wpe.data_ptr(), weight.data_ptr(), bias.data_ptr(), emb.data_ptr(),
          out.data_ptr(), B, L, V, P, H, 1e-5, _dtype_code(wte, "fused_embeddings_layer_norm"))
    return emb, out


def fused_layer_norm(x, weight, bias):
    """LayerNorm over the last dim (eps = 1e-5, biased variance), same shape and dtype as x."""
    assert x.is_contiguous()
    assert weight.is_contiguous()
    assert bias.is_contiguous()
    assert weight.shape == bias.shape
    assert x.shape[-1] == weight.shape[0]
    if not (x.dtype == weight.dtype == bias.dtype):
        raise TypeError("fused_layer_norm: x, weight and bias must share a dtype")
    dev = _on_gpu(x, weight, bias)
    H = x.shape[-1]
    M = x.numel() // H
    z = torch.empty_like(x)
    _call(dev, "fused_layer_norm", _lib.load().gptmi_layernorm, x.data_ptr(), weight.data_ptr(),
          bias.data_ptr(), z.data_ptr(), M, H, 1e-5, _dtype_code(x, "fused_layer_norm"))
    return z


def fused_softmax(x):
    """softmax over the last dim with fp32 statistics, same shape and dtype as x."""
    assert x.is_contiguous()
    dev = _on_gpu(x)
    H = x.shape[-1]
    M = x.numel() // H
    z = torch.empty_like(x)
    _call(dev, "fused_softmax", _lib.load().gptmi_softmax, x.data_ptr(), z.data_ptr(), M, H,
          _dtype_code(x, "fused_softmax"))
    return z


def _linear_workspace(lib, M, N, K, code, wlayout, like):
    """(workspace or None, its bytes).  A packed image under fp16 rows that are whole 128-byte lines
    needs none; that is every product of an eval-mode forward, and not worth a call to be told."""
    if wlayout == _lib.GPTMI_W_PACKED and code == _lib.GPTMI_F16 and K % 64 == 0:
        return None, 0
    nbytes = lib.gptmi_linear_workspace_bytes(M, N, K, code, wlayout)
    return _workspace(nbytes, like), nbytes


def _linear(x, weight, bias, residual, z, gelu, dropout_prob, wlayout, what):
    K, N = x.shape[-1], z.shape[-1]
    M = x.numel() // K
    dtype = x.dtype
    code = _dtype_code(x, what)
    if weight.dtype != dtype:
        raise TypeError(f"{what}: weight is {weight.dtype} but x is {dtype}")
    if bias is not None and bias.dtype != dtype:
        raise TypeError(f"{what}: bias is {bias.dtype} but x is {dtype}")
    if residual is not None and residual.dtype != dtype:
        raise TypeError(f"{what}: residual is {residual.dtype} but x is {dtype}")
    lib = _lib.load()
    ws, ws_bytes = _linear_workspace(lib, M, N, K, code, wlayout, x)
    _call(x.get_device(), what, lib.gptmi_linear, x.data_ptr(), weight.data_ptr(), _ptr(bias),
          _ptr(residual), z.data_ptr(), M, N, K, 1 if gelu else 0, float(dropout_prob), 1337, wlayout,
          _ptr(ws), ws_bytes, code)
    return z


def fused_ffn(x, weight, bias=None, residual=None, add_gelu=False, dropout_prob=0.0):
    """dropout(gelu?(x @ weight + bias)) + residual; weight is [K, N] (in x out)."""
    shape = x.shape
    K = shape[-1]
    N = weight.shape[1]
    _on_gpu(x, weight, bias, residual)
    z = x.new_empty((*shape[:-1], N))

    assert x.is_contiguous()
    assert weight.is_contiguous()
    assert K == weight.shape[0]
    if bias is not None:
        assert bias.is_contiguous()
        assert N == bias.shape[0]
    if residual is not None:
        assert residual.numel() == z.numel()
        assert residual.is_contiguous()

    return _linear(x, weight, bias, residual, z, add_gelu, dropout_prob,
                   _wlayout(weight, _lib.GPTMI_W_KN), "fused_ffn")


def lm_head(x, wte):
    """x @ wte^T: logits [*, V].  `wte` is the [V, H] embedding matrix itself (read in place, no
    transposed copy; the result is contiguous) or its `pack_lm_head` image (the result is then
    the [*, :V] view of a buffer whose rows are padded to a multiple of 64 logits)."""
    shape = x.shape
    H = shape[-1]
    assert x.is_contiguous()
    assert wte.is_contiguous()
    _on_gpu(x, wte)
    if isinstance(wte, PackedWeight):
        assert wte.vocab is not None and H == wte.shape[0]
        z = x.new_empty((*shape[:-1], wte.shape[1]))
        _linear(x, wte, None, None, z, False, 0.0, _lib.GPTMI_W_PACKED, "lm_head")
        return z[..., :wte.vocab]
    assert H == wte.shape[1]
    z = x.new_empty((*shape[:-1], wte.shape[0]))
    return _linear(x, wte, None, None, z, False, 0.0, _lib.GPTMI_W_NK, "lm_head")


def matmul_and_split_qkv(x, weight, bias, num_heads):
    """x [B, L, h] @ weight [h, 3h] + bias, returned as q, k, v [B, num_heads, L, h/num_heads],
    each contiguous; the GEMM's store does the head split."""
    batch_size, seqlen, _ = x.shape
    assert x.is_contiguous()
    assert weight.is_contiguous()
    assert x.shape[2] == weight.shape[0]
    hidden_size = weight.shape[1]
    assert hidden_size % 3 == 0, hidden_size
    hidden_size = hidden_size // 3
    assert hidden_size % num_heads == 0, (hidden_size, num_heads)
    head_size = hidden_size // num_heads
    if bias is not None:
        assert bias.is_contiguous()
        assert weight.shape[1] == bias.shape[0]
    dev = _on_gpu(x, weight, bias)
    code = _dtype_code(x, "matmul_and_split_qkv")
    if weight.dtype != x.dtype or (bias is not None and bias.dtype != x.dtype):
        raise TypeError("matmul_and_split_qkv: x, weight and bias must share a dtype")
    if head_size % 8 != 0 and isinstance(weight, PackedWeight):
        raise NotImplementedError("matmul_and_split_qkv: packed weights need head_size % 8 == 0")
    if head_size % 8 != 0:
        # the scatter epilogue stores 8-element groups; other head sizes take the plain GEMM
        y = fused_ffn(x, weight, bias=bias)
        q, k, v = y.split(hidden_size, dim=2)
        return tuple(t.view(batch_size, seqlen, num_heads, head_size).transpose(1, 2).contiguous()
                     for t in (q, k, v))
    shape = (batch_size, num_heads, seqlen, head_size)
    q = x.new_empty(shape)
    k = torch.empty_like(q)
    v = torch.empty_like(q)
    lib = _lib.load()
    M, K, N = batch_size * seqlen, x.shape[2], 3 * hidden_size
    wl = _wlayout(weight, _lib.GPTMI_W_KN)
    ws, ws_bytes = _linear_workspace(lib, M, N, K, code, wl, x)
    _call(dev, "matmul_and_split_qkv", lib.gptmi_linear_qkv, x.data_ptr(), weight.data_ptr(),
          _ptr(bias), q.data_ptr(), k.data_ptr(), v.data_ptr(), batch_size, seqlen, num_heads,
          head_size, K, wl, _ptr(ws), ws_bytes, code)
    return q, k, v


def layer_norm_linear_supported(x, weight):
    """True where `layer_norm_ffn` / `layer_norm_matmul_and_split_qkv` take these operands: fp16,
    a packed weight image, a row width the kernel's LDS panel holds."""
    if not isinstance(weight, PackedWeight) or x.dtype != torch.float16:
        return False
    H = x.shape[-1]
    return bool(_lib.load().gptmi_layernorm_linear_supported(x.numel() // H, H, _lib.GPTMI_F16))


def _check_layer_norm_linear(x, ln_weight, ln_bias, weight, bias, what):
    assert x.is_contiguous() and ln_weight.is_contiguous() and ln_bias.is_contiguous()
    assert ln_weight.shape == ln_bias.shape == (x.shape[-1],)
    assert x.shape[-1] == weight.shape[0]
    if not isinstance(weight, PackedWeight):
        raise NotImplementedError(f"{what}: takes the packed image of the weight (pack_weight)")
    if not (x.dtype == ln_weight.dtype == ln_bias.dtype == weight.dtype == torch.float16):
        raise NotImplementedError(f"{what}: fp16 operands only")
    if bias is not None:
        assert bias.is_contiguous() and bias.shape == (weight.shape[1],)
        if bias.dtype != x.dtype:
            raise TypeError(f"{what}: bias is {bias.dtype} but x is {x.dtype}")
    return _on_gpu(x, ln_weight, ln_bias, weight, bias)


def layer_norm_ffn(x, ln_weight, ln_bias, weight, bias=None, add_gelu=False, then=None):
    """gelu?(fused_layer_norm(x, ln_weight, ln_bias) @ weight + bias) in one launch: the
    LayerNorm runs in the GEMM's operand prologue (the fusion marked as to do in the reference,
    kernels.py:132-133) and gives the bits of fused_layer_norm followed by fused_ffn.  Meant for
    few rows; `weight` is a `pack_weight` image, fp16 only (NotImplementedError otherwise, and
    for row widths `layer_norm_linear_supported` turns down).

    then=(weight2, bias2), with add_gelu and bias: the MLP's second product behind it in the same
    call -- the result is x + that @ weight2 + bias2 (fused_ffn with x as the residual, same bits)."""
    if then is not None:
        assert add_gelu and bias is not None
        return mlp_block(x, ln_weight, ln_bias, weight, bias, *then, layer_norm_in_gemm=True)
    dev = _check_layer_norm_linear(x, ln_weight, ln_bias, weight, bias, "layer_norm_ffn")
    K, N = weight.shape
    M = x.numel() // K
    z = x.new_empty((*x.shape[:-1], N))
    _call(dev, "layer_norm_ffn", _lib.load().gptmi_layernorm_linear, x.data_ptr(),
          ln_weight.data_ptr(), ln_bias.data_ptr(), 1e-5, weight.data_ptr(), _ptr(bias),
          z.data_ptr(), M, N, K, 1 if add_gelu else 0, _lib.GPTMI_F16)
    return z


def layer_norm_matmul_and_split_qkv(x, ln_weight, ln_bias, weight, bias, num_heads):
    """matmul_and_split_qkv(fused_layer_norm(x, ln_weight, ln_bias), weight, bias, num_heads) in
    one launch, same bits; see `layer_norm_ffn`.  x [B, L, h]; head size a multiple of 8."""
    dev = _check_layer_norm_linear(x, ln_weight, ln_bias, weight, bias,
                                   "layer_norm_matmul_and_split_qkv")
    batch_size, seqlen, K = x.shape
    hidden_size = weight.shape[1] // 3
    assert weight.shape[1] == 3 * hidden_size and hidden_size % num_heads == 0
    head_size = hidden_size // num_heads
    shape = (batch_size, num_heads, seqlen, head_size)
    q = x.new_empty(shape)
    k = torch.empty_like(q)
    v = torch.empty_like(q)
    _call(dev, "layer_norm_matmul_and_split_qkv", _lib.load().gptmi_layernorm_linear_qkv,
          x.data_ptr(), ln_weight.data_ptr(), ln_bias.data_ptr(), 1e-5, weight.data_ptr(),
          _ptr(bias), q.data_ptr(), k.data_ptr(), v.data_ptr(), batch_size, seqlen, num_heads,
          head_size, K, _lib.GPTMI_F16)
    return q, k, v


def flash_attention_v1(q, k, v, dropout_prob=0.0, *, merged_heads_layout=False):
    """Causal softmax(q k^T / sqrt(d)) v for q, k, v [B, N, L, d] -> [B, N, L, d].

    merged_heads_layout=True (an extension; the default is the reference's behaviour)
    returns the same values as a [B, N, L, d]-shaped view of a [B, L, N, d] buffer, so the
    caller's `.transpose(1, 2).contiguous()` head merge costs no copy.
    """
    assert q.shape[:2] == k.shape[:2]
    assert q.shape[-1] == k.shape[-1]
    assert k.shape == v.shape
    B, N, Lq, H = q.shape
    Lk = k.shape[2]
    assert H in HEAD_SIZES
    assert q.is_contiguous()
    assert k.is_contiguous()
    assert v.is_contiguous()
    if not (q.dtype == k.dtype == v.dtype):
        raise TypeError("flash_attention_v1: q, k and v must share a dtype")
    dev = _on_gpu(q, k, v)
    code = _dtype_code(q, "flash_attention_v1")
    if merged_heads_layout:
        buf = q.new_empty((B, Lq, N, H))
        layout = _lib.GPTMI_O_BLND
    else:
        buf = torch.empty_like(q)
        layout = _lib.GPTMI_O_BNLD
    _call(dev, "flash_attention_v1", _lib.load().gptmi_flash_attn, q.data_ptr(), k.data_ptr(),
          v.data_ptr(), buf.data_ptr(), B, N, Lq, Lk, H, 1 / math.sqrt(H), float(dropout_prob), 1337,
          layout, code)
    return buf.transpose(1, 2) if merged_heads_layout else buf


class DropoutMask:
    """Bits of the dropout mask that `fused_ffn` (offset m * N + n) and `flash_attention_v1` (offset
    query * Lk + key) draw for probability p: both count flat indices from 0 under one seed, so the
    mask of the largest matrix serves all of them.  `bits` offsets are held."""

    __slots__ = ("data", "bits", "p", "device")

    def __init__(self, data, bits, p):
        self.data, self.bits, self.p, self.device = data, bits, p, data.device

    def serves(self, x, bits, p):
        return self.p == p and bits <= self.bits and self.data.get_device() == x.get_device()


def dropout_mask(bits, p, like):
    """DropoutMask of `bits` offsets (at most 2^32) for 0 < p < 1 on the GPU of `like`."""
    dev = _on_gpu(like)
    lib = _lib.load()
    buf = like.new_empty(lib.gptmi_dropout_mask_bytes(bits), dtype=torch.uint8)
    _call(dev, "dropout_mask", lib.gptmi_dropout_mask, buf.data_ptr(), bits, float(p), 1337)
    return DropoutMask(buf, bits, p)


def _keep_args(keep, x, dropout_prob, what):
    if keep is None:
        return None, 0
    if dropout_prob != keep.p or keep.data.get_device() != x.get_device():
        raise ValueError(f"{what}: the dropout mask is for p = {keep.p} on {keep.device}")
    return keep.data.data_ptr(), keep.bits


# Head sizes of the attention kernels (the reference's set, kernels.py:490).
HEAD_SIZES = frozenset((16, 32, 64, 128, 256))


def block_supported(x, width):
    """True where `attention_block` / `mlp_block` take rows of this width."""
    return width % 64 == 0 and width <= 8192 and x.dtype in _DTYPES


def _block_layout(first, second, what):
    packed = isinstance(first, PackedWeight)
    if packed != isinstance(second, PackedWeight):
        raise TypeError(f"{what}: both weights packed or neither")
    return _lib.GPTMI_W_PACKED if packed else _lib.GPTMI_W_KN


def _in_gemm_code(layer_norm_in_gemm):
    return -1 if layer_norm_in_gemm is None else 1 if layer_norm_in_gemm else 0


def attention_block(x, ln_weight, ln_bias, qkv_weight, qkv_bias, proj_weight, proj_bias, num_heads,
                    dropout_prob=0.0, normed=None, layer_norm_in_gemm=False, keep=None):
    """x + dropout(proj(attention(qkv(LayerNorm(x))))) for x [B, L, h]: the operators of an attention
    block (gpt.py:39-60) behind one call of the library, with their bits in fp16 (fp32: up to the fp16
    rounding of the projection's operands).  `normed`: LayerNorm(x), if the caller has it; layer_norm_in_gemm: as in `layer_norm_matmul_and_split_qkv`
    (False: fp32 blocks of few rows with packed weights all the same; None: in no case); keep: a
    `dropout_mask` for dropout_prob of at least max(x.numel(), L * L) offsets, read instead of
    generating the masks here."""
    B, L, h = x.shape
    dtype = x.dtype
    assert ln_weight.shape[0] == ln_bias.shape[0] == proj_bias.shape[0] == h
    assert qkv_bias.shape[0] == 3 * h
    dev = _on_gpu(x, ln_weight, ln_bias, qkv_weight, qkv_bias, proj_weight, proj_bias, normed)
    assert x.is_contiguous() and (normed is None or normed.is_contiguous() and normed.shape == x.shape)
    assert ln_weight.is_contiguous() and ln_bias.is_contiguous()
    assert qkv_bias.is_contiguous() and proj_bias.is_contiguous()
    assert qkv_weight.is_contiguous() and proj_weight.is_contiguous()
    assert tuple(qkv_weight.shape) == (h, 3 * h) and tuple(proj_weight.shape) == (h, h)
    assert h % num_heads == 0 and h // num_heads in HEAD_SIZES
    if not (dtype == ln_weight.dtype == ln_bias.dtype == qkv_weight.dtype == qkv_bias.dtype ==
            proj_weight.dtype == proj_bias.dtype and (normed is None or normed.dtype == dtype)):
        raise TypeError("attention_block: x and the parameters must share a dtype")
    code = _dtype_code(x, "attention_block")
    layout = _block_layout(qkv_weight, proj_weight, "attention_block")
    d = h // num_heads
    lib = _lib.load()
    nbytes = lib.gptmi_attention_block_workspace_bytes(B, L, num_heads, d, layout)
    ws = _workspace(nbytes, x)
    out = torch.empty_like(x)
    _call(dev, "attention_block", lib.gptmi_attention_block, x.data_ptr(), _ptr(normed),
          ln_weight.data_ptr(), ln_bias.data_ptr(), 1e-5, qkv_weight.data_ptr(), qkv_bias.data_ptr(),
          proj_weight.data_ptr(), proj_bias.data_ptr(), out.data_ptr(), B, L, num_heads, d,
          float(dropout_prob), 1337, *_keep_args(keep, x, dropout_prob, "attention_block"),
          _in_gemm_code(layer_norm_in_gemm), layout, _ptr(ws), nbytes, code)
    return out


def mlp_block(x, ln_weight, ln_bias, weight1, bias1, weight2, bias2, dropout_prob=0.0,
              layer_norm_in_gemm=False, keep=None):
    """x + dropout(W2 . dropout(gelu(W1 . LayerNorm(x)))): the operators of an MLP block
    (gpt.py:91-111) behind one call of the library, with their bits; layer_norm_in_gemm: as in
    `layer_norm_ffn` and `attention_block`; keep: as in `attention_block`, of at least (rows of x) * max(inner, h) offsets."""
    h = x.shape[-1]
    dtype = x.dtype
    inner = weight1.shape[1]
    assert ln_weight.shape[0] == ln_bias.shape[0] == bias2.shape[0] == h and bias1.shape[0] == inner
    dev = _on_gpu(x, ln_weight, ln_bias, weight1, bias1, weight2, bias2)
    assert x.is_contiguous() and ln_weight.is_contiguous() and ln_bias.is_contiguous()
    assert weight1.is_contiguous() and weight2.is_contiguous()
    assert bias1.is_contiguous() and bias2.is_contiguous()
    assert weight1.shape[0] == h and tuple(weight2.shape) == (inner, h)
    if not (dtype == ln_weight.dtype == ln_bias.dtype == weight1.dtype == bias1.dtype ==
            weight2.dtype == bias2.dtype):
        raise TypeError("mlp_block: x and the parameters must share a dtype")
    code = _dtype_code(x, "mlp_block")
    layout = _block_layout(weight1, weight2, "mlp_block")
    M = x.numel() // h
    lib = _lib.load()
    nbytes = lib.gptmi_mlp_block_workspace_bytes(M, h, inner, layout)
    ws = _workspace(nbytes, x)
    out = torch.empty_like(x)
    _call(dev, "mlp_block", lib.gptmi_mlp_block, x.data_ptr(), ln_weight.data_ptr(),
          ln_bias.data_ptr(), 1e-5, weight1.data_ptr(), bias1.data_ptr(), weight2.data_ptr(),
          bias2.data_ptr(), out.data_ptr(), M, h, inner, float(dropout_prob), 1337,
          *_keep_args(keep, x, dropout_prob, "mlp_block"), _in_gemm_code(layer_norm_in_gemm), layout,
          _ptr(ws), nbytes, code)
    return out


def blocks_workspace(x, num_heads, inner):
    """(scratch that serves `block_layers` for x and these sizes, its bytes)."""
    B, L, h = x.shape
    nbytes = _lib.load().gptmi_blocks_workspace_bytes(B, L, num_heads, h // num_heads, inner,
                                                      _dtype_code(x, "block_layers"))
    return _workspace(nbytes, x), nbytes


def block_layers(x, pointers, num_heads, inner, normed=None, layer_norm_in_gemm=False, out=None, workspace=None):
    """`attention_block` then `mlp_block` for each of some layers of a model in one call of the library, packed
    weights, no dropout; same launches, same bits.  pointers: 12 device addresses a layer, as gptmi_blocks
    lists them, of tensors that the caller has checked and keeps (`FusedGPT.forward` does).  out: where the
    result goes, x itself included; workspace: `blocks_workspace`, if the caller has it."""
    B, L, h = x.shape
    dev = _on_gpu(x, normed, out)
    code = _dtype_code(x, "block_layers")
    assert x.is_contiguous() and (normed is None or normed.is_contiguous() and normed.shape == x.shape)
    assert out is None or out.is_contiguous() and out.shape == x.shape and out.dtype == x.dtype
    assert len(pointers) % 12 == 0 and h % num_heads == 0
    ws, nbytes = workspace or blocks_workspace(x, num_heads, inner)
    if out is None:
        out = torch.empty_like(x)
    table = array.array("Q", pointers)
    _call(dev, "block_layers", _lib.load().gptmi_blocks, x.data_ptr(), _ptr(normed), table.buffer_info()[0],
          len(pointers) // 12, 1e-5, out.data_ptr(), B, L, num_heads, h // num_heads, inner,
          _in_gemm_code(layer_norm_in_gemm), _ptr(ws), nbytes, code)
    return out


def blocks_forward(x, pointers, num_heads, inner, normed=None, layer_norm_in_gemm=False, workspace=None):
    """`block_layers` for a model's layers, or for those that are left of them."""
    return block_layers(x, pointers, num_heads, inner, normed=normed, layer_norm_in_gemm=layer_norm_in_gemm,
                        workspace=workspace)
