"""The work that a user of this framework has it do, as cases that can be timed and compared.

A case is one of two kinds:

  "forward"  FusedGPT.forward for a batch of token sequences: the four GPT-2 sizes, fp16 or fp32
             storage, hidden state or logits, in eval mode (eager, or replayed by GraphedForward)
             or in training mode (dropout 0.1);
  "block"    one transformer block wired from the operator functions with the plain [in, out]
             weight matrices, as a program does that keeps its own modules and takes only the
             operators (head sizes 32 to 256).

`listed()` holds the sizes that the benchmark, the configurations and the tests of this
repository name, and ordinary ones between them; `draw` gives more of the same ranges."""
import math

import torch

from gpt_triton_amd import gpt, kernels

VOCAB, CONTEXT = 50257, 1024

# name: layers, heads, width
ARCHS = {
    "124m": (12, 12, 768),
    "medium": (24, 16, 1024),
    "large": (36, 20, 1280),
    "xl": (48, 25, 1600),
}

DTYPES = {"fp16": torch.float16, "fp32": torch.float32}


def _forward(name, arch, batch, seqlen, dtype="fp16", logits=False, graph=False, train=False):
    return {"name": name, "kind": "forward", "arch": arch, "batch": batch, "seqlen": seqlen,
            "dtype": dtype, "logits": logits, "graph": graph, "train": train}


def _block(name, width, heads, batch, seqlen, dtype="fp16"):
    return {"name": name, "kind": "block", "width": width, "heads": heads, "batch": batch,
            "seqlen": seqlen, "dtype": dtype}


def listed():
    return [
        # one short prompt, scored or continued: the smallest call an interactive program makes
        _forward("prompt_1x24_logits", "124m", 1, 24, logits=True),
        # two short sequences, the size of the reference's CPU-runnable case, in both storage types
        _forward("short_2x64", "124m", 2, 64),
        _forward("short_2x64_fp32", "124m", 2, 64, dtype="fp32"),
        # the same from a serving loop of one shape, which captures the forward once
        _forward("short_2x64_graph", "124m", 2, 64, graph=True),
        # a handful of documents of odd length, embedded
        _forward("odd_7x211", "124m", 7, 211),
        # a batch scored for its log-likelihood (evaluation): every logit
        _forward("score_16x300_logits", "124m", 16, 300, logits=True),
        # the fp32 parity path at an ordinary batch
        _forward("batch_32x300_fp32", "124m", 32, 300, dtype="fp32"),
        # the next GPT-2 size, sequences near its context length
        _forward("medium_5x777", "medium", 5, 777),
        # the forward half of a training step: dropout, weights that change from step to step
        _forward("train_16x300", "124m", 16, 300, train=True),
        # a block of a program's own, with wider heads
        _block("block_12x499_d128", 1024, 8, 12, 499),
        # the headline benchmark
        _forward("batch_512x300", "124m", 512, 300),
        # the largest model of the family at its full context
        _forward("xl_64x1024", "xl", 64, 1024),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: sizes spread over the logarithm of the range between the listed ones."""
    if rng.random() < 0.2:
        head = rng.choice([32, 64, 64, 128, 256])
        heads = rng.randint(2, 1536 // head)
        seqlen = _log_int(rng, 16, 1024)
        batch = _log_int(rng, 1, max(2, 65536 // seqlen))
        case = _block("", head * heads, heads, batch, seqlen,
                      dtype="fp32" if rng.random() < 0.25 else "fp16")
    else:
        arch = rng.choice(["124m", "124m", "124m", "medium", "large", "xl"])
        layers, _, width = ARCHS[arch]
        seqlen = _log_int(rng, 8, CONTEXT)
        mode = rng.random()
        train, fp32 = mode < 0.12, 0.12 <= mode < 0.32
        logits = rng.random() < 0.3
        # tokens of a batch: no more work than the listed cases of the same kind have
        most = 1.2e13 / (12 * layers * width * width)
        if train or fp32:
            most /= 8
        if logits:
            most = min(most, 16384)
        batch = _log_int(rng, 1, max(2, int(most / seqlen)))
        graph = not train and batch * seqlen <= 2048 and rng.random() < 0.4
        case = _forward("", arch, batch, seqlen, dtype="fp32" if fp32 else "fp16", logits=logits,
                        graph=graph, train=train)
    del case["name"]
    return case


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, shape, std, dtype, mean=0.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std + mean).to(dtype)


def _prepare_forward(case, seed):
    gen = _generator(seed)
    layers, heads, width = ARCHS[case["arch"]]
    config = gpt.GPTConfig(vocab_size=VOCAB, block_size=CONTEXT, n_layer=layers, n_head=heads,
                           n_embd=width, dropout=0.1)
    default = torch.get_default_dtype()
    torch.set_default_dtype(DTYPES[case["dtype"]])
    try:
        with torch.device("cuda"):
            model = gpt.FusedGPT(config)
    finally:
        torch.set_default_dtype(default)
    # weights as GPT-2 starts from, with LayerNorms and biases that are not the identity
    with torch.no_grad():
        for name, prm in model.named_parameters():
            if name.endswith("layer_norm_weight"):
                prm.normal_(1.0, 0.1, generator=gen)
            else:
                prm.normal_(0.0, 0.02, generator=gen)
    model.train(case["train"])
    # tokens by rank: the frequency of a word piece falls about as one over its rank
    rank = torch.rand((case["batch"], case["seqlen"]), generator=gen, device="cuda")
    ids = torch.exp(rank * math.log(VOCAB)).long().clamp_(max=VOCAB - 1)
    state = {"model": model, "ids": ids, "logits": case["logits"], "graph": None}
    if case["graph"]:
        state["graph"] = gpt.GraphedForward(model, ids, return_logits=case["logits"])
    return state


def _run_forward(state):
    if state["graph"] is not None:
        return state["graph"](state["ids"])
    with torch.no_grad():
        return state["model"](state["ids"], return_logits=state["logits"])


def _prepare_block(case, seed):
    gen, dtype, h = _generator(seed), DTYPES[case["dtype"]], case["width"]
    std = 0.02 * math.sqrt(768 / h)
    state = {"heads": case["heads"],
             "x": _normal(gen, (case["batch"], case["seqlen"], h), 1.0, dtype)}
    for ln in ("ln1", "ln2"):
        state[ln + "_weight"] = _normal(gen, (h,), 0.1, dtype, mean=1.0)
        state[ln + "_bias"] = _normal(gen, (h,), 0.02, dtype)
    for name, fan_in, fan_out in (("qkv", h, 3 * h), ("proj", h, h), ("ffn1", h, 4 * h),
                                  ("ffn2", 4 * h, h)):
        state[name + "_weight"] = _normal(gen, (fan_in, fan_out), std, dtype)
        state[name + "_bias"] = _normal(gen, (fan_out,), 0.02, dtype)
    return state


def _run_block(s):
    x = s["x"]
    y = kernels.fused_layer_norm(x, s["ln1_weight"], s["ln1_bias"])
    q, k, v = kernels.matmul_and_split_qkv(y, s["qkv_weight"], s["qkv_bias"], s["heads"])
    y = kernels.flash_attention_v1(q, k, v)
    y = y.transpose(1, 2).contiguous().view(x.shape)
    x = kernels.fused_ffn(y, s["proj_weight"], bias=s["proj_bias"], residual=x)
    y = kernels.fused_layer_norm(x, s["ln2_weight"], s["ln2_bias"])
    y = kernels.fused_ffn(y, s["ffn1_weight"], bias=s["ffn1_bias"], add_gelu=True)
    return kernels.fused_ffn(y, s["ffn2_weight"], bias=s["ffn2_bias"], residual=x)


def prepare(case, seed):
    """Model and token ids, or a block's input and weights, on the GPU; the captured graph of a
    serving loop."""
    state = (_prepare_forward if case["kind"] == "forward" else _prepare_block)(case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    """One forward pass: the hidden state, or (hidden state, logits), or the block's output."""
    return _run_forward(state) if state["kind"] == "forward" else _run_block(state)


def _attention_flops(batch, width, seqlen):
    return 4 * batch * width * seqlen * (seqlen + 1) // 2


def work(case):
    """Every parameter that takes part and every input read once, every output written once; the
    products of the matrix multiplications and of the causal half of the attention."""
    size = 2 if case["dtype"] == "fp16" else 4
    batch, seqlen = case["batch"], case["seqlen"]
    tokens = batch * seqlen
    layers, width = (1, case["width"]) if case["kind"] == "block" else ARCHS[case["arch"]][::2]
    params = layers * (12 * width * width + 13 * width)
    flops = layers * (24 * tokens * width * width + _attention_flops(batch, width, seqlen))
    values = tokens * width  # the block's input, or the gathered embedding rows
    values += tokens * width  # the output
    if case["kind"] == "forward":
        params += 2 * width + min(seqlen, CONTEXT) * width
        if case["logits"]:
            params += VOCAB * width
            values += tokens * VOCAB
            flops += 2 * tokens * width * VOCAB
    return {"bytes": size * (params + values) + (8 * tokens if case["kind"] == "forward" else 0),
            "flops": flops}


def tolerance(case):
    """About four times how far a pass was from itself with every sum formed in 64 bits at the
    same rounding points.  One block: 1.5e-4 in fp16 storage, 0.2 to 0.4e-4 in fp32 (operands of
    a product are fp16 there too, so a last-bit difference now and then turns a rounding).  Whole
    models: 1.2e-3 (12 layers), 1.5e-3 (24), 2.1e-3 (48) in fp16 and 4.9e-4 (12), 6.3e-4 (48) in
    fp32."""
    fp16 = case["dtype"] == "fp16"
    if case["kind"] == "block":
        return {"rel": 6e-4 if fp16 else 1.8e-4}
    if not fp16:
        return {"rel": 2.5e-3}
    return {"rel": 5e-3 * math.sqrt(ARCHS[case["arch"]][0] / 12)}
