"""Performance cases of the framework: what a training or inference program has it do, through
the public entry points of `slapo_amd.op`, with the sizes such a program would bring.

A case is a dict of plain values.  `listed()` returns the standing ones, `draw(rng)` one more of
the same ranges.  `prepare(case, seed)` makes what the program has in hand before the call
(tensors, modules with their weights), `run(state)` makes one pass and returns everything the pass
computes, `work(case)` counts the bytes and operations the pass cannot do without, and
`tolerance(case)` bounds the relative difference between two correct implementations.

Kinds of case
  attention   `FlashAttentionOp` on [batch, seq, heads, head_dim] tensors, forward only or forward
              and backward; optional causal mask, local window, padding mask and dropout
  epilogue    the bias epilogues that follow the projections of an MLP or attention block
  loss        `ParallelCrossEntropy` on the logits of a language model
  layer       one transformer layer assembled from the modules, with the vendor's matrix products
"""
import math

import torch
import torch.nn.functional as F
from torch import nn

from slapo_amd import op

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}


def listed():
    return [
        # a short sentence through an encoder at inference: latency of one call
        _attention("attn_infer_short", "fp16", batch=1, seq=128, heads=12, head_dim=64,
                   mask="padding", train=False),
        # one generation step: a single query per sequence against the keys so far
        _attention("attn_infer_step", "bf16", batch=8, seq=1, seq_k=2000, heads=16, head_dim=128,
                   train=False),
        # the benchmark's workload: a decoder's causal attention in training
        _attention("attn_train_1k", "fp16", batch=8, seq=1024, heads=16, head_dim=64, causal=True),
        # a larger decoder, sequences padded to a common length, head_dim that is no power of two
        _attention("attn_train_padded", "bf16", batch=4, seq=2048, heads=32, head_dim=80,
                   causal=True, mask="padding"),
        # a local-attention layer with attention dropout
        _attention("attn_train_window", "bf16", batch=4, seq=2048, heads=16, head_dim=128,
                   causal=True, window=256, p=0.1),
        # an encoder's training batch of odd length, padded, with attention dropout
        _attention("attn_train_ragged", "bf16", batch=3, seq=777, heads=12, head_dim=64,
                   mask="padding", p=0.1),
        # long-context training, one sequence
        _attention("attn_train_long", "bf16", batch=1, seq=16384, heads=16, head_dim=128,
                   causal=True),
        # an encoder kept in single precision, forward
        _attention("attn_infer_fp32", "fp32", batch=4, seq=512, heads=16, head_dim=64,
                   train=False),
        # the activation between the two projections of an MLP in training
        _epilogue("gelu_train", "bf16", "bias_gelu", rows=8192, cols=4096),
        # bias, dropout, residual and normalisation after a projection, a small ragged batch
        _epilogue("norm_train_ragged", "fp16", "layer_norm", rows=1537, cols=768, p=0.1),
        # the loss of a language model with an unpadded vocabulary
        _loss("loss_train", "fp16", tokens=8192, vocab=50257),
        # a whole decoder layer in training with its usual dropout
        _layer("layer_train", "fp16", "decoder", batch=8, seq=1024, hidden=1024, head_dim=64,
               p=0.1),
    ]


def draw(rng):
    kind = rng.choices(["attention", "epilogue", "loss", "layer"], [6, 3, 1, 2])[0]
    dtype = rng.choices(["bf16", "fp16", "fp32"], [4, 4, 1])[0]
    if kind == "attention":
        return _draw_attention(rng, dtype)
    if kind == "epilogue":
        which = rng.choice(["bias_gelu", "bias_dropout", "bias_dropout_residual", "layer_norm"])
        cols = rng.choice([768, 1024, 2048, 2560, 4096, _spread(rng, 96, 8192)])
        rows = min(_size(rng, 32, 32768), (1 << 25) // cols)
        p = 0.0 if which == "bias_gelu" else rng.choice([0.0, 0.1, 0.1])
        return _epilogue(None, dtype, which, rows=rows, cols=cols, p=p, train=rng.random() < 0.75)
    if kind == "loss":
        vocab = rng.choice([50257, 50304, _spread(rng, 1000, 65536)])
        return _loss(None, dtype, tokens=min(_size(rng, 32, 8192), (1 << 28) // vocab),
                     vocab=vocab, smoothing=rng.choice([0.0, 0.0, 0.1]),
                     train=rng.random() < 0.75)
    dtype = rng.choice(["bf16", "fp16"])
    hidden, head_dim = rng.choice([(512, 64), (768, 64), (1024, 64), (2048, 128), (2560, 80)])
    seq = _size(rng, 64, 2048)
    batch = max(1, min(_spread(rng, 1, 16), 16384 * 1024 // (seq * hidden)))
    return _layer(None, dtype, rng.choice(["decoder", "encoder", "encoder_fused_qkv"]),
                  batch=batch, seq=seq, hidden=hidden, head_dim=head_dim,
                  p=rng.choice([0.0, 0.1]), train=rng.random() < 0.75)


def _draw_attention(rng, dtype):
    head_dim = rng.choice([64, 64, 64, 128, 128, 80, 96, 32, 72])
    heads, batch = _spread(rng, 2, 40), _spread(rng, 1, 32)
    if rng.random() < 0.15:  # generation steps
        case = dict(batch=batch, seq=1, seq_k=_size(rng, 64, 8192), heads=heads, train=False,
                    mask=rng.choice(["none", "none", "padding"]))
    else:
        seq, train = _size(rng, 32, 8192), rng.random() < 0.7
        causal = rng.random() < 0.6
        window = _spread(rng, 32, max(33, seq)) if causal and rng.random() < 0.2 else 0
        case = dict(batch=batch, seq=seq, heads=heads, causal=causal, window=window, train=train,
                    mask=rng.choices(["none", "padding", "square"], [5, 3, 1])[0],
                    p=rng.choice([0.0, 0.0, 0.1]) if train else 0.0)
    # no dearer than the dearest listed case: fewer sequences, then fewer heads, then shorter ones
    most_flops, most_values = (1.2e10, 1 << 25) if dtype == "fp32" else (1.0e12, 1 << 26)
    while True:
        full = dict(case, seq_k=case.get("seq_k", case["seq"]))
        pairs = full["batch"] * full["heads"] * full["seq"] * full["seq_k"]
        values = full["batch"] * full["heads"] * full["seq_k"] * head_dim
        if pairs * head_dim * 14 <= most_flops and values <= most_values and pairs <= 1 << 32:
            return _attention(None, dtype, head_dim=head_dim, **case)
        which = ("batch" if case["batch"] > 1 else "heads" if case["heads"] > 2
                 else "seq_k" if case["seq"] == 1 else "seq")
        case[which] = max(1, case[which] * 3 // 4)


def _spread(rng, lo, hi):
    """An integer of [lo, hi], evenly over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _size(rng, lo, hi):
    """A length: half of them multiples of 64 (where the range has one), half as they come."""
    n = _spread(rng, lo, hi)
    return max(64, n // 64 * 64) if rng.random() < 0.5 else n


def _named(name, case):
    return case if name is None else dict(name=name, **case)


def _attention(name, dtype, *, batch, seq, heads, head_dim, seq_k=None, causal=False, window=0,
               mask="none", p=0.0, train=True):
    return _named(name, dict(kind="attention", dtype=dtype, batch=batch, seq=seq,
                             seq_k=seq if seq_k is None else seq_k, heads=heads,
                             head_dim=head_dim, causal=causal, window=window, mask=mask, p=p,
                             train=train))


def _epilogue(name, dtype, which, *, rows, cols, p=0.0, train=True):
    return _named(name, dict(kind="epilogue", dtype=dtype, op=which, rows=rows, cols=cols, p=p,
                             train=train))


def _loss(name, dtype, *, tokens, vocab, smoothing=0.0, train=True):
    return _named(name, dict(kind="loss", dtype=dtype, tokens=tokens, vocab=vocab,
                             smoothing=smoothing, train=train))


def _layer(name, dtype, which, *, batch, seq, hidden, head_dim, p=0.0, train=True):
    return _named(name, dict(kind="layer", dtype=dtype, layer=which, batch=batch, seq=seq,
                             hidden=hidden, head_dim=head_dim, p=p, train=train))


# ---- what the program has before the call -------------------------------------------------------
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)

    # dropout draws from the device's default generator; a pass starts it from the step's seed, as
    # a resumed step does
    state = {"kind": case["kind"], "train": case["train"], "seed": seed,
             "generator": torch.cuda.default_generators[torch.cuda.current_device()],
             "random": case.get("p", 0.0) > 0.0}
    if case["kind"] == "attention":
        b, h, d = case["batch"], case["heads"], case["head_dim"]
        q = randn(b, case["seq"], h, d)
        k, v = randn(b, case["seq_k"], h, d), randn(b, case["seq_k"], h, d)
        mask = _mask(case, gen, dtype)
        core = op.FlashAttentionOp("hip_cdna4", case["causal"], window=case["window"] or None)
        state.update(call=lambda q, k, v: core(q, k, v, mask, case["p"]), inputs=[q, k, v],
                     grads=[randn(b, case["seq"], h, d)])
    elif case["kind"] == "epilogue":
        rows, cols, p, train = case["rows"], case["cols"], case["p"], case["train"]
        x, bias = randn(rows, cols), randn(cols)
        if case["op"] == "bias_gelu":
            state.update(call=op.bias_gelu, inputs=[x, bias])
        elif case["op"] == "bias_dropout":
            state.update(call=lambda x, b: op.bias_dropout(x, b, p, True), inputs=[x, bias])
        elif case["op"] == "bias_dropout_residual":
            state.update(call=lambda x, b, r: op.bias_dropout_residual(x, b, r, p, True),
                         inputs=[x, bias, randn(rows, cols)])
        else:
            norm = op.HipBiasDropoutResidualLayerNorm(cols, p, device="cuda", dtype=dtype)
            with torch.no_grad():
                norm.weight.add_(randn(cols) * 0.1)
                norm.bias.add_(randn(cols) * 0.1)
            state.update(call=norm.train(), inputs=[x, bias, randn(rows, cols)],
                         params=list(norm.parameters()))
        state["grads"] = [randn(rows, cols)]
    elif case["kind"] == "loss":
        tokens, vocab = case["tokens"], case["vocab"]
        target = torch.randint(0, vocab, (tokens,), generator=gen, device="cuda")
        smoothing = case["smoothing"]
        if smoothing:
            call = lambda x: op.vocab_parallel_cross_entropy(x, target, smoothing)  # noqa: E731
        else:
            loss = op.ParallelCrossEntropy()
            call = lambda x: loss(x, target)  # noqa: E731
        # gradient of the mean over the tokens, with the loss scale of fp16 training
        scale = (65536.0 if case["dtype"] == "fp16" else 1.0) / tokens
        state.update(call=call, inputs=[randn(tokens, vocab) * 3.0],
                     grads=[torch.full((tokens,), scale, device="cuda")])
    else:
        layer = _Layer(case).to(dtype=dtype).train()
        with torch.no_grad():
            for name, param in layer.named_parameters():
                param.copy_(randn(*param.shape) * 0.02)
                if "norm" in name and name.endswith("weight"):
                    param.add_(1.0)
        shape = (case["batch"], case["seq"], case["hidden"])
        state.update(call=layer, inputs=[randn(*shape)], params=list(layer.parameters()),
                     grads=[randn(*shape)])
    if case["train"]:
        for t in state["inputs"]:
            t.requires_grad_()
    return state


def _lengths(case):
    """Valid lengths of a padded batch, evenly over the upper three quarters of the length."""
    n, b = case["seq_k"], case["batch"]
    return [max(1, round(n * (0.25 + 0.75 * (i + 0.5) / b))) for i in range(b)]


def _mask(case, gen, dtype):
    """Additive masks as models hand them over: the model's dtype, the dtype's lowest value at what
    is padded; [B,1,1,Sk], or with the query dimension written out [B,1,Sq,Sk]."""
    if case["mask"] == "none":
        return None
    lengths = torch.tensor(_lengths(case), device="cuda")
    lengths = lengths[torch.randperm(case["batch"], generator=gen, device="cuda")]
    pad = torch.arange(case["seq_k"], device="cuda")[None, :] >= lengths[:, None]
    mask = torch.zeros(pad.shape, device="cuda", dtype=dtype)
    mask = mask.masked_fill(pad, torch.finfo(dtype).min)[:, None, None, :]
    if case["mask"] == "square":
        mask = mask.expand(-1, -1, case["seq"], -1).contiguous()
    return mask


class _Layer(nn.Module):
    """decoder: normalisation before each half, residuals added by the model.
    encoder: normalisation after each half, in one pass with bias, dropout and residual."""

    def __init__(self, case):
        super().__init__()
        hidden, p = case["hidden"], case["p"]
        heads = hidden // case["head_dim"]
        self.kind, self.p = case["layer"], p
        with torch.device("cuda"):
            if self.kind == "decoder":
                self.norm_1, self.norm_2 = nn.LayerNorm(hidden), nn.LayerNorm(hidden)
                self.attn = op.FlashAttention(hidden, heads, p, p, "hip_cdna4", fused_qkv=True)
                self.mlp = op.FusedMLP(hidden, 4 * hidden, "gelu_new", p)
                return
            if self.kind == "encoder":
                self.attn = op.FlashAttention(hidden, heads, p, 0.0, "hip_cdna4",
                                              output_proj=False)
            else:
                self.qkv = op.FusedQKV(hidden, heads, 1)
                self.core = op.FlashAttentionOp("hip_cdna4", False)
            self.out = nn.Linear(hidden, hidden)
            self.norm_1 = op.HipBiasDropoutResidualLayerNorm(hidden, p)
            self.fc_in = op.LinearWithAct(hidden, 4 * hidden)
            self.fc_out = nn.Linear(4 * hidden, hidden)
            self.norm_2 = op.HipBiasDropoutResidualLayerNorm(hidden, p)

    def forward(self, x):
        if self.kind == "decoder":
            x = x + self.attn(self.norm_1(x))[0]
            return x + self.mlp(self.norm_2(x))
        if self.kind == "encoder":
            context = self.attn(x)[0]
        else:
            context = self.core(*self.qkv(x), None, self.p).flatten(2)
        h = self.norm_1(F.linear(context, self.out.weight), self.out.bias, x)
        return self.norm_2(F.linear(self.fc_in(h), self.fc_out.weight), self.fc_out.bias, h)


# ---- one pass -----------------------------------------------------------------------------------
def run(state):
    if state["random"]:
        state["generator"].manual_seed(state["seed"])
    if not state["train"]:
        with torch.no_grad():
            return state["call"](*state["inputs"])
    wanted = state["inputs"] + state.get("params", [])
    out = state["call"](*state["inputs"])
    return [out, *torch.autograd.grad([out], wanted, state["grads"])]


# ---- what a pass cannot do without --------------------------------------------------------------
def _pairs(case):
    """Attended (query, key) pairs of one head, summed over the batch."""
    sq, sk = case["seq"], case["seq_k"]
    lengths = [sk] * case["batch"] if case["mask"] == "none" else _lengths(case)

    def below(n, reach):  # sum over queries i < n of min(i + 1, reach)
        full = min(n, reach)
        return full * (full + 1) // 2 + (n - full) * reach

    pairs = 0
    for length in lengths:
        if not case["causal"]:
            pairs += sq * length
        elif not case["window"]:
            pairs += below(sq, length)
        else:  # keys j <= i, j > i - window, j < length
            pairs += below(sq, length) - below(max(0, sq - case["window"]), length)
    return pairs


def work(case):
    e, train = SIZE[case["dtype"]], case["train"]
    if case["kind"] == "attention":
        rows_q = case["batch"] * case["seq"] * case["heads"] * case["head_dim"]
        rows_k = case["batch"] * case["seq_k"] * case["heads"] * case["head_dim"]
        values = 2 * rows_q + 2 * rows_k  # q, o; k, v
        if train:
            values += 2 * rows_q + 2 * rows_k  # dO, dQ; dK, dV
        if case["mask"] != "none":
            values += case["batch"] * case["seq_k"] * (case["seq"] if case["mask"] == "square"
                                                       else 1)
        products = 14 if train else 4
        return {"bytes": values * e,
                "flops": products * case["head_dim"] * case["heads"] * _pairs(case)}
    if case["kind"] == "epilogue":
        rows, cols = case["rows"], case["cols"]
        tensors = {"bias_gelu": 2, "bias_dropout": 2}.get(case["op"], 3)
        if train:  # upstream gradient in, input gradient out; the activation needs its input again
            tensors += {"bias_gelu": 3, "bias_dropout": 2, "bias_dropout_residual": 2,
                        "layer_norm": 4}[case["op"]]
        vectors = (3 if case["op"] == "layer_norm" else 1) * (2 if train else 1)
        return {"bytes": (tensors * rows * cols + vectors * cols) * e,
                "flops": 10 * rows * cols * (2 if train else 1)}
    if case["kind"] == "loss":
        values = case["tokens"] * case["vocab"]
        return {"bytes": values * e * (3 if train else 1) + case["tokens"] * (16 if train else 12),
                "flops": values * (6 if train else 3)}
    tokens, hidden = case["batch"] * case["seq"], case["hidden"]
    inner = dict(case, seq_k=case["seq"], causal=case["layer"] == "decoder", window=0, mask="none")
    attended = (14 if train else 4) * hidden * _pairs(inner)
    weights = 12 * hidden * hidden
    return {"bytes": (weights * (2 if train else 1) + tokens * hidden * (4 if train else 2)) * e,
            "flops": 2 * weights * tokens * (3 if train else 1) + attended}


def tolerance(case):
    """Relative 2-norm differences between correct implementations: sums in fp32, operands and
    results rounded to the tensor's type."""
    if case["dtype"] == "fp32":
        return {"rel": 2e-5}
    half = case["dtype"] == "fp16"
    if case["kind"] in ("epilogue", "loss"):
        return {"rel": 1e-3 if half else 6e-3}
    return {"rel": 3e-3 if half else 1.5e-2}
