"""The work that is timed: what a user of this package has it do, through its public entry points.

Five kinds of work, each over the range of sizes, element types and options it is used with:

  layer      one training step of a `TransformerLayer` (forward, backward, every gradient)
  attention  one training step or one forward pass of the attention core (`ops.attention`)
  decode     one cached decode step of the attention core (`ops.decode_attention`: rotary, cache append, attention)
  loss       the loss side of a training step (`CrossEntropyLoss` on logits, or `TransformerLMHead.loss` on activations)
  generate   greedy completion of a batch of prompts (`TransformerInferenceModule.generate`)
"""

import math
import random

import torch

from scaling_amd import ops
from scaling_amd.config import RotaryConfig, TransformerArchitectureConfig
from scaling_amd.inference import TransformerInferenceModule
from scaling_amd.layer import TransformerLayer, TransformerLayerIO
from scaling_amd.loss import CrossEntropyLoss, TransformerLMHead
from scaling_amd.nn import KVCache, RotaryEmbedding

DEVICE = "cuda"
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def listed():
    return [
        # The smallest layer step: the per-step cost of a unit test, a toy model or a debugging run.  float32 is the
        # default precision of an architecture config.
        layer("layer_tiny_f32", batch=2, seq=128, hidden=256, heads=4, kv_heads=4, inter=688, norm="rms", mlp="swiglu",
              in_one=False, bias=False, dtype="float32"),
        # The default architecture block (LayerNorm, GELU MLP, one QKV projection, biases everywhere) on packed documents
        # of very different lengths, at the size of a small model and an odd sequence length.
        layer("layer_default_packed_bf16", batch=4, seq=1021, hidden=1024, heads=16, kv_heads=16, inter=4096,
              norm="layernorm", mlp="default", in_one=True, bias=True, dtype="bfloat16", doc_min=16, doc_max=600),
        # One layer of an 8B-class decoder in training: the largest piece of work, mostly projections.
        layer("layer_8b_bf16", batch=2, seq=4096, hidden=4096, heads=32, kv_heads=8, inter=14336, norm="rms", mlp="swiglu",
              in_one=False, bias=False, dtype="bfloat16", base=500000),
        # Long-context training: one causal sequence, grouped heads.
        attention("attention_long_bf16", batch=1, seq=8192, heads=32, kv_heads=8, dim=128, dtype="bfloat16"),
        # Training on packed documents with the rotary embedding inside.
        attention("attention_packed_rotary_bf16", batch=1, seq=8192, heads=32, kv_heads=8, dim=128, dtype="bfloat16",
                  doc_min=256, doc_max=2048, rotary=True),
        # float32 training, the default precision.
        attention("attention_f32", batch=1, seq=4096, heads=32, kv_heads=8, dim=128, dtype="float32"),
        # Short ragged documents with narrow heads in float16: fine-tuning on chat turns.
        attention("attention_short_f16", batch=1, seq=3001, heads=12, kv_heads=12, dim=64, dtype="float16",
                  doc_min=17, doc_max=400),
        # One layer's decode attention while serving a full batch of long prompts ...
        decode("decode_batch32", batch=32, heads=32, kv_heads=8, dim=128, dtype="bfloat16", ctx_min=4096, ctx_max=4096),
        # ... and while serving one user.
        decode("decode_single", batch=1, heads=32, kv_heads=8, dim=128, dtype="bfloat16", ctx_min=1500, ctx_max=1500),
        # Loss of a training step on materialised logits of a large vocabulary.
        loss("loss_logits_128k", rows=4096, vocab=128256, hidden=0, dtype="bfloat16"),
        # LM head and loss in one call, with a vocabulary whose rows are not a whole number of 16-byte vectors.
        loss("loss_head_odd_vocab", rows=2047, vocab=50257, hidden=1024, dtype="bfloat16"),
        # Completion of a few prompts by a small model: prefill, then one token at a time.
        generate("generate_small", batch=3, prompt=201, tokens=24, layers=4, hidden=1024, heads=16, kv_heads=4, inter=2816,
                 vocab=32000, dtype="bfloat16"),
    ]


# ---- the kinds and their defaults ----------------------------------------------------------------------------------
def layer(name=None, *, batch, seq, hidden, heads, kv_heads, inter, norm, mlp, in_one, bias, dtype, doc_min=0, doc_max=0,
          base=10000):
    case = dict(kind="layer", batch=batch, seq=seq, hidden=hidden, heads=heads, kv_heads=kv_heads, inter=inter, norm=norm,
                mlp=mlp, in_one=in_one, bias=bias, dtype=dtype, doc_min=doc_min, doc_max=doc_max, base=base)
    return _named(case, name)


def attention(name=None, *, batch, seq, heads, kv_heads, dim, dtype, train=True, causal=True, doc_min=0, doc_max=0,
              rotary=False, dropout=0.0, precise=False):
    case = dict(kind="attention", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, dim=dim, dtype=dtype, train=train,
                causal=causal, doc_min=doc_min, doc_max=doc_max, rotary=rotary, dropout=dropout, precise=precise)
    return _named(case, name)


def decode(name=None, *, batch, heads, kv_heads, dim, dtype, ctx_min, ctx_max):
    return _named(dict(kind="decode", batch=batch, heads=heads, kv_heads=kv_heads, dim=dim, dtype=dtype, ctx_min=ctx_min,
                       ctx_max=ctx_max), name)


def loss(name=None, *, rows, vocab, hidden, dtype):
    """hidden = 0: the loss of given logits; otherwise LM head and loss of given activations."""
    return _named(dict(kind="loss", rows=rows, vocab=vocab, hidden=hidden, dtype=dtype), name)


def generate(name=None, *, batch, prompt, tokens, layers, hidden, heads, kv_heads, inter, vocab, dtype):
    return _named(dict(kind="generate", batch=batch, prompt=prompt, tokens=tokens, layers=layers, hidden=hidden, heads=heads,
                       kv_heads=kv_heads, inter=inter, vocab=vocab, dtype=dtype), name)


def _named(case, name):
    if name is not None:
        case["name"] = name
    return case


# ---- drawn cases ---------------------------------------------------------------------------------------------------
def draw(rng: random.Random):
    kind = rng.choice(("layer", "layer", "attention", "attention", "attention", "decode", "decode", "loss", "loss", "generate"))
    limit = {"layer": 1.0, "attention": 0.5, "decode": 1.0, "loss": 0.5, "generate": 0.25}[kind] * _estimated_seconds(listed()[2])
    while True:
        case = _DRAW[kind](rng)
        if _estimated_seconds(case) <= limit:
            return case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tokens(rng, lo, hi):
    """(batch, seq) with lo .. hi tokens in all, often odd."""
    total = _log_int(rng, lo, hi)
    batch = rng.choice((1, 1, 2, 3, 4, 8))
    return batch, max(16, total // batch)


def _docs(rng, seq):
    """(doc_min, doc_max): packed documents for about half of the cases that are long enough for them."""
    if seq < 64 or rng.random() < 0.5:
        return 0, 0
    hi = _log_int(rng, 48, seq)
    return max(4, hi // rng.choice((4, 16))), hi


def _heads(rng, choices=(1, 2, 4, 8)):
    kv = rng.choice(choices)
    return kv * rng.choice((1, 2, 4)), kv


def _draw_layer(rng):
    dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float16", "float32"))
    dim = rng.choice((64, 64, 128))
    heads, kv = rng.choice(((4, 4), (8, 8), (12, 12), (16, 16), (16, 4), (32, 8)))
    hidden = dim * heads
    swiglu = rng.random() < 0.5
    inter = (hidden * 11 // 4) if swiglu else 4 * hidden
    batch, seq = _tokens(rng, 256, 8192)
    doc_min, doc_max = _docs(rng, seq)
    in_one = heads == kv and rng.random() < 0.7
    return layer(batch=batch, seq=seq, hidden=hidden, heads=heads, kv_heads=kv, inter=inter,
                 norm="rms" if swiglu else "layernorm", mlp="swiglu" if swiglu else "default", in_one=in_one, bias=not swiglu,
                 dtype=dtype, doc_min=doc_min, doc_max=doc_max)


def _draw_attention(rng):
    dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float16", "float32"))
    heads, kv = rng.choice(((4, 4), (8, 2), (12, 12), (16, 16), (16, 2), (32, 8), (32, 32), (32, 1)))
    batch, seq = _tokens(rng, 128, 8192)
    doc_min, doc_max = _docs(rng, seq)
    dim = rng.choice((32, 64, 64, 96, 128, 128, 128))
    rotary = dim in (64, 128) and rng.random() < 0.4
    train = rng.random() < 0.75
    option = rng.choice(("", "", "", "dropout", "precise")) if dtype != "float32" and train else ""
    return attention(batch=batch, seq=seq, heads=heads, kv_heads=kv, dim=dim, dtype=dtype, train=train,
                     causal=rng.random() < 0.85, doc_min=doc_min, doc_max=doc_max, rotary=rotary,
                     dropout=0.1 if option == "dropout" else 0.0, precise=option == "precise")


def _draw_decode(rng):
    heads, kv = rng.choice(((8, 8), (16, 16), (16, 4), (32, 8), (32, 32), (32, 1)))
    ctx_max = _log_int(rng, 64, 16384)
    batch = _log_int(rng, 1, 64)
    return decode(batch=batch, heads=heads, kv_heads=kv, dim=rng.choice((64, 128, 128)),
                  dtype=rng.choice(("bfloat16", "bfloat16", "float16")), ctx_min=rng.choice((1, ctx_max // 2 + 1, ctx_max)),
                  ctx_max=ctx_max)


def _draw_loss(rng):
    hidden = rng.choice((0, 0, 256, 1024, 2048))
    vocab = rng.choice((_log_int(rng, 500, 131072), 32000, 50257, 128256))
    return loss(rows=_log_int(rng, 64, 8192), vocab=vocab, hidden=hidden, dtype=rng.choice(("bfloat16", "bfloat16", "float16", "float32")))


def _draw_generate(rng):
    dim = rng.choice((64, 128))
    heads, kv = rng.choice(((8, 8), (16, 4), (16, 16)))
    hidden = dim * heads
    return generate(batch=_log_int(rng, 1, 16), prompt=_log_int(rng, 5, 600), tokens=rng.randint(2, 24), layers=rng.randint(2, 4),
                    hidden=hidden, heads=heads, kv_heads=kv, inter=hidden * 11 // 4, vocab=rng.choice((1000, 32000, 50257)),
                    dtype=rng.choice(("bfloat16", "bfloat16", "float16")))


_DRAW = {"layer": _draw_layer, "attention": _draw_attention, "decode": _draw_decode, "loss": _draw_loss, "generate": _draw_generate}


def _estimated_seconds(case):
    """Rough upper bound of a pass on one MI355X, used only to keep drawn cases below the largest listed one."""
    w = work(case)
    rate = 40e12 if case["dtype"] == "float32" else 600e12
    return w["bytes"] / 2e12 + w["flops"] / rate


# ---- inputs --------------------------------------------------------------------------------------------------------
def _cumulative(case):
    """Document offsets on the flattened (batch seq) axis: every row of the batch is cut into documents with lengths
    uniform in [doc_min, doc_max] (the whole row is one document when doc_max is 0).  The cuts belong to the case."""
    batch, seq, lo, hi = case["batch"], case["seq"], case["doc_min"], case["doc_max"]
    if hi == 0:
        return [r * seq for r in range(batch + 1)]
    rng = random.Random(f"{batch} {seq} {lo} {hi}")
    cu = [0]
    for r in range(batch):
        end = (r + 1) * seq
        while cu[-1] < end:
            cu.append(min(end, cu[-1] + rng.randint(lo, hi)))
    return cu


def _pairs(case):
    lengths = [b - a for a, b in zip(_cumulative(case)[:-1], _cumulative(case)[1:])]
    if case.get("causal", True):
        return sum(n * (n + 1) // 2 for n in lengths)
    return sum(n * n for n in lengths)


def _positions(cu):
    return torch.cat([torch.arange(b - a) for a, b in zip(cu[:-1], cu[1:])])


class _Source:
    """Seeded values, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * std).to(dtype)

    def integers(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.gen, device=DEVICE)

    def fill_parameters(self, module, std=0.02):
        """Projections N(0, std), norm weights around one, biases small: what a trained module holds."""
        with torch.no_grad():
            for p in module.parameters():
                if p.dim() > 1:
                    p.copy_(self.normal(*p.shape, std=std))
                else:
                    one = 1.0 if bool((p == 1).all()) else 0.0
                    p.copy_(one + self.normal(*p.shape, std=0.05))


def _architecture(case, num_layers, vocab, seq, weight_tying):
    return TransformerArchitectureConfig.from_dict(dict(
        vocab_size=vocab, hidden_size=case["hidden"], num_layers=num_layers, num_attention_heads=case["heads"],
        attention_num_kv_heads=None if case.get("in_one", False) else case["kv_heads"], attention_qkv_in_one=case.get("in_one", False),
        norm_type=case.get("norm", "rms"), mlp_type=case.get("mlp", "swiglu"), mlp_factor=case["inter"] / case["hidden"],
        attention_bias=case.get("bias", False), mlp_bias=case.get("bias", False), precision=case["dtype"], sequence_length=seq,
        rotary_embedding_base=case.get("base", 10000), weight_tying=weight_tying,
        masked_softmax={"kernel": "hip", "softmax_in_fp32": True}))


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _Source(seed), DTYPES[case["dtype"]])


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_layer(case, src, dtype):
    cu = _cumulative(case)
    module = TransformerLayer(_architecture(case, 1, 128, case["seq"], True), layer_index=0, init_method=lambda w: w, device=torch.device(DEVICE))
    src.fill_parameters(module)
    shape = (case["batch"], case["seq"], case["hidden"])
    return dict(kind="layer", module=module, x=src.normal(*shape, dtype=dtype).requires_grad_(), dy=src.normal(*shape, dtype=dtype),
                pos=_positions(cu).view(case["batch"], case["seq"]).to(DEVICE), cu=torch.tensor(cu, dtype=torch.int32, device=DEVICE))


def _run_layer(st):
    module, x = st["module"], st["x"]
    x.grad = None
    for p in module.parameters():
        p.grad = None
    out = module(TransformerLayerIO(activations=x, position_ids=st["pos"], cumulative_seq_lengths=st["cu"])).activations
    out.backward(st["dy"])
    return [out.detach(), x.grad] + [p.grad for p in module.parameters()]


def _prepare_attention(case, src, dtype):
    cu = _cumulative(case)
    tokens = case["batch"] * case["seq"]
    heads, kv, dim = case["heads"], case["kv_heads"], case["dim"]
    st = dict(kind="attention", train=case["train"], causal=case["causal"], dropout=case["dropout"], precise=case["precise"],
              q=src.normal(tokens, heads, dim, dtype=dtype), k=src.normal(tokens, kv, dim, dtype=dtype),
              v=src.normal(tokens, kv, dim, dtype=dtype), cu=torch.tensor(cu, dtype=torch.int32, device=DEVICE), rotary=None)
    if case["train"]:
        st["do"] = src.normal(tokens, heads, dim, dtype=dtype)
        for name in ("q", "k", "v"):
            st[name].requires_grad_()
    if case["rotary"]:
        cos, sin = RotaryEmbedding(RotaryConfig(dimensions=dim, max_seq_length=case["seq"], base=500000), torch.device(DEVICE), dtype).tables()
        pos = _positions(cu).to(DEVICE)
        st["rotary"] = (cos, sin, pos, pos)
    return st


def _run_attention(st):
    q, k, v = st["q"], st["k"], st["v"]
    # the seed is passed, as a program that recomputes activations passes it, so that every pass drops the same probabilities
    args = dict(causal=st["causal"], dropout_p=st["dropout"], dropout_seed=7 if st["dropout"] > 0.0 else None, rotary=st["rotary"],
                precise=st["precise"])
    if not st["train"]:
        with torch.no_grad():
            return ops.attention(q, k, v, st["cu"], **args)
    q.grad = k.grad = v.grad = None
    o = ops.attention(q, k, v, st["cu"], **args)
    o.backward(st["do"])
    return [o.detach(), q.grad, k.grad, v.grad]


def _contexts(case):
    """Context lengths, the token of this step included; they belong to the case."""
    rng = random.Random(f"{case['batch']} {case['ctx_min']} {case['ctx_max']}")
    return [rng.randint(case["ctx_min"], case["ctx_max"]) for _ in range(case["batch"])]


def _prepare_decode(case, src, dtype):
    batch, heads, kv, dim = case["batch"], case["heads"], case["kv_heads"], case["dim"]
    max_ctx = case["ctx_max"] + 64
    cache = KVCache(batch, max_ctx, kv, dim, dtype, torch.device(DEVICE))
    cache.k.copy_(src.normal(batch, max_ctx, kv, dim, dtype=dtype))
    cache.v.copy_(src.normal(batch, max_ctx, kv, dim, dtype=dtype))
    ctx = torch.tensor(_contexts(case), dtype=torch.int32)
    cache.ctx_len.copy_(ctx)
    cache.workspace = ops.decode_workspace(batch, heads, dim, max_ctx, torch.device(DEVICE))
    cos, sin = RotaryEmbedding(RotaryConfig(dimensions=dim, max_seq_length=max_ctx, base=500000), torch.device(DEVICE), dtype).tables()
    # q, k and v of the new token are column slices of one projection output
    qkv = src.normal(batch, heads + 2 * kv, dim, dtype=dtype)
    return dict(kind="decode", cache=cache, q=qkv[:, :heads], k=qkv[:, heads:heads + kv], v=qkv[:, heads + kv:],
                rotary=(cos, sin, (ctx.long() - 1).to(DEVICE)))


def _run_decode(st):
    cache = st["cache"]
    o = ops.decode_attention(st["q"], cache.k, cache.v, cache.ctx_len, st["k"], st["v"], rotary=st["rotary"], workspace=cache.workspace)
    return [o, cache.k, cache.v]


class _Batch:
    def __init__(self, targets, weights):
        self.target_token_ids = targets
        self.loss_weights = weights


def _prepare_loss(case, src, dtype):
    rows, vocab, hidden = case["rows"], case["vocab"], case["hidden"]
    # a tenth of the tokens (prompts, padding) carry no weight
    weights = (src.normal(1, rows) > -1.2816).float()
    batch = _Batch(src.integers(0, vocab, 1, rows), weights)
    if hidden == 0:
        logits = src.normal(1, rows, vocab, dtype=dtype, std=2.0).requires_grad_()
        return dict(kind="loss", fn=CrossEntropyLoss(), x=logits, batch=batch, params=[])
    cfg = TransformerArchitectureConfig.from_dict(dict(
        vocab_size=vocab, hidden_size=hidden, num_layers=1, num_attention_heads=hidden // 64, precision=case["dtype"],
        masked_softmax={"kernel": "hip", "softmax_in_fp32": True}))
    head = TransformerLMHead(cfg, init_method=lambda w: w, device=torch.device(DEVICE))
    src.fill_parameters(head, std=2.0 / math.sqrt(hidden))
    return dict(kind="loss", fn=head.loss, x=src.normal(1, rows, hidden, dtype=dtype).requires_grad_(), batch=batch,
                params=list(head.parameters()))


def _run_loss(st):
    x = st["x"]
    x.grad = None
    for p in st["params"]:
        p.grad = None
    value, metrics = st["fn"](TransformerLayerIO(activations=x, position_ids=None), st["batch"])
    value.backward()
    return [value.detach(), metrics["accuracy"], x.grad] + [p.grad for p in st["params"]]


def _prepare_generate(case, src, dtype):
    cfg = _architecture(case, case["layers"], case["vocab"], case["prompt"] + case["tokens"], True)
    model = TransformerInferenceModule(cfg, device=DEVICE)
    src.fill_parameters(model)
    # tied embeddings of unit scale: the model is sure of its next token, as a trained one is, so that the greedy choice
    # does not hang on the last bit of a logit
    with torch.no_grad():
        model._layers[0].embedding.weight.mul_(50.0)
    # token 0 would end a document
    return dict(kind="generate", model=model, ids=src.integers(1, case["vocab"], case["batch"], case["prompt"]), tokens=case["tokens"])


def _run_generate(st):
    completions, logits = st["model"].generate(st["tokens"], st["ids"])
    return [torch.tensor(completions), logits]


_PREPARE = {"layer": _prepare_layer, "attention": _prepare_attention, "decode": _prepare_decode, "loss": _prepare_loss,
            "generate": _prepare_generate}
_RUN = {"layer": _run_layer, "attention": _run_attention, "decode": _run_decode, "loss": _run_loss, "generate": _run_generate}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    kind, e = case["kind"], DTYPES[case["dtype"]].itemsize
    if kind == "layer":
        tokens, weights = case["batch"] * case["seq"], _layer_weights(case)
        dim = case["hidden"] // case["heads"]
        return {"bytes": e * (4 * tokens * case["hidden"] + 2 * weights),
                "flops": 6 * tokens * weights + 14 * dim * case["heads"] * _pairs(case)}
    if kind == "attention":
        tokens, q, kv = case["batch"] * case["seq"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        passes = (4, 4) if case["train"] else (2, 2)     # q, o (do, dq); k, v (dk, dv)
        return {"bytes": e * tokens * (passes[0] * q + passes[1] * kv),
                "flops": (14 if case["train"] else 4) * case["dim"] * case["heads"] * _pairs(case)}
    if kind == "decode":
        keys, q, kv = sum(_contexts(case)), case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        return {"bytes": e * (2 * keys * kv + case["batch"] * (2 * q + 2 * kv)), "flops": 4 * keys * q}
    if kind == "loss":
        rows, vocab, hidden = case["rows"], case["vocab"], case["hidden"]
        if hidden == 0:
            return {"bytes": 2 * e * rows * vocab, "flops": 8 * rows * vocab}
        return {"bytes": e * 2 * (rows * hidden + vocab * hidden), "flops": 6 * rows * vocab * hidden}
    # generate: the prefill takes every prompt token through the weights, a decode step reads the weights and the cache
    batch, prompt, tokens, hidden, layers = case["batch"], case["prompt"], case["tokens"], case["hidden"], case["layers"]
    weights, head = layers * _layer_weights(case), case["vocab"] * hidden
    dim = hidden // case["heads"]
    keys = sum(prompt + i for i in range(tokens))
    kv_bytes = 2 * layers * batch * case["kv_heads"] * dim
    attn = 4 * dim * case["heads"] * layers * batch
    return {"bytes": e * (tokens * (weights + head) + kv_bytes * keys + tokens * batch * case["vocab"]),
            "flops": 2 * batch * ((prompt + tokens - 1) * weights + tokens * head) + attn * (prompt * (prompt + 1) // 2 + keys - prompt)}


def _layer_weights(case):
    hidden, kv = case["hidden"], case["hidden"] // case["heads"] * case["kv_heads"]
    matrices = 3 if case.get("mlp", "swiglu") == "swiglu" else 2
    return 2 * hidden * hidden + 2 * hidden * kv + matrices * hidden * case["inter"]


# ---- how far two correct implementations may be apart --------------------------------------------------------------
def tolerance(case):
    """About four times the largest relative error that the work shows against the same inputs at higher precision:

      bfloat16   layer 2.5e-3 .. 1.05e-2 (float32 modules), where twice is stated: two implementations round at the same
                 places but one; attention 2.1e-3 .. 3.5e-3, decode 2.7e-3 (64 bits); loss 1.0e-3 .. 1.8e-3 (64 bits);
                 generate 5.9e-3 (float32 modules)
      float16    layer 5.3e-4, attention 4.5e-4, loss 9.9e-4; an eighth of the bfloat16 figures
      float32    layer 9.9e-7, attention 2.5e-6, loss 2.0e-6 (64 bits)
    """
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    if case["dtype"] == "float16":
        return {"rel": 4e-3 if case["kind"] in ("loss", "generate") else 2.5e-3}
    return {"rel": {"layer": 2e-2, "attention": 1.2e-2, "decode": 1e-2, "loss": 7e-3, "generate": 2e-2}[case["kind"]]}
