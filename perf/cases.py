"""What this package is timed on: the calls a ranking service or a trainer makes, through the public entry points.

Three kinds of pass ("path" of a case):

  hook     one attention layer that scores: the attention hook with ``layers_to_return_scores``, then the per-document
           scores of its handle.  "drop_in": the scores come from ``compute_auxiliary_attention_loss`` on the labels,
           the way an evaluation script asks for them; otherwise from rows known beforehand, the way a serving loop does.
  forward  what this package does of a ranking forward, start to end: the mask hook and its plan, and for every layer
           the two norms, the rotary embedding, the attention and the gate; of the scoring layer only what the scores
           need.  The projections between them are library GEMMs and are left out: their results are inputs.
  train    one attention layer in training: forward and backward through autograd.  "scored": the layer also returns
           its score logits and the ranking loss trains through them.

A request is a prefix block, "docs" documents of "lo".."hi" tokens and a query block.  The document lengths are the
quantiles of their distribution in an order drawn from the seed, so that every seed is another layout of the same work.
"""
import math
import statistics

import torch

import blockrank_amd as br
from blockrank_amd import synthetic

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
SCORE_LAYER = 20

# (query heads, kv heads, head dim, hidden size, intermediate size)
LARGE = dict(heads=32, kv_heads=8, dim=128, hidden=4096, inter=14336)
GROUPS_OF_7 = dict(heads=28, kv_heads=4, dim=128, hidden=3584, inter=18944)
GROUPS_OF_8 = dict(heads=32, kv_heads=4, dim=128, hidden=4096, inter=11008)
SMALL = dict(heads=8, kv_heads=2, dim=64, hidden=512, inter=1536)
SMALL_GROUPS_OF_7 = dict(heads=14, kv_heads=2, dim=64, hidden=896, inter=4864)
NARROW = dict(heads=32, kv_heads=8, dim=64, hidden=2048, inter=8192)


def _case(path, shape, batch, prefix, docs, lo, hi, query, dtype="bf16", packed=False, tail="uniform", **more):
    c = dict(path=path, batch=batch, prefix=prefix, docs=docs, lo=lo, hi=hi, query=query, tail=tail, dtype=dtype, packed=packed, **shape)
    c.update({"hook": dict(fp8=False, drop_in=False), "forward": dict(layers=8), "train": dict(scored=False)}[path])
    c.update(more)
    return c


def listed():
    return [
        # the smallest call there is: one short request in fp32, every document of one length
        dict(_case("hook", SMALL, 1, 32, 8, 64, 64, 16, dtype="fp32", drop_in=True), name="hook fp32 small"),
        # short ragged passages on a small model in fp16: blocks below one tile, nothing a multiple of anything
        dict(_case("hook", SMALL_GROUPS_OF_7, 2, 37, 7, 9, 61, 21, dtype="fp16"), name="hook fp16 ragged"),
        # one request of 20 passages at the shape of a 7B model: the latency of one user's query
        dict(_case("hook", LARGE, 1, 64, 20, 160, 160, 32, drop_in=True), name="hook one request"),
        # the same as a batch of four: the headline workload of bench.py
        dict(_case("hook", LARGE, 4, 64, 20, 160, 160, 32), name="hook batch of 4"),
        # one request over a long list of documents of very different lengths, padded to the longest
        dict(_case("hook", LARGE, 1, 64, 100, 64, 384, 48), name="hook long list"),
        # heavy-tailed document lengths, seven query heads to a kv head, logits in fp8
        dict(_case("hook", GROUPS_OF_7, 4, 32, 50, 16, 512, 24, tail="lognormal", fp8=True), name="hook fp8 heavy tail"),
        # the largest batch: eight lists of long documents
        dict(_case("hook", LARGE, 8, 64, 50, 384, 512, 48), name="hook long documents"),
        # a whole ranking forward of one request
        dict(_case("forward", LARGE, 1, 64, 20, 96, 224, 32), name="forward one request"),
        # ... and of a batch of eight, packed (no padded slots)
        dict(_case("forward", LARGE, 8, 64, 20, 96, 224, 32, packed=True), name="forward batch of 8 packed"),
        # a training step's attention layer, documents of one length
        dict(_case("train", LARGE, 4, 64, 20, 160, 160, 32), name="train batch of 4"),
        # ... of the layer whose scores the ranking loss trains, ragged documents
        dict(_case("train", LARGE, 2, 61, 12, 33, 250, 45, scored=True), name="train scored ragged"),
        # ... with long documents, packed
        dict(_case("train", LARGE, 2, 64, 16, 256, 512, 64, packed=True), name="train long packed"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["hook", "hook", "forward", "train"])
    most = {"hook": 160_000, "forward": 24_000, "train": 16_000}[path]      # slots of the batch, padding included
    while True:
        lo = _log_int(rng, 8, 400)
        hi = min(512, _log_int(rng, lo, 6 * lo))
        c = dict(batch=_log_int(rng, 1, 16), prefix=rng.randint(16, 96), docs=_log_int(rng, 3, 100), lo=lo, hi=hi, query=rng.randint(16, 64),
                 tail=rng.choice(["uniform", "uniform", "lognormal"]), packed=rng.random() < 0.4)
        slots = c["batch"] * (c["docs"] + 2) * _block_slots(c)
        if 500 <= slots <= most:
            break
    shape = rng.choice([LARGE, LARGE, GROUPS_OF_7, GROUPS_OF_8, NARROW, SMALL, SMALL_GROUPS_OF_7])
    if path == "hook":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"] + (["fp32"] if slots <= 4000 else []))
        fp8 = dtype == "bf16" and shape["dim"] == 128 and rng.random() < 0.2
        return _case(path, shape, dtype=dtype, fp8=fp8, drop_in=not c["packed"] and rng.random() < 0.4, **c)
    if path == "forward":
        return _case(path, shape, layers=rng.randint(6, 10), **c)
    return _case(path, shape, scored=not c["packed"] and rng.random() < 0.4, **c)


# ---- the batch of a case ------------------------------------------------------------------------------------------

def _doc_lengths(c):
    """The case's document lengths of one request, ascending."""
    at = [(i + 0.5) / c["docs"] for i in range(c["docs"])]
    if c["tail"] == "uniform":
        return [int(c["lo"] + (c["hi"] - c["lo"] + 1) * p) for p in at]
    normal = statistics.NormalDist(0.0, 0.6)
    median = max(c["lo"], min(c["hi"], math.sqrt(c["lo"] * c["hi"]) * 1.3))
    return [max(c["lo"], min(c["hi"], round(median * math.exp(normal.inv_cdf(p))))) for p in at]


def _block_slots(c):
    longest = max(c["prefix"], c["query"], max(_doc_lengths(c)))
    return (longest + 15) // 16 * 16


def _layout(c, seed):
    g = torch.Generator().manual_seed(seed)
    docs = _doc_lengths(c)
    rows = [[c["prefix"]] + [docs[i] for i in torch.randperm(len(docs), generator=g).tolist()] + [c["query"]] for _ in range(c["batch"])]
    return synthetic.make_layout(rows)


class _Attention:
    """What the attention hook reads of a decoder layer's attention module."""

    def __init__(self, c, layer_idx, training=False):
        self.layer_idx, self.num_key_value_groups, self.training = layer_idx, c["heads"] // c["kv_heads"], training


def prepare(case, seed):
    c, dev = case, torch.device("cuda:0")
    dtype = DTYPES[c["dtype"]]
    lay = _layout(c, seed)
    g = torch.Generator(device=dev).manual_seed(seed)
    B, S = (1, lay.valid_tokens) if c["packed"] else (lay.B, lay.S)

    def randn(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype).mul_(std)

    def heads(n):
        # a projection of unit-variance hidden states by weights of 0.02, as the head-transposed view the hook is given
        return randn(B, S, n, c["dim"], std=0.02 * math.sqrt(4096)).transpose(1, 2)

    s = dict(case=c, scale=c["dim"] ** -0.5, q=heads(c["heads"]), k=heads(c["kv_heads"]), v=heads(c["kv_heads"]),
             valid=lay.valid.to(dev), labels=lay.labels.to(dev), H=lay.H)
    # the rows that are scored: the completion, which is the last token of the query block, and the token before it
    rows = min(16, lay.H)
    s["rows"] = torch.tensor([[rows - 2, rows - 1]] * lay.B, dtype=torch.int32, device=dev)
    if c["packed"]:
        s["lengths"] = torch.as_tensor(lay.lengths, dtype=torch.int32).to(dev)
    if c["path"] == "forward":
        pos = lay.position_ids.to(dev)
        if c["packed"]:
            pos = pos[s["valid"].view(lay.B, lay.S)][None]
        s["cos"], s["sin"] = synthetic.rope_cos_sin(pos, c["dim"], 1e6, dtype, dev)
        s["x"] = randn(B, S, c["hidden"])
        s["gate"], s["up"] = randn(B, S, c["inter"]), randn(B, S, c["inter"])
        s["norms"] = [1 + randn(c["hidden"], std=0.1) for _ in range(2)]
        s["layers"] = [_Attention(c, i) for i in range(c["layers"])]
        if c["packed"]:
            block = torch.repeat_interleave(torch.arange(lay.B * lay.M), torch.as_tensor(lay.lengths).reshape(-1))
            s["query_tokens"] = ((block % lay.M) == lay.M - 1).nonzero().squeeze(-1).to(dev)
        return s
    # the mask and its plan are made once per forward, by the first layer: the layers after it share them
    s["mask"] = _mask(s)
    s["mask"].plan(c["heads"], c["kv_heads"])
    s["layer"] = _Attention(c, SCORE_LAYER, training=c["path"] == "train")
    if c["path"] == "train":
        for t in ("q", "k", "v"):
            s[t].requires_grad_()
        s["dout"] = randn(B, S, c["heads"], c["dim"])
        s["answers"] = torch.randint(0, c["docs"], (lay.B, 1), generator=g, device=dev)
    return s


def _mask(s):
    if s["case"]["packed"]:
        return br.BlockMask.from_lengths(s["lengths"], H=s["H"], packed=True, dtype=s["q"].dtype)
    return br.blockrank_attention_mask(batch_size=s["valid"].shape[0], attention_mask=s["valid"], dtype=s["q"].dtype)


# ---- one pass -----------------------------------------------------------------------------------------------------

def run(state):
    return {"hook": _hook, "forward": _forward, "train": _train}[state["case"]["path"]](state)


@torch.no_grad()
def _hook(s):
    c = s["case"]
    out, handle = br.blockrank_attention_forward(s["layer"], s["q"], s["k"], s["v"], s["mask"], s["scale"],
                                                 layers_to_return_scores=[SCORE_LAYER], **({"qk_fp8": True} if c["fp8"] else {}))
    if c["drop_in"]:
        scores = br.compute_auxiliary_attention_loss(handle, s["labels"], s["valid"], return_logits=True)
    else:
        scores = handle.doc_scores_window(s["rows"])
    return out, scores


@torch.no_grad()
def _forward(s):
    c, H = s["case"], s["H"]
    cos, sin, (w1, w2) = s["cos"], s["sin"], s["norms"]
    mask = _mask(s)
    outs = []
    for layer in s["layers"]:
        br.rms_norm(s["x"], w1, 1e-5)
        q, k = br.apply_rotary_pos_emb(s["q"], s["k"], cos, sin)
        outs.append(br.blockrank_attention_forward(layer, q, k, s["v"], mask, s["scale"])[0])
        post = br.rms_norm(s["x"], w2, 1e-5)
        gated = br.silu_mul(s["gate"], s["up"])
    # the scoring layer: keys of all tokens, queries of the query block
    normed = br.rms_norm(s["x"], w1, 1e-5)
    k = br.rotate_k(s["k"], cos, sin)
    at = s["rows"] + (H - min(16, H))
    if c["packed"]:
        i = s["query_tokens"]
        q = torch.empty_like(s["q"])
        q[:, :, i] = br.rotate_q(s["q"][:, :, i], cos[:, i], sin[:, i])
        scores = br.doc_scores(q, k, mask, at, s["scale"])
    else:
        q = br.rotate_q(s["q"][:, :, -H:], cos[:, -H:], sin[:, -H:])
        scores = br.doc_scores(q, k, mask, at, s["scale"], query_block_only=True)
    return outs, normed, post, gated, scores


def _train(s):
    qkv = (s["q"], s["k"], s["v"])
    if not s["case"]["scored"]:
        out, _ = br.blockrank_attention_forward(s["layer"], *qkv, s["mask"], s["scale"])
        return (out.detach(), *torch.autograd.grad(out, qkv, s["dout"]))
    out, logits = br.blockrank_attention_forward(s["layer"], *qkv, s["mask"], s["scale"], layers_to_return_scores=[SCORE_LAYER])
    loss, _, scores = br.compute_auxiliary_attention_loss(logits, s["labels"], s["valid"], answer_ids=s["answers"], return_logits=True)
    return (out.detach(), loss.detach(), scores.detach(), *torch.autograd.grad((out, loss), qkv, (s["dout"], torch.ones_like(loss))))


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def work(case):
    c = case
    lay = _layout(c, 0)
    es = 4 if c["dtype"] == "fp32" else 2
    pairs, real = lay.unmasked_pairs(), lay.valid_tokens
    slots = real if c["packed"] else lay.B * lay.S
    Nq, Nkv, D = c["heads"], c["kv_heads"], c["dim"]
    row = D * es
    # q, k and v of the real tokens in, the whole output (zeros in the padded slots) out
    attn_bytes, attn_flops = real * row * (Nq + 2 * Nkv) + slots * row * Nq, 4.0 * D * pairs * Nq
    if c["path"] == "hook":
        return {"bytes": attn_bytes, "flops": attn_flops}
    if c["path"] == "train":
        # the same, the output's gradient in, three gradients out; five products per pair in the backward pass
        return {"bytes": attn_bytes + real * row * Nq + slots * row * (Nq + 2 * Nkv), "flops": 3.5 * attn_flops}
    glue = slots * es * (4 * c["hidden"] + 3 * c["inter"] + 2 * D)
    last = slots * es * 2 * c["hidden"] + real * row * Nkv
    return {"bytes": c["layers"] * (attn_bytes + glue) + last, "flops": c["layers"] * attn_flops}


def tolerance(case):
    # results rounded to the data type after sums in fp32; in fp8 the logits of the documents' rows carry 4 bits
    if case["path"] == "hook" and case["fp8"]:
        return {"rel": 2e-2}
    return {"rel": {"fp32": 1e-5, "fp16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
