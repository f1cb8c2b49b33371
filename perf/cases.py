"""What a user of this package has it do, as measurable cases: a quantized Linear on its own (the drop-in replacement of
one ``F.linear`` call), a decoder block and the whole model, through the modules that a program calls.

Three kinds of case, each at the sizes of the package's own configurations and over the range around them:

* ``linear``: ``QuantLinear`` (int8) or ``Fp8Linear`` (fp8) called on ``rows`` tokens -- decode batches of 1 to 16 rows,
  speculative or chunked batches of a few dozen, prompts of thousands -- in bf16 or fp32, with and without a bias and
  the residual stream that a block hands over.
* ``block``: one quantized decoder block with its paged KV cache, as a serving program sets it up (all fusions on):
  a step of one new token per sequence, or a prompt, on an empty cache or on top of cached tokens.
* ``model``: the 24-layer model of the generation benchmark with its int8 vocabulary projection: decode steps (all
  sequences at one position, or each at its own as a serving loop batches them) and prompts.

The package is inference only: there is no backward direction.
"""
import math

import torch

from khaosz_amd import AutoRegressiveLM, Fp8Linear, Linear, LMConfig, QuantLinear, fuse_shared_inputs, quantize_model
from khaosz_amd.block import DecoderBlock, PagedKV, rotary_table

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
# hidden, query heads, KV heads, FFN width, tokens per page: the 1B-class block and the generation benchmark's model
SIZES = {2048: (16, 4, 5632, 64), 1536: (24, 4, 6912, 128)}
LAYERS, VOCAB, MAX_LEN = 24, 10000, 2048
PROJECTIONS = {"q_proj", "k_proj", "v_proj", "o_proj", "up", "gate", "down"}


def _linear(name, mode, rows, k, n, dtype="bf16", bias=False, residual=False):
    return dict(name=name, kind="linear", mode=mode, rows=rows, k=k, n=n, dtype=dtype, bias=bias, residual=residual)


def _block(name, hidden, batch, new, cached, qk_norm=False, gate=False):
    return dict(name=name, kind="block", hidden=hidden, batch=batch, new=new, cached=cached, qk_norm=qk_norm, gate=gate)


def _model(name, batch, new, cached, mixed=False):
    return dict(name=name, kind="model", batch=batch, new=new, cached=cached, mixed=mixed)


def listed():
    return [
        # one sequence generating alone: an attention projection of the 1536-wide model on a single token
        _linear("int8_1x1536x1536", "int8", 1, 1536, 1536),
        # a decode batch against an MLP's up projection: the decode configuration at its largest M
        _linear("int8_16x2048x8192", "int8", 16, 2048, 8192),
        # the fp32 configuration: activations that were never cast down, a small batch
        _linear("int8_64x2048x2048_f32", "int8", 64, 2048, 2048, dtype="f32"),
        # a ragged batch of prompt tails through a down projection that ends in the residual stream
        _linear("int8_333x6912x1536_residual", "int8", 333, 6912, 1536, residual=True),
        # the prefill configuration, with its bias
        _linear("int8_4096x2048x2048_bias", "int8", 4096, 2048, 2048, bias=True),
        # the fp8 variant at decode
        _linear("fp8_8x2048x8192", "fp8", 8, 2048, 8192),
        # the fp8 configuration: a down projection over a long prompt
        _linear("fp8_2048x8192x2048", "fp8", 2048, 8192, 2048),
        # the decoder block configuration: 8 sequences, a step in the middle of its 64, and the prompts before it
        _block("block_decode_8_at_543", 2048, 8, 1, 543),
        _block("block_prefill_8x512", 2048, 8, 512, 0),
        # the generation benchmark: a decode step of 4 sequences in the middle of its 128, and the prompts before it
        _model("model_decode_4_at_575", 4, 1, 575),
        _model("model_prefill_4x512", 4, 512, 0),
        # a serving loop's step: 11 sequences, each at a position of its own
        _model("model_decode_11_mixed", 11, 1, 1400, mixed=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_linear(rng):
    mode = rng.choice(("int8", "int8", "fp8"))
    rows = rng.randint(1, 16) if rng.random() < 0.45 else _log(rng, 17, 8192)
    k = 16 * _log(rng, 512 // 16, 8192 // 16)
    n = _log(rng, 512, 11264)
    if rng.random() < 0.75:
        n = -(-n // 16) * 16  # the widths of a model's layers; a vocabulary has any size
    dtype = "f32" if mode == "int8" and rng.random() < 0.2 else "bf16"
    return dict(_linear("", mode, rows, k, n, dtype, rng.random() < 0.3, rng.random() < 0.3))


def _draw_tokens(rng, most_tokens, most_batch):
    """(batch, new tokens of each sequence, tokens cached before them)"""
    if rng.random() < 0.5:
        return rng.randint(1, most_batch), 1, _log(rng, 16, MAX_LEN - 1)
    new = _log(rng, 17, 1024)
    batch = rng.randint(1, max(1, min(most_batch, most_tokens // new)))
    return batch, new, rng.choice((0, 0, _log(rng, 16, MAX_LEN - new)))


def draw(rng):
    kind = rng.choices(("linear", "block", "model"), (7, 2, 3))[0]
    if kind == "linear":
        case = _draw_linear(rng)
    elif kind == "block":
        batch, new, cached = _draw_tokens(rng, 4096, 16)
        option = rng.random()
        case = _block("", rng.choice(sorted(SIZES)), batch, new, cached, qk_norm=option < 0.2, gate=0.2 <= option < 0.35)
    else:
        batch, new, cached = _draw_tokens(rng, 1024, 16)
        case = _model("", batch, new, cached, mixed=new == 1 and rng.random() < 0.5)
    del case["name"]
    return case


# ---- what is in hand before the call -----------------------------------------------------------------------------

def _activations(gen, *shape, dtype):
    """N(0, 1) with one channel in a hundred ten times as large, as trained models have them."""
    x = torch.randn(*shape, generator=gen, device=DEVICE)
    loud = torch.randperm(shape[-1], generator=gen, device=DEVICE)[:max(1, shape[-1] // 100)]
    x[..., loud] *= 10.0
    return x.to(dtype)


def _table(gen, case, page):
    """Every sequence's pages, handed out in the order a pool that has been in use gives them."""
    per_seq = -(-(case["cached"] + case["new"]) // page)
    n = case["batch"] * per_seq
    return torch.randperm(n, generator=gen, device=DEVICE).view(case["batch"], per_seq), n


def _fill(gen, cache):
    """Keys and values of the tokens that earlier calls cached."""
    for t in (cache.k_layers, cache.v_layers):
        t.copy_(torch.randn(t.shape, generator=gen, device=DEVICE, dtype=t.dtype))


def _prepare_linear(case, gen):
    dtype = DTYPES[case["dtype"]]
    base = Linear(case["k"], case["n"], bias=case["bias"]).to(DEVICE)
    with torch.no_grad():
        base.weight.copy_(torch.randn(base.weight.shape, generator=gen, device=DEVICE) * 0.02)
        if case["bias"]:
            base.bias.copy_(torch.randn(case["n"], generator=gen, device=DEVICE) * 0.01)
    base = base.to(dtype)
    layer = (QuantLinear if case["mode"] == "int8" else Fp8Linear).from_linear(base)
    x = _activations(gen, case["rows"], case["k"], dtype=dtype)
    residual = torch.randn(case["rows"], case["n"], generator=gen, device=DEVICE).to(dtype) if case["residual"] else None
    return {"kind": "linear", "layer": layer, "x": x, "residual": residual}


def _prepare_block(case, gen):
    hidden = case["hidden"]
    heads, kv_heads, ffn, page = SIZES[hidden]
    with torch.device(DEVICE):
        block = DecoderBlock(hidden, heads, ffn, kv_heads, use_qk_norm=case["qk_norm"], use_gated_attention=case["gate"])
    block.reset_parameters()
    block.to(torch.bfloat16).eval()
    quantize_model(block)
    fuse_shared_inputs(block, norms=True, decode_attention=True, residuals=True)
    table, pages = _table(gen, case, page)
    cache = PagedKV(pages, page, kv_heads, hidden // heads, DEVICE, torch.bfloat16)
    _fill(gen, cache)
    freqs = rotary_table(hidden // heads, MAX_LEN, device=DEVICE)[case["cached"]:case["cached"] + case["new"]]
    return {"kind": "block", "block": block, "cache": cache, "table": table, "total": case["cached"] + case["new"],
            "freqs": freqs.unsqueeze(0).expand(case["batch"], -1, -1),
            "x": _activations(gen, case["batch"], case["new"], hidden, dtype=torch.bfloat16)}


def _prepare_model(case, gen):
    heads, kv_heads, ffn, page = SIZES[1536]
    config = LMConfig(vocab_size=VOCAB, dim=1536, n_layers=LAYERS, n_heads=heads, n_kv_heads=kv_heads, dim_ffn=ffn,
                      max_len=MAX_LEN)
    with torch.device(DEVICE):
        model = AutoRegressiveLM(config)
    model.to(torch.bfloat16).eval()
    quantize_model(model, target_modules=PROJECTIONS | {"lm_head"})
    fuse_shared_inputs(model, norms=True, decode_attention=True, residuals=True)
    table, pages = _table(gen, case, page)
    cache = model.new_cache(pages, page)
    _fill(gen, cache)
    ids = torch.randint(0, VOCAB, (case["batch"], case["new"]), generator=gen, device=DEVICE)
    positions = None
    if case["mixed"]:
        positions = torch.randint(0, case["cached"] + 1, (case["batch"], 1), generator=gen, device=DEVICE)
        positions[0] = case["cached"]
    return {"kind": "model", "model": model, "cache": cache, "table": table, "ids": ids, "positions": positions,
            "start": case["cached"], "total": case["cached"] + case["new"]}


def prepare(case, seed):
    torch.manual_seed(seed)  # the modules' own initialisation
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    with torch.no_grad():
        return {"linear": _prepare_linear, "block": _prepare_block, "model": _prepare_model}[case["kind"]](case, gen)


# ---- the call ------------------------------------------------------------------------------------------------------

def run(state):
    with torch.inference_mode():
        if state["kind"] == "linear":
            if state["residual"] is None:
                return state["layer"](state["x"])
            return state["layer"](state["x"], residual=state["residual"])
        cache = state["cache"].bind(state["table"], state["total"])
        if state["kind"] == "block":
            y = state["block"](state["x"], state["freqs"], None, cache)
            return {"y": y, "keys": cache.k_layers, "values": cache.v_layers}
        if state["positions"] is None:
            out = state["model"](state["ids"], paged_cache=cache, start_pos=state["start"])
        else:
            out = state["model"](state["ids"], paged_cache=cache, position_ids=state["positions"])
        return {"logits": out["logits"], "hidden": out["hidden_states"], "keys": cache.k_layers, "values": cache.v_layers}


# ---- what it cannot do without -----------------------------------------------------------------------------------

def _linear_work(rows, k, n):
    return n * k, 2.0 * rows * n * k  # weight bytes, operations


def _block_work(case, hidden):
    heads, kv_heads, ffn, _ = SIZES[hidden]
    batch, new, cached = case["batch"], case["new"], case["cached"]
    rows, kv = batch * new, kv_heads * (hidden // heads)
    shapes = [(hidden, hidden + 2 * kv), (hidden, hidden), (hidden, 2 * ffn), (ffn, hidden)]
    if case.get("gate"):
        shapes.append((hidden, hidden))
    work = [_linear_work(rows, k, n) for k, n in shapes]
    seen = batch * (new * cached + new * (new + 1) / 2)  # (query, position) pairs
    if case.get("mixed"):
        seen *= 0.5  # positions are spread evenly up to the longest
    cache = 2 * 2 * kv * (batch * cached * (0.5 if case.get("mixed") else 1.0) + rows)  # earlier tokens read, new ones written
    return sum(w for w, _ in work) + cache, sum(f for _, f in work) + 4.0 * heads * (hidden // heads) * seen


def work(case):
    if case["kind"] == "linear":
        rows, k, n = case["rows"], case["k"], case["n"]
        size = 2 if case["dtype"] == "bf16" else 4
        weight, flops = _linear_work(rows, k, n)
        scales = 4 * n if case["mode"] == "int8" else 4
        extra = (size * n if case["bias"] else 0) + (size * rows * n if case["residual"] else 0)
        return {"bytes": weight + scales + size * rows * (k + n) + extra, "flops": flops}
    rows = case["batch"] * case["new"]
    if case["kind"] == "block":
        nbytes, flops = _block_work(case, case["hidden"])
        return {"bytes": nbytes + 2 * 2 * rows * case["hidden"], "flops": flops}
    nbytes, flops = _block_work(case, 1536)
    weight, head = _linear_work(rows, 1536, VOCAB)
    return {"bytes": LAYERS * nbytes + weight + 2 * rows * (2 * 1536 + VOCAB), "flops": LAYERS * flops + head}


def tolerance(case):
    if case["kind"] == "linear":
        # int8 codes and sums are whole numbers and the scaling is three rounded fp32 operations: one result.
        # fp8 sums in fp32, the order left open, and rounds to bf16.
        return "exact" if case["mode"] == "int8" else {"rel": 5e-3, "max": 0.02}
    # bf16 activations: a rounding that falls the other way moves an int8 code of the next projection by one, and the
    # model does that through 24 layers.  Both return keys and values too.
    return {"rel": 1e-2 if case["kind"] == "block" else 2e-2, "max": 0.5}
