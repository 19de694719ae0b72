"""What this framework's performance is measured on: calls a program makes through the public entry points.

A case is a dict of plain values with a ``kind``:

``linear``         one quantized layer, ``E8RHTLinear(x)``: trellis (``bits`` 2-8; 5-8 = a 4-bit and a residual
                   stream) or E8 shell (``stages`` of 2 bits per weight), one token to prefill
``merged``         separately quantized shards behind one input (fused q/k/v, gate/up),
                   ``MergedTrellisLinear.apply(x)``: the serving layer's call
``experts``        the routed experts of a mixture-of-experts layer, ``torch.ops.glq.fused_moe_trellis_3inst``
``decoder``        one greedy decode step of ``TrellisDecoder`` as its users run it, replayed from its HIP graph
``encode_trellis`` quantizing a weight matrix to a trellis stream, ``ext.trellis_quantize_matrix``
``encode_e8``      nearest codewords of the E8 shell table, ``ext.e8_quantize``

Streams are random bits where every bit pattern is a valid code (trellis) and codes of Gaussian weights where the
codes' distribution matters to the path (E8); activations are N(0, 1); sign vectors are random.
"""
from __future__ import annotations

import math

import torch

from glq_amd import custom_ops, ext, hadamard
from glq_amd.checkpoint import load_shell_table
from glq_amd.decoder import DecoderConfig, TrellisDecoder
from glq_amd.linear_method import MergedTrellisLinear, trellis_rvq_recipe
from glq_amd.quantized_linear import E8RHTLinear

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
MOST_MACS = 4096 * 14336 * 4096          # multiply-adds of the largest listed layer
MOST_ENCODED = 2048 * 2048               # weights of the largest listed encode


def listed():
    return [
        # the k projection of a 2048-wide model at decode, layer by layer: the smallest call there is
        dict(name="trellis_k_proj_1", kind="linear", codebook="trellis", bits=4, rows=512, cols=2048, tokens=1, dtype="bf16"),
        # fused q/k/v of the same model in a serving engine, one sequence
        dict(name="merged_qkv_1", kind="merged", bits=4, cols=2048, shards="2048,512,512", tokens=1, dtype="bf16"),
        # a 2 bpw layer of a small model (960 = 512 + 256 + 128 + 64), a handful of sequences, fp16 activations
        dict(name="e8_960_5", kind="linear", codebook="e8", stages=1, rows=960, cols=960, tokens=5, dtype="f16"),
        # a large 4 bpw E8 layer at decode
        dict(name="e8_14336_1", kind="linear", codebook="e8", stages=2, rows=14336, cols=4096, tokens=1, dtype="bf16"),
        # the down projection at 6 bpw with a few dozen sequences in the batch
        dict(name="trellis_6bpw_down_37", kind="linear", codebook="trellis", bits=6, rows=2048, cols=11008, tokens=37,
             dtype="f16"),
        # fused gate/up on a 512-token prompt
        dict(name="merged_gate_up_512", kind="merged", bits=4, cols=2048, shards="11008,11008", tokens=512, dtype="bf16"),
        # a large E8 layer on a prompt that is no multiple of anything
        dict(name="e8_4096_1001", kind="linear", codebook="e8", stages=2, rows=4096, cols=14336, tokens=1001, dtype="bf16"),
        # the largest prefill: 4096 tokens through a 14336 x 4096 layer
        dict(name="trellis_14336_4096", kind="linear", codebook="trellis", bits=4, rows=14336, cols=4096, tokens=4096,
             dtype="bf16"),
        # routed experts (128 of 2048 -> 2 x 768 -> 2048, eight per token) with a batch of sequences
        dict(name="experts_16", kind="experts", bits=4, experts=128, hidden=2048, inter=768, top_k=8, tokens=16, dtype="bf16"),
        # greedy decoding at 512 cached positions: eight layers and the output head of the 3B shape
        dict(name="decoder_step_512", kind="decoder", layers=8, context=512, max_len=1024),
        # quantizing: one matrix to 4 bpw trellis, the vectors of one matrix to E8 codewords
        dict(name="encode_trellis_2048", kind="encode_trellis", bits=4, rows=2048, cols=2048),
        dict(name="encode_e8_2048", kind="encode_e8", vectors=2048 * 2048 // 8),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _multiple(rng, lo, hi, of):
    return max(lo, int(_log(rng, lo, hi)) // of * of)


def _tokens(rng, most_tokens, macs_per_token):
    return max(1, min(most_tokens, MOST_MACS // macs_per_token, int(round(_log(rng, 1, most_tokens)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "merged", "experts", "decoder", "encode_trellis", "encode_e8"))
    dtype = rng.choice(("bf16", "f16"))
    if kind == "linear":
        codebook = rng.choice(("trellis", "e8"))
        rows, cols = _multiple(rng, 512, 14336, 32), _multiple(rng, 512, 14336, 64)
        tokens = _tokens(rng, 4096, rows * cols)
        if codebook == "trellis":
            return dict(kind=kind, codebook=codebook, bits=rng.choice((2, 3, 4, 4, 5, 6, 8)), rows=rows, cols=cols,
                        tokens=tokens, dtype=dtype)
        return dict(kind=kind, codebook=codebook, stages=rng.choice((1, 2, 2, 3, 4)), rows=rows, cols=cols, tokens=tokens,
                    dtype=dtype)
    if kind == "merged":
        cols = _multiple(rng, 960, 8192, 64)
        if rng.random() < 0.5:                                  # grouped-query attention: q and two narrower shards
            kv = max(64, cols // rng.choice((2, 4, 8)) // 64 * 64)
            shards = [cols, kv, kv]
        else:
            shards = [_multiple(rng, 2 * cols, 4 * cols, 64)] * 2
        return dict(kind=kind, bits=rng.choice((4, 4, 6)), cols=cols, shards=",".join(str(s) for s in shards),
                    tokens=_tokens(rng, 2048, sum(shards) * cols), dtype=dtype)
    if kind == "experts":
        experts, top_k = rng.choice((16, 32, 64, 128)), rng.choice((2, 4, 8))
        return dict(kind=kind, bits=rng.choice((4, 4, 6)), experts=experts, hidden=_multiple(rng, 1024, 4096, 64),
                    inter=_multiple(rng, 512, 2048, 64), top_k=top_k, tokens=int(round(_log(rng, 1, 1024))), dtype=dtype)
    if kind == "decoder":
        max_len = rng.choice((1024, 2048, 4096))
        return dict(kind=kind, layers=rng.randint(2, 8), context=int(_log(rng, 8, max_len - 8)), max_len=max_len)
    if kind == "encode_trellis":
        rows = _multiple(rng, 256, 4096, 32)
        cols = min(_multiple(rng, 256, 4096, 64), MOST_ENCODED // rows // 64 * 64)
        return dict(kind=kind, bits=rng.choice((2, 3, 4, 4)), rows=rows, cols=cols)
    return dict(kind=kind, vectors=int(_log(rng, 960, MOST_ENCODED // 8)))


# ---- inputs ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _bits(g, *shape):
    return torch.randint(-32768, 32768, shape, generator=g, device=DEV, dtype=torch.int16)


def _signs(g, n):
    return (torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1).to(torch.float16)


def _acts(g, case, tokens, width):
    return torch.randn(tokens, width, generator=g, device=DEV).to(DTYPES[case["dtype"]])


_TABLE = []


def _table():
    """The shell table, one tensor per process: layers share it."""
    if not _TABLE:
        _TABLE.append(load_shell_table().to(DEV))
    return _TABLE[0]


def _trellis_layer(g, rows, cols, bits):
    with torch.device(DEV):
        lin = E8RHTLinear(cols, rows, codebook_type="trellis")
    tiles, recipe = (rows // 16) * (cols // 16), trellis_rvq_recipe(bits)
    lin.trellis_packed = _bits(g, tiles, 16 * recipe[0])
    if len(recipe) > 1:
        lin.trellis_packed2 = _bits(g, tiles, 16 * recipe[1])
        lin.inv_resid_scale2 = torch.tensor(0.25, device=DEV)
    lin.SU, lin.SV = _signs(g, rows), _signs(g, cols)
    lin.Wscale = torch.tensor(0.9 / math.sqrt(cols), device=DEV)
    return lin


def _e8_layer(g, rows, cols, stages):
    table = _table()
    with torch.device(DEV):
        lin = E8RHTLinear(cols, rows, block_diagonal=True)
    # codes of Gaussian weights: the first stage of N(0, 1), the residual stages of what is left over
    v = torch.randn(16384, 8, generator=g, device=DEV)
    for s, name in enumerate(("Qidxs", "Qidxs2", "Qidxs3", "Qidxs4")[:stages]):
        dec, idx = ext.e8_quantize(v, table)
        pick = torch.randint(0, v.shape[0], (rows, cols // 8), generator=g, device=DEV)
        setattr(lin, name, torch.where(idx > 32767, idx - 65536, idx).to(torch.int16)[pick])
        v = (v - dec) * 3.0
        if s:
            setattr(lin, ("inv_resid_scale", "inv_resid_scale2", "inv_resid_scale3")[s - 1],
                    torch.tensor(3.0 ** -s, device=DEV))
    lin.SU, lin.SV = _signs(g, rows), _signs(g, cols)
    lin.Wscale = torch.tensor(0.9 / math.sqrt(cols), device=DEV)
    lin.set_codebook(table, table)
    return lin


def _experts(g, case):
    E, hid, inter, recipe = case["experts"], case["hidden"], case["inter"], trellis_rvq_recipe(case["bits"])

    def proj(m, n):
        tiles = (m // 16) * (n // 16)
        second = len(recipe) > 1
        return [_bits(g, E, tiles, 16 * recipe[0]),
                _bits(g, E, tiles, 16 * recipe[1]) if second else torch.zeros(E, 1, 1, dtype=torch.int16, device=DEV),
                _signs(g, E * m).view(E, m), _signs(g, n), torch.full((E,), 0.9 / math.sqrt(n), device=DEV),
                torch.full((E,), 0.25 if second else 0.0, device=DEV)]

    def meta(n):
        b = hadamard.block_decompose(n)
        return torch.tensor(b), hadamard.pack_block_meta(b).to(DEV)
    (bn13, bn13m), (bm13, bm13m), (bn2, bn2m), (bm2, bm2m) = meta(hid), meta(2 * inter), meta(inter), meta(hid)
    args = proj(2 * inter, hid) + proj(hid, inter) + [hid, inter, 2 * inter, hid, 2 * inter, inter, hid, bn13, bm13, bn13m,
                                                      bm13m, bn2, bm2, bn2m, bm2m, 0]
    x = _acts(g, case, case["tokens"], hid)
    weights, ids = torch.topk(torch.randn(case["tokens"], E, generator=g, device=DEV).softmax(-1), case["top_k"])
    return x, ids, weights / weights.sum(-1, keepdim=True), args


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        lin = _trellis_layer(g, case["rows"], case["cols"], case["bits"]) if case["codebook"] == "trellis" else \
            _e8_layer(g, case["rows"], case["cols"], case["stages"])
        lin.prepare()                                           # the load-time step
        return kind, lin, _acts(g, case, case["tokens"], case["cols"])
    if kind == "merged":
        lins = [_trellis_layer(g, int(s), case["cols"], case["bits"]) for s in case["shards"].split(",")]
        layer = MergedTrellisLinear.from_linears(lins, bpw=case["bits"]).process_weights_after_loading(DEV)
        return kind, layer, _acts(g, case, case["tokens"], case["cols"])
    if kind == "experts":
        custom_ops.register()
        return kind, _experts(g, case)
    if kind == "decoder":
        dec = TrellisDecoder(DecoderConfig(layers=case["layers"]), device=DEV, seed=seed, max_len=case["max_len"])
        dec.prefill(torch.randint(0, dec.cfg.vocab, (case["context"],), generator=g, device=DEV))
        dec.capture()
        return kind, dec, dec.pos.clone(), dec.tok.clone()
    if kind == "encode_trellis":                                # normalised, transformed weights are close to Gaussian
        return kind, torch.randn(case["rows"], case["cols"], generator=g, device=DEV) * 0.8933837, case["bits"]
    table = _table().float()
    return kind, torch.randn(case["vectors"], 8, generator=g, device=DEV), table, (table * table).sum(-1)


def run(state):
    kind, *held = state
    if kind == "linear":
        lin, x = held
        return lin(x)
    if kind == "merged":
        layer, x = held
        return layer.apply(x)
    if kind == "experts":
        x, ids, weights, args = held[0]
        return torch.ops.glq.fused_moe_trellis_3inst(x, ids, weights, *args)
    if kind == "decoder":
        dec, pos, tok = held
        dec.pos.copy_(pos)                                      # the same step again
        dec.tok.copy_(tok)
        dec.graph.replay()
        return dec.logits, dec.kc, dec.vc
    if kind == "encode_trellis":
        W, bits = held
        return ext.trellis_quantize_matrix(W, bits)
    v, table, norms = held
    return ext.e8_quantize(v, table, norms)


def work(case):
    kind = case["kind"]
    if kind in ("linear", "merged"):
        rows = case["rows"] if kind == "linear" else sum(int(s) for s in case["shards"].split(","))
        cols, tokens = case["cols"], case["tokens"]
        bits = 2 * case["stages"] if case.get("codebook") == "e8" else case["bits"]
        return {"bytes": rows * cols * bits / 8 + 2 * tokens * (rows + cols) + 2 * (rows + cols), "flops": 2.0 * tokens * rows * cols}
    if kind == "experts":
        slots, per = case["tokens"] * case["top_k"], 3 * case["inter"] * case["hidden"]
        used = case["experts"] * (1.0 - (1.0 - case["top_k"] / case["experts"]) ** case["tokens"])   # expected number
        return {"bytes": used * per * case["bits"] / 8 + 4 * case["tokens"] * case["hidden"] + 12 * slots, "flops": 2.0 * slots * per}
    if kind == "decoder":
        c = DecoderConfig()
        layer = c.hidden * (2 * c.heads + 2 * c.kv_heads) * c.head_dim + 3 * c.hidden * c.ffn
        cache = 2 * 2 * case["context"] * c.kv_heads * c.head_dim
        return {"bytes": case["layers"] * (layer * c.bits / 8 + cache) + 2.0 * c.vocab * c.hidden + 4 * c.vocab,
                "flops": 2.0 * (case["layers"] * layer + c.vocab * c.hidden)}
    if kind == "encode_trellis":
        # every one of the 2^16 states is costed (subtract, multiply, add) at every step of both passes
        n = case["rows"] * case["cols"]
        return {"bytes": n * (4 + 4 + case["bits"] / 8), "flops": 2 * 3 * 65536.0 * n}
    # a vector in, its codeword and index out; a lattice point is found in a few operations per coordinate
    return {"bytes": case["vectors"] * (32 + 32 + 8), "flops": 100.0 * case["vectors"]}


def tolerance(case):
    if case["kind"].startswith("encode"):
        return "exact"                                          # indices, bits, and values taken from tables by them
    if case["kind"] == "decoder":
        return {"rel": 2.5e-2}                                  # four bf16 roundings of the residual stream per layer, up to eight layers
    return {"rel": 1e-2}                                        # fp16 / bf16 activations, transforms and results, fp32 sums
