"""The work this package is used for, as timed cases: its packed low-bit operators called from a user's own model code,
and whole decoders prefilled and decoded through the generation loops.

Operators (``kind``)
    linear   one packed projection, ternary (``bits`` 2) or sign weights (``bits`` 1); with ``x`` = "int8" the caller holds
             quantised activations, otherwise it holds bf16 / fp16 ones and quantises them first
    grouped  the seven projections of one decoder layer as independent GEMVs in one call, each with a block of its own width
    mlp      residual add + norm + quantisation, gate|up, SiLU * up + quantisation, down: what a layer of a user's own model runs

Decoders (``kind``), random weights of the two shapes the package names, ternary or sign weights
    prefill      a prompt into the KV history
    ar           prompt, then greedy one-token steps
    speculative  prompt, then draft (9 rows) + verify (9 rows) iterations
    hybrid       prompt, then confident blocks: drafts that carry the block before as pending rows (16 rows)
    confidence   prompt, then the confidence chain with the FP8 draft projection

A trained decoder predicts with a margin; random weights alone give nearly uniform logits, where the argmax is decided by
rounding.  The random layers are therefore scaled so that each adds a small part to the residual stream, and the embedding is
the output projection with its rows permuted: every token has one confident successor."""
import math

import numpy as np
import torch

from bitmtp_amd import generate, ops
from bitmtp_amd.model import BonsaiDecoder, qwen3_1p7b_args, qwen3_4b_args
from bitmtp_amd.runtime import GraphAtlas

DEVICE = "cuda"
EPS = 1e-6

#: hidden, ffn, query width, key / value width, layers
SHAPES = {"1.7b": (2048, 6144, 2048, 1024, 28), "4b": (2560, 9728, 4096, 1024, 36)}
VOCAB = 151936


def listed():
    return [
        # latency of one small projection of a one-token step (1.7B-shaped o / q projection)
        dict(name="linear-t2-one-token", kind="linear", bits=2, m=1, n=2048, k=2048, x="int8", batch=0, fp16_scales=False),
        # a verify block of nine rows through the largest matrix of a 4B-shaped layer
        dict(name="linear-t2-verify", kind="linear", bits=2, m=9, n=19456, k=2560, x="int8", batch=0, fp16_scales=False),
        # sign weights, long rows, fp16 group scales, a block of four
        dict(name="linear-q1-long-rows", kind="linear", bits=1, m=4, n=9728, k=9728, x="int8", batch=0, fp16_scales=True),
        # a batch of prompts through one projection, quantised on the way (rank-3 activations, ragged length)
        dict(name="linear-t2-prompts", kind="linear", bits=2, m=514, n=12288, k=2048, x="bf16", batch=2, fp16_scales=False),
        # independent projections of one layer at the width of a verify block
        dict(name="grouped-layer", kind="grouped", shape="4b", bits=2, m=8, ragged=False),
        # the MLP of a user's own model on a draft block
        dict(name="mlp-draft-block", kind="mlp", shape="1.7b", bits=2, m=9),
        # prompts: a usual one, and a long one of odd length
        dict(name="prefill-usual", kind="prefill", shape="1.7b", bits=2, prompt=256, new=0),
        dict(name="prefill-long", kind="prefill", shape="4b", bits=2, prompt=3001, new=0),
        # greedy decoding of a short chat turn
        dict(name="ar-short", kind="ar", shape="1.7b", bits=2, prompt=24, new=64),
        # greedy decoding over a longer history
        dict(name="ar-history", kind="ar", shape="4b", bits=2, prompt=777, new=96),
        # block decoding where every block is verified, and where the confidence streak carries it
        dict(name="speculative", kind="speculative", shape="1.7b", bits=2, prompt=256, new=48),
        dict(name="confidence-q1", kind="confidence", shape="1.7b", bits=1, prompt=100, new=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "grouped", "mlp", "prefill", "prefill", "ar", "ar", "speculative", "hybrid", "confidence"])
    shape = rng.choice(["1.7b", "4b"])
    bits = rng.choice([2, 2, 1])
    if kind == "linear":
        x = rng.choice(["int8", "int8", "bf16", "fp16"])
        batch = rng.choice([0, 0, 2, 3])
        m = _log_int(rng, 1, 2048)
        if batch:
            m = max(1, m // batch) * batch
        # any row count; K in whole groups of 128
        return dict(kind="linear", bits=bits, m=m, n=_log_int(rng, 1000, 20000), k=128 * _log_int(rng, 8, 76), x=x,
                    batch=batch, fp16_scales=x == "int8" and batch == 0 and rng.random() < 0.4)
    if kind == "grouped":
        return dict(kind="grouped", shape=shape, bits=bits, m=_log_int(rng, 1, 17), ragged=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind="mlp", shape=shape, bits=bits, m=_log_int(rng, 1, 1500))
    if kind == "prefill":
        return dict(kind="prefill", shape=shape, bits=bits, prompt=_log_int(rng, 40, 2900), new=0)
    long = 900 if kind == "ar" else 600
    return dict(kind=kind, shape=shape, bits=1 if kind == "confidence" else bits, prompt=_log_int(rng, 16, long),
                new=rng.randint(24, 90))


def _packed(n, k, bits, gen, dtype=torch.bfloat16):
    """Random packed weights (ternary codes, p = 1/3 each, or sign bits) and log-normal group scales."""
    per = 8 // bits
    lo, hi = (1, 4) if bits == 2 else (0, 2)
    packed = torch.zeros(n, k // per, dtype=torch.uint8, device=DEVICE)
    for j in range(per):
        packed |= torch.randint(lo, hi, (n, k // per), generator=gen, device=DEVICE, dtype=torch.uint8) << (bits * j)
    scale = torch.exp(torch.randn(n, k // 128, generator=gen, device=DEVICE) * 0.5 - 4.0)
    return packed.view(torch.int8), scale.to(dtype)


def _layer_matrices(shape):
    dim, ffn, q, kv, _ = SHAPES[shape]
    return [(q, dim), (kv, dim), (kv, dim), (dim, q), (ffn, dim), (ffn, dim), (dim, ffn)]


def _widths(case):
    m = case["m"]
    return [1 + (m + 3 * i) % (m + 1) if case["ragged"] else m for i in range(7)]


def _decoder(case, seed):
    args = (qwen3_1p7b_args if case["shape"] == "1.7b" else qwen3_4b_args)(kernel_kind="t2g128" if case["bits"] == 2 else "q1")
    model = BonsaiDecoder.random_init(args, seed=seed, device=DEVICE)
    for lw in model.layers:
        lw.wo.weight_scale.mul_(2.0 ** -10)
        lw.w_down.weight_scale.mul_(2.0 ** -10)
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    model.embed = model.embed[torch.randperm(args.vocab_size, generator=gen, device=DEVICE)].contiguous()
    return model


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        x = torch.randn(m, k, generator=gen, device=DEVICE)
        x = x.to(torch.bfloat16 if case["x"] == "bf16" else torch.float16)
        if case["batch"]:
            x = x.view(case["batch"], -1, k)
        b, ws = _packed(n, k, case["bits"], gen, torch.float16 if case["fp16_scales"] else torch.bfloat16)
        state = dict(case=case, b=b, ws=ws, x=x)
        if case["x"] == "int8":
            state["a"], state["s"] = ops.quant_input(x)
        return state
    if kind == "grouped":
        problems = []
        for m, (n, k) in zip(_widths(case), _layer_matrices(case["shape"])):
            a, s = ops.quant_input(torch.randn(m, k, generator=gen, device=DEVICE).to(torch.bfloat16))
            b, ws = _packed(n, k, case["bits"], gen)
            problems.append((a, b, s, ws))
        return dict(case=case, problems=problems)
    if kind == "mlp":
        dim, ffn = SHAPES[case["shape"]][:2]
        rows = [torch.randn(case["m"], dim, generator=gen, device=DEVICE).to(torch.bfloat16) for _ in range(2)]
        norm = (1.0 + 0.1 * torch.randn(dim, generator=gen, device=DEVICE)).to(torch.bfloat16)
        return dict(case=case, x=rows[0], residual=rows[1], norm=norm, gate_up=_packed(2 * ffn, dim, case["bits"], gen),
                    down=_packed(dim, ffn, case["bits"], gen))
    model = _decoder(case, int(seed))
    roles = ("draft", "verify", "ar") + (("draft_fp8",) if kind == "confidence" else ())
    atlas = GraphAtlas(model, roles=roles, threshold=0.9)
    prompt = torch.randint(0, model.args.vocab_size, (case["prompt"],), generator=gen, device=DEVICE).tolist()
    sigma = atlas.select_segment(case["prompt"] + case["new"] + atlas.M_max)
    # a serving program captures the graphs of its loop before the first request
    atlas.get_graph(atlas.prefill_width, sigma, "ar")
    wanted = {"ar": [(1, "ar")], "speculative": [(9, "draft"), (9, "verify")],
              "hybrid": [(9, "draft"), (16, "draft"), (9, "verify")],
              "confidence": [(8, "draft_fp8"), (9, "draft_fp8"), (16, "draft_fp8")]}
    for width, role in wanted.get(kind, ()):
        atlas.get_graph(width, sigma, role)
    return dict(case=case, atlas=atlas, prompt=prompt, sigma=sigma)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["fp16_scales"]:
            return ops.packed_gemv_ex(state["a"], state["b"], state["s"], state["ws"], bits=case["bits"])
        linear = ops.t2g128_int8xint2_linear if case["bits"] == 2 else ops.q1g128_int8xint1_linear
        a, s = (state["a"], state["s"]) if case["x"] == "int8" else ops.quant_input(state["x"])
        return linear(a, state["b"], s, state["ws"])
    if kind == "grouped":
        return ops.packed_gemv_grouped(state["problems"], bits=case["bits"])
    if kind == "mlp":
        h, q, s = ops.fused_add_norm_quant(state["x"], state["residual"], state["norm"], EPS)
        gate_up = ops.packed_int8_linear(q, state["gate_up"][0], s, state["gate_up"][1])
        q, s = ops.silu_mul_quant(gate_up)
        return h, ops.packed_int8_linear(q, state["down"][0], s, state["down"][1])
    atlas, prompt, new = state["atlas"], state["prompt"], case["new"]
    if kind == "prefill":
        first = generate.prefill(atlas, prompt, state["sigma"])
        return first, atlas.kv(state["sigma"])[:, :, :, :len(prompt)]
    if kind == "ar":
        tokens, _ = generate.ar_generate(atlas, prompt, max_gen_len=new)
    elif kind == "speculative":
        tokens, _ = generate.speculative_generate(atlas, prompt, max_gen_len=new)
    elif kind == "hybrid":
        tokens, _ = generate.hybrid_generate(atlas, prompt, threshold=0.9, max_gen_len=new)
    else:
        tokens, _ = generate.confidence_generate(atlas, prompt, threshold=0.9, max_gen_len=new, use_fp8_draft=True)
    # the history behind them, short of the block that may still be pending
    return np.asarray(tokens), atlas.kv(state["sigma"])[:, :, :, :len(prompt) + len(tokens) - 16]


def _weight_bytes(n, k, bits):
    return n * k * bits // 8 + n * (k // 128) * 2


def _pass(case, tokens, history, head_rows, head_bytes):
    """Bytes and operations of one trip through a decoder: every weight and the history's keys and values once, new keys and
    values written; the output projection for `head_rows` rows."""
    dim, ffn, q, kv, layers = SHAPES[case["shape"]]
    matrices = [(q + 2 * kv, dim), (dim, q), (2 * ffn, dim), (dim, ffn)]
    size = sum(n * k for n, k in matrices)
    seen = tokens * history + tokens * tokens / 2
    nbytes = layers * (sum(_weight_bytes(n, k, case["bits"]) for n, k in matrices) + 4 * kv * (history + tokens))
    flops = layers * (2.0 * size * tokens + 4.0 * q * seen) + 2.0 * dim * VOCAB * head_rows
    return nbytes + head_bytes, flops


def work(case):
    kind, bits = case["kind"], case["bits"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        x = m * (k + 4) if case["x"] == "int8" else 2 * m * k
        return {"bytes": _weight_bytes(n, k, bits) + x + 2 * m * n, "flops": 2.0 * m * n * k}
    if kind == "grouped":
        of = list(zip(_widths(case), _layer_matrices(case["shape"])))
        return {"bytes": sum(_weight_bytes(n, k, bits) + m * (k + 4) + 2 * m * n for m, (n, k) in of),
                "flops": sum(2.0 * m * n * k for m, (n, k) in of)}
    if kind == "mlp":
        m, (dim, ffn) = case["m"], SHAPES[case["shape"]][:2]
        return {"bytes": _weight_bytes(2 * ffn, dim, bits) + _weight_bytes(dim, ffn, bits) + 8 * m * dim + 2 * dim,
                "flops": 6.0 * m * dim * ffn}
    dim = SHAPES[case["shape"]][0]
    packed_head, wide_head = _weight_bytes(VOCAB, dim, 2), 2 * VOCAB * dim
    head = packed_head if bits == 2 else wide_head
    prompt, new = case["prompt"], case["new"]
    trips = [(prompt, 0, 1, head)]
    if kind == "ar":
        trips += [(1, prompt + i, 1, head) for i in range(new - 1)]
    elif kind == "speculative":      # one draft accepted and one verifier token an iteration
        for i in range(0, new - 1, 2):
            trips += [(9, prompt + i, 8, head), (9, prompt + i, 9, head)]
    elif kind in ("hybrid", "confidence"):   # eight tokens an iteration
        head = VOCAB * dim if kind == "confidence" else head
        trips += [(9 if i == 0 else 16, prompt + i, 8, head) for i in range(0, new - 1, 8)]
    total = [_pass(case, *t) for t in trips]
    return {"bytes": sum(b for b, _ in total), "flops": sum(f for _, f in total)}


def tolerance(case):
    """bf16 results of fp32 sums over exact integers: one rounding for an operator.  A decoder rounds to bf16 and to int8 between
    its layers, and whatever moves a value across a rounding boundary moves it by a whole int8 step, so its keys and values carry
    more: 1.2e-2 to 1.6e-2 between two correct orders of the attention's sums.  The tokens do not differ."""
    if case["kind"] in ("linear", "grouped"):
        return {"rel": 2e-3, "max": 1e-2}
    if case["kind"] == "mlp":
        return {"rel": 1e-2, "max": 0.3}
    return {"rel": 2e-2, "max": 0.3}
