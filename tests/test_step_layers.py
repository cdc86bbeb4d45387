"""What every layer of a step in one launch adds, against the CPU composition of the oracles: layers whose attention and MLP
are nearly all of the residual stream, scores that single out a few slots of the history, values that differ from slot to
slot and head to head.  On the CPU: mistakes planted in the oracle are farther from it than the bounds allow."""
import math

import numpy as np
import pytest
import torch

from bitmtp_amd import runtime
from bitmtp_amd.model import BonsaiDecoder, ModelArgs, rope_tables
from oracle import decode_oracle as DO
from oracle import oracle as O

D = 8        # block size of ModelArgs
VOCAB = 1000

#: What `_errors` may be.  Two evaluations differ in the rounding of single bf16 values, and a row's maximum or a value on the
#: edge of an int8 step then moves others by whole steps (of a normal row 0.03 in all).  With every attention output moved by
#: up to half a bf16 step, which is what probabilities in bf16 do, the oracle moves by up to 0.05, 0.10, 0.21 and 0.4
#: (test_bounds_reject_mistakes).
BOUNDS = np.array([0.06, 0.12, 0.25, 0.5])

CASES = [
    # bits, dim, ffn, heads, kv heads, rows, role, segment
    (2, 1024, 512, 8, 4, 1, "ar", 256),
    (2, 2304, 6400, 24, 8, 1, "ar", 256),       # three query heads per kv head
    (1, 2560, 9728, 32, 8, 1, "ar", 256),
    (2, 1024, 1024, 16, 8, 1, "ar", 4096),
    (2, 384, 640, 3, 1, 3, "ar", 256),
    (1, 1024, 1024, 8, 2, 16, "draft", 256),
    (2, 2560, 9728, 32, 8, 9, "verify", 256),
    (2, 1024, 1024, 16, 8, 9, "verify", 4096),
]


def _lengths(rows, role, sigma):
    """Histories of no slot or one, at the edges of the attention's parts, and as long as the segment."""
    if sigma > 256:
        return [512, 1023, 4095]
    return ([0] if role == "ar" else []) + [1, 64 - rows, 65 - rows, 128, 255]


def _bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _model(bits, dim, ffn, n_heads, n_kv, device):
    args = ModelArgs(dim=dim, n_layers=3, n_heads=n_heads, n_kv_heads=n_kv, ffn_dim=ffn, vocab_size=VOCAB, mask_token_id=VOCAB - 1,
                     kernel_kind="t2g128" if bits == 2 else "q1")
    model = BonsaiDecoder.random_init(args, seed=3, device=device)
    # Attention and MLP (whose rows are about 0.3 and 0.3 dim / 2048) as large as each other, and every layer larger than
    # what came before it: its mistakes are most of the stream behind it.
    for i, lw in enumerate(model.layers):
        lw.wo.weight_scale.mul_(4.0 ** i)
        lw.w_down.weight_scale.mul_(4.0 ** i * 2.0 ** round(math.log2((args.q_dim / ffn) ** 0.5 * 2048 / dim)))
    return model


def _weights(model, rope):
    def pl(p):
        return p.weight.cpu().numpy().view(np.uint8), _bits(p.weight_scale)
    a = model.args
    return {
        # the final norm's rows themselves come out of a projection onto themselves
        "embed": _bits(model.embed), "norm": _bits(model.norm), "head_bf16": O.f32_to_bf16_bits(np.eye(a.dim, dtype=np.float32)),
        "bits": model.layers[0].wqkv.bits, "cos": _bits(rope[0]), "sin": _bits(rope[1]), "eps": a.norm_eps,
        "n_heads": a.n_heads, "n_kv": a.n_kv_heads,
        "layers": [{
            "wqkv": pl(lw.wqkv), "wo": pl(lw.wo), "w_gu": pl(lw.w_gu), "w_down": pl(lw.w_down),
            "input_layernorm": _bits(lw.input_layernorm), "post_attention_layernorm": _bits(lw.post_attention_layernorm),
            "q_norm": _bits(lw.q_norm), "k_norm": _bits(lw.k_norm)} for lw in model.layers],
    }


def _history(args, slots):
    """Keys half as long again as normed ones: scores of +- 1.5, so that some slots have most of a row's weight."""
    kv = np.random.default_rng(1).standard_normal((2, args.n_layers, args.n_kv_heads, slots, 128), dtype=np.float32)
    kv[0] *= 1.5
    return O.f32_to_bf16_bits(kv)


def _step(n, rows, role):
    tokens = [(7 * n + 13 * i) % VOCAB for i in range(rows)]
    return tokens, [max(n - 1, 0) + i for i in range(rows)], rows - D if role == "draft" else 0


def _oracle(weights, hist, sigma, n, rows, role, attention=None):
    """(final norm's rows, keys, values) in fp32; ``attention(layer, q, k, v, vis, scale)`` in place of the oracle's."""
    tokens, positions, n_pend = _step(n, rows, role)
    vis = runtime.dense_visibility(runtime.step_descriptor(role, rows, D, n, n_pend), rows, sigma)
    k, v = hist[0].copy(), hist[1].copy()
    honest, layer = DO.attention, iter(range(99))
    if attention is not None:
        DO.attention = lambda *args: attention(next(layer), honest, *args)
    try:
        out = DO.decode_step(weights, k, v, tokens, positions, vis, sigma, 0, rows)
    finally:
        DO.attention = honest
    return tuple(O.bf16_bits_to_f32(x) for x in (out, k[:, :, sigma:sigma + rows], v[:, :, sigma:sigma + rows]))


def _errors(got, want):
    """Largest difference of a row, over its norm: of the second layer's keys and values, of the third's, of what the last layer
    leaves; and of eight neighbouring values of that, over the row's root mean square."""
    out = []
    for layer in (1, 2):
        err = 0.0
        for x, y in zip(got[1:], want[1:]):
            x, y = (t[layer].transpose(1, 0, 2).reshape(t.shape[2], -1).astype(np.float64) for t in (x, y))
            err = max(err, (np.linalg.norm(x - y, axis=1) / np.linalg.norm(y, axis=1)).max())
        out.append(err)
    x, y = got[0].astype(np.float64), want[0].astype(np.float64)
    d, rms = (x - y).reshape(len(x), -1, 8), np.sqrt((y * y).mean(axis=1))
    out.append((np.linalg.norm(x - y, axis=1) / np.linalg.norm(y, axis=1)).max())
    out.append((np.sqrt((d * d).mean(axis=2)).max(axis=1) / rms).max())
    return np.array(out)


def _within(errors):
    return (errors <= BOUNDS).all()


def _mistakes(weights, n, rows, role):
    """(name, weights, attention) of steps with one mistake in one layer."""
    def only(at, wrong):
        return lambda layer, honest, *args: wrong(honest, *args) if layer == at else honest(*args)

    def changed(at, name, change):
        layers = [dict(lw) for lw in weights["layers"]]
        layers[at][name] = change(*[x.copy() for x in layers[at][name]])
        return {**weights, "layers": layers}

    def no_slots(first, last):
        def wrong(honest, q, k, v, vis, scale):
            vis = vis.copy()
            vis[:, first:last] = False
            return honest(q, k, v, vis, scale)
        return wrong

    def heads_swapped(honest, *args):
        x = honest(*args).copy()
        x[:, :128], x[:, -128:] = x[:, -128:].copy(), x[:, :128].copy()
        return x

    def next_slots(honest, q, k, v, vis, scale):
        v = v.copy()
        v[:, :n - 1] = v[:, 1:n]
        return honest(q, k, v, vis, scale)

    def other_kv_head(honest, q, k, v, *args):
        return honest(q, k, np.roll(v, 1, axis=0), *args)

    def causal_broken(honest, q, k, v, vis, scale):   # a row does not see itself
        vis = vis.copy()
        vis[np.arange(rows), vis.shape[1] - rows + np.arange(rows)] = False
        return honest(q, k, v, vis, scale)

    out = []
    for at in range(3):
        out.append((f"no attention in layer {at}", weights, only(at, lambda honest, *args: 0 * honest(*args))))
        out.append((f"no MLP in layer {at}", changed(at, "w_down", lambda x, s: (x, 0 * s)), None))
        out.append((f"gate and up swapped in layer {at}",
                    changed(at, "w_gu", lambda x, s: (np.roll(x, len(x) // 2, axis=0), np.roll(s, len(s) // 2, axis=0))), None))
        if weights["n_kv"] > 1:
            out.append((f"heads swapped in layer {at}", weights, only(at, heads_swapped)))
        if n > 1:
            out.append((f"values of the next slot in layer {at}", weights, only(at, next_slots)))
            part = max(n // 32, 64)   # as many slots as a workgroup has at least
            for first in (0, n // 2, max(n - part, 0)) if at == 0 else ():   # (the same in every layer)
                out.append((f"slots {first} .. of layer {at} missing", weights, only(at, no_slots(first, min(first + part, n)))))
            if weights["n_kv"] > 1:
                out.append((f"another head's values in layer {at}", weights, only(at, other_kv_head)))
        if n == 1:
            out.append((f"rows that don't see themselves in layer {at}", weights, only(at, causal_broken)))
    return out


@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv,rows,role,sigma", [c for c in CASES if c[1] <= 1024 and (c[7] == 256 or c[5] == 1)])
def test_bounds_reject_mistakes(oracle, bits, dim, ffn, n_heads, n_kv, rows, role, sigma):
    model = _model(bits, dim, ffn, n_heads, n_kv, "cpu")
    weights, hist = _weights(model, rope_tables(model.args, sigma + 16, "cpu")), _history(model.args, sigma + 16)
    for n in _lengths(rows, role, sigma)[::2]:
        want = _oracle(weights, hist, sigma, n, rows, role)

        def rounded_otherwise(layer, honest, *args):
            x = honest(*args)
            return x * (1.0 + (np.random.default_rng(layer).random(x.shape) - 0.5) * 2.0 ** -8)   # half a step at most

        errors = _errors(_oracle(weights, hist, sigma, n, rows, role, rounded_otherwise), want)
        print(f"[info] history of {n}: rounded otherwise {errors}")
        assert _within(errors)
        for name, w, attention in _mistakes(weights, n, rows, role):
            errors = _errors(_oracle(w, hist, sigma, n, rows, role, attention), want)
            print(f"[info] history of {n}: {name} {errors}")
            assert not _within(errors), f"{name}, history of {n}"


@pytest.mark.gpu
@pytest.mark.parametrize("waits", [(0, 0), (-1, 0)])   # as one launch, and done again behind one that gave up
@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv,rows,role,sigma", CASES)
def test_steps_in_one_launch_against_the_oracle(oracle, bits, dim, ffn, n_heads, n_kv, rows, role, sigma, waits, monkeypatch):
    from bitmtp_amd import decode_ops
    print(f"[case] {bits} bits, {dim} x {ffn}, {n_heads} / {n_kv} heads, {rows} rows, {role}, {sigma} slots, {waits}", flush=True)
    monkeypatch.setattr(decode_ops.StepOne, "waits", waits)
    model = _model(bits, dim, ffn, n_heads, n_kv, "cuda:0")
    atlas = runtime.GraphAtlas(model, segment_ladder=(sigma,))
    g = atlas.get_graph(rows, sigma, role)
    assert g.one is not None
    kv = atlas.kv(sigma)
    weights, hist = _weights(model, atlas.rope), _history(model.args, kv.shape[3])
    exact = 0
    for n in _lengths(rows, role, sigma):
        kv.copy_(torch.from_numpy(hist.view(np.int16)).view(torch.bfloat16))
        g.one.failed[0] = 0
        tokens, positions, n_pend = _step(n, rows, role)
        atlas.replay(g, tokens, positions, n, n_pend)
        h, new = _bits(atlas.workspace.h[0][:rows]), _bits(kv[:, :, :, sigma:sigma + rows])   # (in stream order)
        assert g.one.failed[0] == (waits != (0, 0))
        normed, _ = O.c_rmsnorm(h, weights["norm"], weights["eps"])
        got = tuple(O.bf16_bits_to_f32(x) for x in (normed, new[0], new[1]))
        want = _oracle(weights, hist, sigma, n, rows, role)
        errors = _errors(got, want)
        exact += not errors.any()
        print(f"[info] history of {n}: {errors}", flush=True)
        assert _within(errors), f"history of {n}"
        if n == (0 if role == "ar" else 1) and role != "draft":   # the first row sees nothing but itself
            assert not _errors(*([t[:1] if t.ndim == 2 else t[:, :, :1] for t in x] for x in (got, want))).any()
    # Group sums are exact, and one token, or a step done again, keeps its probabilities in fp32: a value of a step has to
    # lie on the edge of a bf16 step to be rounded otherwise.
    if rows == 1 or waits != (0, 0):
        assert exact >= len(_lengths(rows, role, sigma)) - 1
