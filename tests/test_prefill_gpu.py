"""The prompt path: causal attention of wide blocks against float64, and whole prompts against the same decoder
stepped through its captured graphs."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,n_heads,n_kv,base,slots", [
    (1, 16, 8, 0, 40), (64, 16, 8, 0, 96), (65, 16, 8, 63, 160), (127, 4, 4, 1, 128), (130, 32, 8, 190, 400),
    (300, 6, 2, 77, 500), (33, 3, 1, 1000, 1100), (515, 16, 8, 0, 515), (1024, 16, 8, 0, 1024), (1030, 16, 8, 3, 1040),
    (700, 32, 8, 64, 800)])
def test_prefill_attention_against_float64(m, n_heads, n_kv, base, slots):
    from bitmtp_amd import decode_ops
    print(f"[case] prefill attention m={m} heads={n_heads}/{n_kv} base={base}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m + base)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    q = rnd(m, n_heads, 128).to(torch.bfloat16)
    k, v = rnd(n_kv, slots, 128).to(torch.bfloat16), rnd(n_kv, slots, 128).to(torch.bfloat16)
    k[:, base + m:] = float("nan")   # slots behind the block are never read
    v[:, base + m:] = float("nan")
    out = decode_ops.prefill_attention(q, k, v, base)
    torch.cuda.synchronize()
    seen = base + m
    hpg = n_heads // n_kv
    qd = q.double().transpose(0, 1).reshape(n_kv, hpg * m, 128)
    s = torch.bmm(qd, k[:, :seen].double().transpose(1, 2).contiguous()) / np.sqrt(128.0)
    s = s.view(n_kv, hpg, m, seen)
    ok = torch.arange(seen, device=DEV)[None, :] <= base + torch.arange(m, device=DEV)[:, None]
    p = torch.softmax(s.masked_fill(~ok, float("-inf")), dim=-1)
    want = torch.bmm(p.view(n_kv, hpg * m, seen), v[:, :seen].double()).view(n_heads, m, 128).transpose(0, 1)
    got = out.view(m, n_heads, 128).double()
    assert torch.isfinite(got).all()
    assert ((got - want).abs() <= 2e-3 + 2e-2 * want.abs()).all()


def _assert_causal_attention(got, q, k, v, base):
    """`got` [M, heads, 128] against float64, head by head: probabilities are rounded to bf16 and divided by their rounded
    sum (2 * 2^-9 of sum p |v|), the row is rounded once more (2^-9); scores and sums are fp32."""
    m, n_heads = q.shape[:2]
    seen = base + m
    ok = torch.arange(seen, device=DEV)[None, :] <= base + torch.arange(m, device=DEV)[:, None]
    for h in range(n_heads):
        kh, vh = (t[h // (n_heads // k.shape[0]), :seen].double() for t in (k, v))
        p = torch.softmax((q[:, h].double() @ kh.T / np.sqrt(128.0)).masked_fill(~ok, float("-inf")), dim=-1)
        want = p @ vh
        bound = 2.0 ** -8 * (p @ vh.abs()) + 2.0 ** -9 * want.abs() + 1e-4
        assert ((got[:, h].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("m,n_heads,n_kv", [(40, 16, 8), (1030, 16, 8)])
def test_prefill_attention_with_a_history_of_minus_infinity(m, n_heads, n_kv):
    """Scores of -inf in the first slots (more than a whole 64-slot chunk of them) weigh nothing, in either kernel."""
    from bitmtp_amd import decode_ops
    print(f"[case] prefill attention, -inf scores, m={m}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m)
    base, hidden = 100, 70
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    q, k, v = rnd(m, n_heads, 128), rnd(n_kv, base + m, 128), rnd(n_kv, base + m, 128)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, :hidden, 0] = float("-inf")
    got = decode_ops.prefill_attention(q, k, v, base).view(m, n_heads, 128)
    torch.cuda.synchronize()
    _assert_causal_attention(got, q, k[:, hidden:], v[:, hidden:], base - hidden)


@pytest.mark.parametrize("m,n_heads,n_kv,base,slots,split", [
    # two rounds of 32-pair workgroups on 256 CUs, and the first row count beyond
    (1024, 16, 8, 5, 1040, True), (1025, 16, 8, 5, 1040, False),
    # ratios that leave pairs of the 128 idle (3, 5, 7, 24), and one that has none to spare
    (2571, 6, 2, 30, 2610, False), (1540, 20, 4, 0, 1540, False), (600, 56, 8, 65, 670, False), (200, 120, 5, 10, 210, False),
    (1100, 16, 16, 63, 1200, False),
    # more than 32 query heads a kv head: never the 32-pair kernel
    (1, 33, 1, 0, 8, False), (70, 40, 1, 129, 200, False), (67, 128, 2, 0, 67, False), (131, 128, 1, 1, 140, False)])
def test_which_prefill_attention_kernel_runs(m, n_heads, n_kv, base, slots, split):
    from bitmtp_amd import decode_ops
    hpg, cus = n_heads // n_kv, torch.cuda.get_device_properties(0).multi_processor_count
    if cus == 256:  # (the line lies elsewhere on a part of another size; the results below hold there too)
        assert split == (hpg <= 32 and -(-m // (32 // hpg)) * n_kv <= 2 * cus)
    print(f"[case] prefill attention kernel m={m} heads={n_heads}/{n_kv} base={base}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m + base)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    q, k, v = rnd(m, n_heads, 128), rnd(n_kv, slots, 128), rnd(n_kv, slots, 128)
    seen = base + m
    k[:, seen:] = float("nan")
    v[:, seen:] = float("nan")
    got = decode_ops.prefill_attention(q, k, v, base).view(m, n_heads, 128)
    torch.cuda.synchronize()
    if cus == 256:
        assert decode_ops.prefill_attention_kernel() == ("prefill_attn_split_kernel" if split else "prefill_attn_kernel")
    _assert_causal_attention(got, q, k, v, base)


@pytest.mark.parametrize("m,n_heads,n_kv", [(1, 4, 2), (33, 3, 1), (67, 16, 8)])
def test_prompt_rows_rope_is_the_steps_own(m, n_heads, n_kv):
    """q / k norm + RoPE + KV write of prompt rows: the bits of the step's entry point, 32 rows at a time."""
    from bitmtp_amd import decode_ops
    print(f"[case] prompt rope m={m} heads={n_heads}/{n_kv}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    x, qw, kw, cos, sin = rnd(m, (n_heads + 2 * n_kv) * 128), rnd(128), rnd(128), rnd(90, 128), rnd(90, 128)
    pos = torch.randint(-2, 95, (m,), generator=gen, device=DEV, dtype=torch.int32)
    got, want = (torch.zeros(2, n_kv, m + 8, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    q_got, q_want = (torch.zeros(m, n_heads, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    lib, p = decode_ops.decode_lib(), lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = lib.bonsai_prefill_rope_kv_write(p(x), p(qw), p(kw), 1e-6, p(cos), p(sin), p(pos), p(q_got), p(got[0]), p(got[1]),
                                          m, n_heads, n_kv, m + 8, 5, 90, stream)
    assert rc == 0
    for r in range(0, m, 32):
        rows = min(32, m - r)
        decode_ops.qk_norm_rope_kv_write(x[r:r + rows], qw, kw, 1e-6, cos, sin, pos[r:r + rows], q_want[r:r + rows], want[0],
                                         want[1], n_heads, n_kv, 5 + r)
    assert torch.equal(q_got.view(torch.int16), q_want.view(torch.int16))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_prefill_attention_argument_checks():
    from bitmtp_amd import decode_ops
    q = torch.zeros(8, 4, 128, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(2, 16, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError):
        decode_ops.prefill_attention(q, k, k, 9)          # runs past the slots
    with pytest.raises(RuntimeError):
        decode_ops.prefill_attention(q[:, :3].contiguous(), k, k, 0)   # heads not a multiple of the kv heads


def _replayed(atlas, prompt, sigma):
    """The prompt through width-32 replays of the captured AR graph; the last row's logits."""
    W = atlas.prefill_width
    g = atlas.get_graph(W, sigma, "ar")
    for c in range(0, len(prompt), W):
        take = min(W, len(prompt) - c)
        atlas.replay(g, list(prompt[c:c + take]) + [0] * (W - take), [c + i for i in range(W)], c)
        atlas.commit_kv(sigma, c, take)
    atlas.read_outputs(g)
    logits = atlas.workspace.logits_buf[: W * atlas.workspace.logits.shape[1]].view(W, -1)
    return logits[take - 1].float().clone()


@pytest.mark.parametrize("kind,head,n,block", [("t2g128", None, 33, None), ("t2g128", None, 200, 96),
                                               ("q1", "bf16", 157, None), ("q1", "q1", 70, 64)])
def test_prompt_block_against_replayed_steps(kind, head, n, block, monkeypatch):
    """Keys, values and last-row logits of the prompt path are those of the stepped decoder: the first layer to the
    bit (K = 512 is one K slice in every kernel: the same sums), deeper ones and the logits within the order of the
    attention's sums (which moves single int8 steps; equal to the bit as well at these sizes when this was written)."""
    from bitmtp_amd import generate, runtime
    from bitmtp_amd.model import BonsaiDecoder, ModelArgs
    from bitmtp_amd.runtime import GraphAtlas
    print(f"[case] prompt {kind} head={head} n={n} block={block}", flush=True)
    args = ModelArgs(dim=512, n_layers=3, n_heads=4, n_kv_heads=2, ffn_dim=1024, vocab_size=1000,
                     mask_token_id=999, kernel_kind=kind)
    model = BonsaiDecoder.random_init(args, seed=5, device=DEV, head_kind=head)
    atlas = GraphAtlas(model, segment_ladder=(256,))
    prompt = np.random.default_rng(n).integers(0, 1000, n).tolist()
    want_logits = _replayed(atlas, prompt, 256)
    want = atlas.kv(256)[:, :, :, :n].clone()
    atlas.kv(256).fill_(float("nan"))
    if block is not None:
        monkeypatch.setattr(runtime, "PROMPT_BLOCK_MAX", block)
    first = generate.prefill(atlas, prompt, 256)
    got = atlas.kv(256)[:, :, :, :n]
    logits = atlas.workspace.logits_buf[: want_logits.numel()].float()
    scale = want_logits.abs().max()
    assert (logits - want_logits).abs().max() <= 2e-2 * scale
    assert first == int(logits[:1000].argmax())
    assert torch.equal(got[:, 0].view(torch.int16), want[:, 0].view(torch.int16))
    assert (got.float() - want.float()).norm() <= 2e-2 * want.float().norm()


def test_prompt_longer_than_its_segment_is_refused():
    from bitmtp_amd import generate
    from bitmtp_amd.model import BonsaiDecoder, ModelArgs
    from bitmtp_amd.runtime import GraphAtlas
    args = ModelArgs(dim=512, n_layers=1, n_heads=4, n_kv_heads=2, ffn_dim=1024, vocab_size=1000, mask_token_id=999)
    atlas = GraphAtlas(BonsaiDecoder.random_init(args, seed=5, device=DEV), segment_ladder=(64,))
    with pytest.raises(RuntimeError):
        generate.prefill(atlas, [1] * 65, 64)


@pytest.mark.parametrize("m,ffn", [(300, 65536), (300, 65664), (530, 65664)])   # (the wide kernel's by its estimate)
def test_mlp_rows_up_to_and_past_the_longest_in_operand_order(m, ffn):
    """A down projection whose rows the quantiser leaves in the order of the wide kernel's operands, and the first one whose rows it
    cannot: the product of the same quantised rows."""
    from bitmtp_amd import model as md
    from bitmtp_amd import ops
    print(f"[case] prompt of {m} rows, {ffn} wide", flush=True)
    args = md.ModelArgs(dim=1024, n_layers=1, n_heads=2, n_kv_heads=1, ffn_dim=ffn, vocab_size=1000, mask_token_id=999)
    model = md.BonsaiDecoder.random_init(args, seed=5, device=DEV)
    buffers = md.PromptBuffers(args, m, DEV)
    kv = torch.zeros(2, 1, 1, 640, 128, dtype=torch.bfloat16, device=DEV)
    positions = torch.arange(m, dtype=torch.int32, device=DEV)
    lib, p = ops.t2_lib(), lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    down, inner = model.layers[0].w_down, buffers._rest[7].view(-1)[:m * ffn].view(m, ffn)
    q, s = torch.empty(m, ffn, dtype=torch.int8, device=DEV), torch.empty(m, 1, device=DEV)
    want = torch.empty(m, args.dim, dtype=torch.bfloat16, device=DEV)
    assert lib.t2g128_gemv_ordered(p(q), p(down.weight), p(want), p(s), p(down.weight_scale), m, args.dim, ffn, 0, 1,
                                   stream) == (0 if ffn <= 65536 else -1)
    md.enqueue_prompt_block(model, buffers, torch.arange(m, device=DEV), 0, positions, kv, md.rope_tables(args, 640, DEV))
    assert ops.actq_lib().bonsai_act_quant_int8(p(inner), 0, p(q), p(s), m, ffn, stream) == 0
    assert lib.t2g128_gemv_ex(p(q), p(down.weight), p(want), p(s), p(down.weight_scale), m, args.dim, ffn, 0, 0, stream) == 0
    # Sums of 513 groups at most in another order: 513 * 2^-24 of the sum of their magnitudes, which is at most sqrt(513) of their
    # root sum of squares, and that is the rms of results whose groups have random signs: 2^-10 of it, and a bf16 step each.
    got, want = buffers.proj[:m].double(), want.double()
    assert torch.isfinite(want).all() and bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -10 * want.pow(2).mean().sqrt()).all())
