"""All layers of a one-token step as one launch (``decode_ops.StepOne``) against the separate launches of the same step:
shapes at the edges of what the launch takes, histories at the edges of its attention's parts, sets of exchange memory
used in turn, and what happens after a launch that did not get the whole device."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _model(bits, dim, ffn, n_heads, n_kv, layers=3, seed=3):
    from bitmtp_amd.model import BonsaiDecoder, ModelArgs
    args = ModelArgs(dim=dim, n_layers=layers, n_heads=n_heads, n_kv_heads=n_kv, ffn_dim=ffn, vocab_size=1000, mask_token_id=999,
                     kernel_kind="t2g128" if bits == 2 else "q1")
    model = BonsaiDecoder.random_init(args, seed=seed, device=DEV)
    for lw in model.layers:   # layers that add a small part to the residual stream, as trained ones do
        lw.wo.weight_scale.mul_(2.0 ** -10)
        lw.w_down.weight_scale.mul_(2.0 ** -10)
    return model


def _pair(model, sigma, monkeypatch):
    """Atlases whose one-token step is one launch / separate launches."""
    from bitmtp_amd.runtime import GraphAtlas
    atlases = []
    for flag in ("1", "0"):
        monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", flag)
        a = GraphAtlas(model, segment_ladder=(sigma,))
        g = a.get_graph(1, sigma, "ar")
        assert (g.one is not None) == (flag == "1")
        atlases.append((a, g))
    return atlases


def _compare(model, sigma, lengths, monkeypatch):
    (a1, g1), (a0, g0) = _pair(model, sigma, monkeypatch)
    gen = torch.Generator(device=DEV).manual_seed(1)
    hist = (torch.randn(tuple(a1.kv(sigma).shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)
    for n in lengths:
        outs = []
        for a, g in ((a1, g1), (a0, g0), (a1, g1)):
            a.kv(sigma).copy_(hist)
            a.replay(g, [n % 1000], [n], n)
            a.read_outputs(g)
            outs.append((a.workspace.h[0][0].clone() if g.one is not None else None, a.kv(sigma)[:, :, :, sigma].clone(),
                         a.workspace.logits[0, :1000].clone()))
        assert torch.equal(outs[0][1], outs[2][1]) and torch.equal(outs[0][2], outs[2][2])   # other set, same bits
        assert torch.equal(a1.kv(sigma)[:, :, :, :sigma], hist[:, :, :, :sigma])
        # layer 0 sees no attention: its keys and values differ by the order of a projection's sums at most
        first = (outs[0][1][:, 0].view(torch.int16).int() - outs[1][1][:, 0].view(torch.int16).int()).abs()
        assert first.max() <= 1
        # Behind the attention (fp32 probabilities here, bf16 there) int8 roundings of a row move by whole steps.  If every
        # value of a normal row moved by one, 1 / 127 of its maximum of about 3.5 rms, a product of it would change by
        # 2.8e-2; the row itself differs by less than a bf16 step, 4e-3, a layer.
        for x, y in ((outs[0][1], outs[1][1]), (outs[0][2], outs[1][2])):
            x, y = x.float(), y.float()
            assert float((x - y).norm() / y.norm()) <= 4e-2, f"history of {n}"
        assert a1._one.failed[0] == 0


SHAPES = [
    # bits, dim, ffn, heads, kv heads
    (2, 256, 256, 2, 1),        # one unit of K, most workgroups without rows
    (2, 1024, 512, 8, 4),       # some waves without a unit
    (2, 1280, 2304, 8, 8),      # five units, nine units: remainders in the split of K, rows that leave workgroups idle
    (2, 2048, 6144, 16, 8),     # the smaller build at its largest
    (2, 2560, 9728, 32, 8),     # the larger build at its largest
    (2, 2304, 6400, 24, 8),     # three query heads per kv head
    (1, 1024, 1024, 8, 2),
    (1, 2048, 6144, 16, 8),
    (1, 2560, 9728, 32, 8),
]


@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv", SHAPES)
def test_one_launch_against_the_separate_launches(bits, dim, ffn, n_heads, n_kv, monkeypatch):
    print(f"[case] {bits} bits, {dim} x {ffn}, {n_heads} / {n_kv} heads", flush=True)
    _compare(_model(bits, dim, ffn, n_heads, n_kv), 256, (0, 1, 7, 63, 64, 127, 128, 255), monkeypatch)


@pytest.mark.parametrize("n_heads,n_kv", [(16, 8), (32, 8), (8, 1)])
def test_long_histories(n_heads, n_kv, monkeypatch):
    """More slots than one request ahead covers, up to several passes of every wave."""
    print(f"[case] long histories, {n_heads} / {n_kv} heads", flush=True)
    _compare(_model(2, 1024, 1024, n_heads, n_kv), 4096, (300, 511, 512, 1000, 1023, 1024, 2047, 3333, 4095), monkeypatch)


@pytest.mark.parametrize("width", [1, 9])
def test_history_lengths_outside_the_segment(width):
    """``cache_len`` below 0 is an empty history and above the segment a full one, as for every other attention kernel."""
    from bitmtp_amd.runtime import GraphAtlas, step_descriptor
    model, sigma = _model(2, 1024, 512, 8, 4), 200
    atlas = GraphAtlas(model, segment_ladder=(sigma,))
    g = atlas.get_graph(width, sigma, "ar")
    assert g.one is not None
    kv = atlas.kv(sigma)
    gen = torch.Generator(device=DEV).manual_seed(1)
    hist = (torch.randn(tuple(kv.shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)
    outs = {}
    for n in (0, -1, -1000, -2 ** 31, sigma, sigma + 1, sigma + 70, 2 ** 31 - 1):
        kv.copy_(hist)
        inputs = [n] + step_descriptor("ar", width, model.args.block_size, 0)[1:] + list(range(width)) + list(range(width))
        g.io.step_in.copy_(torch.tensor(inputs, dtype=torch.int32))
        h = atlas.workspace.h[0][:width]
        g.one.enqueue(model.embed, g.io.step_in, kv, *atlas.rope, sigma, 1e-6, h, width)
        torch.cuda.synchronize()
        assert g.one.failed[0] == 0
        outs[n] = (h.clone(), kv.clone())
    for n, (h, after) in outs.items():
        want = outs[0 if n < 0 else min(n, sigma)]
        assert torch.equal(h, want[0]) and torch.equal(after, want[1]), n
    assert not torch.equal(outs[0][0], outs[sigma][0])


def test_shapes_that_keep_the_separate_launches(monkeypatch):
    from bitmtp_amd import decode_ops
    from bitmtp_amd.model import step_one
    ok = (2, 3, 2048, 6144, 16, 8)
    assert decode_ops.StepOne.exchange_bytes(ok, torch.device(DEV)) > 0
    for shape in ((2, 1, 2048, 6144, 16, 8),        # one layer
                  (2, 3, 1152, 6144, 16, 8),        # half a unit of K
                  (1, 3, 1280, 6144, 16, 8),
                  (2, 3, 8192, 28672, 64, 8),       # more rows than a lane holds weights for
                  (2, 3, 2048, 6144, 15, 8),
                  (3, 3, 2048, 6144, 16, 8)):
        assert decode_ops.StepOne.exchange_bytes(shape, torch.device(DEV)) == 0, shape
    assert step_one(_model(2, 1024, 512, 8, 4, layers=1)) is None
    monkeypatch.setenv("BONSAI_FUSED_STEP", "0")
    assert step_one(_model(2, 1024, 512, 8, 4)) is None


def _refused(width, cases):
    """Every case is refused by the host.  The other arguments are those of a step that could run, in its own memory, and a
    shape is known to be refused before the call."""
    import ctypes
    from bitmtp_amd import decode_ops
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 256, 256, 2, 1)
    atlas = GraphAtlas(model, segment_ladder=(64,))
    g = atlas.get_graph(width, 64, "ar")
    seen = []
    g.one._launch = lambda d, rows: seen.append(d) or 0    # the arguments of a step, which is not queued
    norm = decode_ops.FinalNorm(model.norm, 0, width, q=atlas.workspace.l_q, s=atlas.workspace.l_s)
    g.one.enqueue(model.embed, g.io.step_in, atlas.kv(64), *atlas.rope, 64, 1e-6, atlas.workspace.h[0][:width], width, norm)
    good = {name: getattr(seen[0], name) for name, _ in decode_ops.StepOneDesc._fields_}
    for rows, change in cases:
        d = dict(good)
        for name, value in change.items():
            d[name] = good[name] + int(value[1:]) if isinstance(value, str) else value
        if set(change) & {"dim", "n_layers", "n_heads", "bits"}:
            shape = [d[k] for k in ("bits", "n_layers", "dim", "ffn", "n_heads", "n_kv")]
            assert g.one.exchange_bytes(shape, torch.device(DEV)) == 0, shape
        assert type(g.one)._launch(g.one, decode_ops.StepOneDesc(**d), rows) != 0, (rows, change)


#: addresses that are not there or not aligned ("+4": four bytes on), sizes, and the final norm's
BAD_ARGUMENTS = [dict(layers=0), dict(status=0), dict(exchange="+64"), dict(kv="+8"), dict(embed="+8"), dict(sigma=96),
                 dict(sigma=-1), dict(vocab=0), dict(max_pos=0), dict(n_layers=1), dict(n_heads=0), dict(bits=4),
                 dict(norm_w=0), dict(norm_w="+8"), dict(norm_q=0), dict(norm_q="+4"), dict(norm_s=0), dict(norm_s="+2"),
                 dict(h_out="+4"), dict(norm_out=1 << 40 | 8), dict(norm_rows=-1), dict(norm_first=-1), dict(norm_first=1),
                 dict(norm_rows=17)]


def test_argument_checks():
    from bitmtp_amd import decode_ops
    _refused(1, [(1, bad) for bad in BAD_ARGUMENTS + [dict(dim=640)]])
    assert decode_ops.decode_lib().bonsai_decode_step_one(None, None) != 0


@pytest.mark.parametrize("use_graphs", [True, False])
def test_steps_are_repeated_after_a_launch_that_gave_up(use_graphs, monkeypatch):
    """One step of a loop finds the mark of a launch that gave up: the launch behind it does it again, and the separate
    launches stay for a while."""
    from bitmtp_amd import generate
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 1024, 1024, 8, 4)
    prompt = list(range(40, 90))
    monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", "0")
    want, _ = generate.ar_generate(GraphAtlas(model, segment_ladder=(256,)), prompt, max_gen_len=24)
    monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", "1")
    atlas = GraphAtlas(model, segment_ladder=(256,), use_graphs=use_graphs)
    sigma = 256
    token = generate.prefill(atlas, prompt, sigma)
    n, out = len(prompt), [token]
    g = atlas.get_graph(1, sigma, "ar")
    assert g.one is not None
    for step in range(23):
        if step == 5:
            atlas._one.exchange[4:8].view(torch.int32).fill_(1)
        atlas.replay(g, [token], [n], n)
        atlas.commit_kv(sigma, n, 1)
        n += 1
        token = int(atlas.read_outputs(g)[0][0])
        out.append(token)
        assert atlas._one.failed[0] == (step == 5) and atlas._separate_for == (64 - (step - 5) if step > 5 else 0)
    assert out == want
    for _ in range(atlas._separate_for):
        atlas.replay(g, [token], [n], n)
    kept = atlas.read_outputs(g)[0][0]
    atlas.replay(g, [token], [n], n)      # one launch again
    assert atlas._separate_for == 0 and atlas.read_outputs(g)[0][0] == kept and atlas._one.failed[0] == 0


def test_several_steps_before_a_read():
    """Steps and commits queued without a read in between, read out of order."""
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 1024, 512, 8, 4)
    atlas = GraphAtlas(model, segment_ladder=(64, 256))
    ga, gb = atlas.get_graph(1, 64, "ar"), atlas.get_graph(1, 256, "ar")
    for n in range(10):
        atlas.replay(ga, [n], [n], n)
        atlas.commit_kv(64, n, 1)
    atlas.migrate_segment(64, 256, 10)
    atlas.replay(gb, [10], [10], 10)
    a = atlas.read_outputs(ga)[0].copy()
    b = atlas.read_outputs(gb)[0].copy()
    kv = atlas.kv(256)[:, :, :, :10].clone()
    for n in range(10):   # the same one by one
        atlas.replay(gb, [n], [n], n)
        atlas.commit_kv(256, n, 1)
        out = atlas.read_outputs(gb)[0].copy()
    assert np.array_equal(a, out)
    atlas.replay(gb, [10], [10], 10)
    assert np.array_equal(b, atlas.read_outputs(gb)[0]) and torch.equal(kv, atlas.kv(256)[:, :, :, :10])


def test_results_that_look_as_if_they_had_not_come():
    """Results are waited for by a mark in the pinned buffer; where a word keeps that value, by the event behind the replay.
    Replays without a read in between, and reads without a replay."""
    from bitmtp_amd.model import StepIO
    from bitmtp_amd.runtime import GraphAtlas
    atlas = GraphAtlas(_model(2, 1024, 512, 8, 4), segment_ladder=(64,))
    g = atlas.get_graph(9, 64, "verify")
    tokens, positions = list(range(9)), list(range(4, 13))
    atlas.replay(g, tokens, positions, 5)
    want = [np.copy(x) for x in atlas.read_outputs(g)]
    assert g.io.arrived
    for marked in (False, True):
        atlas.replay(g, [7] * 9, positions, 5)
        atlas.replay(g, tokens, positions, 5)
        assert not g.io.arrived
        torch.cuda.synchronize()
        if marked:
            g.io.out_host[8] = StepIO.PENDING
        for _ in range(2):
            got = atlas.read_outputs(g)
            assert g.io.arrived != marked
            assert all(np.array_equal(x[:8], y[:8]) for x, y in zip(got[:2], want[:2])) and got[2] == want[2]
