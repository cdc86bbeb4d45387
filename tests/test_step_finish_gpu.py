"""Steps in one launch that did not get the whole device (``csrc/step_finish.hip.h``): their results are right in stream
order, without a read in between, and the exchange memory serves the next step.  The device gives up by its own bounded
waits, which are told not to wait at all."""
import threading

import pytest
import torch

from test_step_one_gpu import DEV, _model

pytestmark = pytest.mark.gpu

CASES = [
    # bits, dim, ffn, heads, kv heads, width, role, segment
    (2, 256, 256, 2, 1, 1, "ar", 256),
    (2, 1280, 2304, 8, 8, 1, "ar", 256),
    (1, 1024, 1024, 8, 2, 1, "ar", 4096),
    (2, 384, 640, 3, 1, 3, "ar", 256),
    (1, 384, 640, 3, 1, 9, "verify", 256),
    (2, 1024, 512, 8, 4, 16, "draft", 256),
    (1, 1024, 1024, 8, 2, 2, "ar", 4096),
    (2, 2560, 9728, 32, 8, 9, "verify", 256),
]
#: (first, later): gives up in the first layer, where nothing has been handed over, and in the second
WAITS = [(-1, 0), (0, -1)]


def _atlases(model, sigma, width, role, waits, monkeypatch):
    from bitmtp_amd import decode_ops
    from bitmtp_amd.runtime import GraphAtlas
    out = []
    for flag in ("1", "0"):
        monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", flag)
        monkeypatch.setattr(decode_ops.StepOne, "waits", waits)
        a = GraphAtlas(model, segment_ladder=(sigma,))
        out.append((a, a.get_graph(width, sigma, role)))
    assert out[0][1].one is not None and out[1][1].one is None
    return out


@pytest.mark.parametrize("waits", WAITS)
@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv,width,role,sigma", CASES)
def test_results_without_the_whole_device(bits, dim, ffn, n_heads, n_kv, width, role, sigma, waits, monkeypatch):
    print(f"[case] {bits} bits, {dim} x {ffn}, {n_heads} / {n_kv} heads, {width} rows, {role}, {sigma} slots, {waits}", flush=True)
    (a1, g1), (a0, g0) = _atlases(_model(bits, dim, ffn, n_heads, n_kv), sigma, width, role, waits, monkeypatch)
    gen = torch.Generator(device=DEV).manual_seed(1)
    hist = (torch.randn(tuple(a1.kv(sigma).shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)
    rows = slice(sigma, sigma + width)
    for n in (1, 7, 64 - width, 65 - width, 200, sigma) + ((0,) if role == "ar" else ()):
        tokens = [(7 * n + 13 * i) % 1000 for i in range(width)]
        positions = [max(n - 1, 0) + i for i in range(width)]
        outs = []
        for a, g in ((a1, g1), (a0, g0), (a1, g1)):
            kv = a.kv(sigma)
            kv.copy_(hist)
            if g.one is not None:
                g.one.failed[0] = 0     # (or the separate launches would take over)
            a.replay(g, tokens, positions, n, width - 8 if role == "draft" else 0)
            outs.append((kv[:, :, :, rows].clone(), a.workspace.logits[:g.logits_end - g.logits_start, :1000].clone(), kv.clone(),
                         g.io.out.clone()))
        torch.cuda.synchronize()
        assert g1.one.failed[0] == 1
        assert all(torch.equal(x, y) for x, y in zip(outs[0], outs[2]))
        assert torch.equal(outs[0][2][:, :, :, :sigma], hist[:, :, :, :sigma])
        assert torch.equal(outs[0][2][:, :, :, sigma + width:], hist[:, :, :, sigma + width:])
        # Layer 0 sees no attention: exact integer sums, scaled in another order: one bf16 step before a key's norm and
        # rotation, two behind it.
        first = (outs[0][0][:, 0].float() - outs[1][0][:, 0].float()).abs()
        assert bool((first <= 2.0 ** -6 * outs[1][0][:, 0].float().abs().clamp(min=2.0 ** -3)).all())
        # Behind the attention int8 roundings of a row move by whole steps (as in the comparisons of test_step_block_gpu).
        for x, y in ((outs[0][0].transpose(0, 3), outs[1][0].transpose(0, 3)), (outs[0][1], outs[1][1])):
            x, y = x.float().flatten(1), y.float().flatten(1)
            assert float(((x - y).norm(dim=1) / y.norm(dim=1)).max()) <= 4e-2, f"history of {n}"


@pytest.mark.parametrize("width", [1, 9])
def test_the_exchange_memory_serves_the_next_step(width):
    """Undisturbed steps between such that give up in the first layer, in a later one, and before they begin, on either set
    of exchange memory."""
    from bitmtp_amd.runtime import GraphAtlas, step_descriptor
    model, sigma = _model(2, 1024, 512, 8, 4), 200
    atlas = GraphAtlas(model, segment_ladder=(sigma,))
    g = atlas.get_graph(width, sigma, "ar")
    one, kv, h = g.one, atlas.kv(sigma), atlas.workspace.h[0][:width]
    kv.copy_((torch.randn(tuple(kv.shape), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV) * 0.5).to(torch.bfloat16))
    g.io.step_in.copy_(torch.tensor(step_descriptor("ar", width, model.args.block_size, 150) + [150 + i for i in range(width)]
                                    + list(range(width)), dtype=torch.int32))
    want = None
    for what in ("", "", "first", "", "later", "", "", "later", "first", "mark", "", "mark", ""):
        one.waits = {"first": (-1, 0), "later": (0, -1)}.get(what, (0, 0))
        if what == "mark":
            one.exchange[4:8].view(torch.int32).fill_(1)
        one.failed[0] = 0
        h.zero_()
        kv[:, :, :, sigma:].zero_()
        one.enqueue(model.embed, g.io.step_in, kv, *atlas.rope, sigma, 1e-6, h, width)
        got = (h.float(), kv[:, :, :, sigma:sigma + width].float())
        torch.cuda.synchronize()
        assert one.failed[0] == (what != "")
        if want is None:
            want = got
        for x, y in zip(got, want):
            assert torch.equal(x, y) if what == "" else float((x - y).norm() / y.norm()) <= 4e-2, what


def test_atlases_on_two_streams_take_turns():
    """Steps of two atlases on two streams, made to start together, don't keep each other from the device."""
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 1024, 512, 8, 4)
    atlases = [GraphAtlas(model, segment_ladder=(256,)) for _ in range(2)]
    graphs = [(a.get_graph(1, 256, "ar"), a.get_graph(9, 256, "verify")) for a in atlases]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for n in range(1, 41):
        torch.cuda._sleep(200000)
        start = torch.cuda.Event()
        start.record()
        for a, (ar, verify), stream in zip(atlases, graphs, streams):
            with torch.cuda.stream(stream):
                stream.wait_event(start)
                if n % 2:
                    a.replay(ar, [n], [n], n)
                    a.commit_kv(256, n, 1)
                else:
                    a.replay(verify, [n] * 9, list(range(n, n + 9)), n)
                    a.commit_kv(256, n, 1, 1)
    results = [a.read_outputs(verify)[0] for a, (_, verify) in zip(atlases, graphs)]
    torch.cuda.synchronize()
    for a in atlases:
        assert a._one.failed[0] == 0 and a._block.failed[0] == 0 and a._separate_for == 0
    assert (results[0] == results[1]).all() and torch.equal(atlases[0].kv(256)[:, :, :, :41], atlases[1].kv(256)[:, :, :, :41])


@pytest.mark.parametrize("waits", [(0, 0), (-1, 0)])
def test_atlases_in_two_threads(waits, monkeypatch):
    """The same, queued by two threads, undisturbed and where the steps give up and the separate launches take over."""
    from bitmtp_amd import decode_ops
    from bitmtp_amd.runtime import GraphAtlas
    monkeypatch.setattr(decode_ops.StepOne, "waits", waits)
    model = _model(2, 1024, 512, 8, 4)
    atlases = [GraphAtlas(model, segment_ladder=(256,)) for _ in range(2)]
    graphs = [(a.get_graph(1, 256, "ar"), a.get_graph(9, 256, "verify")) for a in atlases]
    results, errors = [None, None], []

    def steps(i, stream):
        try:
            a, (ar, verify) = atlases[i], graphs[i]
            with torch.cuda.stream(stream):
                for n in range(1, 61):
                    a.replay(ar, [n], [n], n)
                    a.commit_kv(256, n, 1)
                    a.replay(verify, [n] * 9, list(range(n, n + 9)), n + 1)
                results[i] = a.read_outputs(verify)[0].copy(), a.kv(256)[:, :, :, :61].clone()
                stream.synchronize()
        except Exception as e:   # noqa: BLE001 - reported by the test
            errors.append(e)

    threads = [threading.Thread(target=steps, args=(i, torch.cuda.Stream())) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for a in atlases:
        assert (a._separate_for > 0 or a._one.failed[0] + a._block.failed[0] > 0) == (waits != (0, 0))
    (t0, k0), (t1, k1) = results
    if waits == (0, 0):
        assert (t0 == t1).all() and torch.equal(k0, k1)
    else:   # (which steps were separate launches depends on when the flag was seen)
        assert float((k0.float() - k1.float()).norm() / k0.float().norm()) <= 4e-2


@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv,width,first,rows", [
    (2, 256, 256, 2, 1, 1, 0, 1), (1, 384, 640, 3, 1, 9, 1, 8), (2, 1280, 2304, 8, 8, 16, 8, 8), (2, 2560, 9728, 32, 8, 9, 0, 9)])
def test_final_norm(bits, dim, ffn, n_heads, n_kv, width, first, rows):
    """The bits of the launches that norm the rows of separate launches, also behind a step that was done again."""
    from bitmtp_amd import ops
    from bitmtp_amd.decode_ops import FinalNorm
    from bitmtp_amd.model import _vp
    from bitmtp_amd.runtime import GraphAtlas, step_descriptor
    model, sigma = _model(bits, dim, ffn, n_heads, n_kv), 64
    atlas = GraphAtlas(model, segment_ladder=(sigma,))
    g = atlas.get_graph(width, sigma, "ar")
    h = torch.zeros(width, dim, dtype=torch.bfloat16, device=DEV)
    g.io.step_in.copy_(torch.tensor(step_descriptor("ar", width, model.args.block_size, 5) + [5 + i for i in range(width)]
                                    + list(range(width)), dtype=torch.int32))

    def buffers():   # one row more than asked for, which stays
        return (torch.full((rows + 1, dim), 77, dtype=torch.int8, device=DEV), torch.full((rows + 1,), 77.0, device=DEV),
                torch.full((rows + 1, dim), 77.0, dtype=torch.bfloat16, device=DEV))

    for waits in ((0, 0), (-1, 0)):
        g.one.waits = waits
        q, s, out = buffers()
        step = (model.embed, g.io.step_in, atlas.kv(sigma), *atlas.rope, sigma, 1e-6, h, width)
        g.one.enqueue(*step, FinalNorm(model.norm, first, rows, q=q, s=s))
        first_h = h.clone()
        g.one.enqueue(*step, FinalNorm(model.norm, first, rows, out=out))
        assert torch.equal(h, first_h)
        want_q, want_s, want_out = buffers()
        stream = torch.cuda.current_stream().cuda_stream
        x = h[first:first + rows]
        assert ops.actq_lib().bonsai_rmsnorm_quant_int8(_vp(x), _vp(model.norm), 1e-6, _vp(want_q), _vp(want_s), rows, dim, stream) == 0
        assert ops.actq_lib().bonsai_add_rmsnorm_bf16(_vp(x), None, _vp(model.norm), 1e-6, None, _vp(want_out), rows, dim, stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(q, want_q) and torch.equal(s, want_s) and torch.equal(out, want_out)
        assert g.one.failed[0] == (waits != (0, 0))


@pytest.mark.parametrize("width", [1, 9])
def test_a_step_that_did_not_end_is_told_until_the_memory_is_reset(width):
    """Behind a step of which a task was lost (the mark is set from the host) no step pretends to have results."""
    from bitmtp_amd.runtime import GraphAtlas
    atlas = GraphAtlas(_model(2, 1024, 512, 8, 4), segment_ladder=(64,))
    g = atlas.get_graph(width, 64, "ar")
    step = (g, list(range(width)), list(range(5, 5 + width)), 5)
    atlas.replay(*step)
    want = atlas.read_outputs(g)[0].copy()
    g.one.exchange[4:8].view(torch.int32).fill_(2)
    for _ in range(2):
        g.one.failed[0] = 0
        atlas.replay(*step)
        torch.cuda.synchronize()
        assert g.one.failed[0] == 2
        with pytest.raises(RuntimeError, match="did not end"):
            atlas.read_outputs(g)
        with pytest.raises(RuntimeError, match="did not end"):
            atlas.replay(*step)
    g.one.reset()
    atlas.replay(*step)
    assert (atlas.read_outputs(g)[0] == want).all() and g.one.failed[0] == 0


@pytest.mark.parametrize("use_graphs", [True, False])
def test_results_read_on_another_stream(use_graphs):
    """Where separate launches stand in for a step, too, its results are those of that step on whatever stream they are read."""
    from bitmtp_amd.runtime import GraphAtlas
    atlas = GraphAtlas(_model(2, 1024, 512, 8, 4), segment_ladder=(64,), use_graphs=use_graphs)
    g = atlas.get_graph(9, 64, "verify")
    tokens, positions = list(range(9)), list(range(4, 13))
    want = []
    for first in (7, 0):
        atlas.replay(g, [first] + tokens[1:], positions, 5)
        want.append(atlas.read_outputs(g)[0].copy())
    assert (want[0] != want[1]).any()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    for separate in (0, 1):
        atlas._separate_for = separate
        atlas.replay(g, tokens, positions, 5)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            torch.cuda._sleep(20000000)
            atlas._separate_for = separate
            atlas.replay(g, [7] + tokens[1:], positions, 5)
        assert (atlas.read_outputs(g)[0] == want[0]).all(), separate
        stream.synchronize()
