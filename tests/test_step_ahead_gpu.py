"""Steps queued behind steps whose results the host has not seen: one-token steps one after the other, a verification behind its
draft, and results that a captured step stores to pinned memory itself."""
import itertools

import numpy as np
import pytest
import torch

from test_step_one_gpu import DEV, _model

pytestmark = pytest.mark.gpu


def _atlas(ladder=(64, 256), **kw):
    from bitmtp_amd.runtime import GraphAtlas
    return GraphAtlas(_model(2, 1024, 512, 8, 4), segment_ladder=ladder, **kw)


def _history(atlas, tokens):
    sigma = max(s for s in atlas.kv_buffers)
    return atlas.kv(sigma)[:, :, :, :tokens].clone()


@pytest.mark.parametrize("loop", ["ar", "speculative"])
@pytest.mark.parametrize("prompt,length", [(1, 2), (17, 3), (20, 40), (50, 90), (150, 60)])
def test_the_same_tokens_and_history_as_steps_that_wait(loop, prompt, length, monkeypatch):
    """Across segments, with and without an end-of-text token, several times with the same graphs."""
    from bitmtp_amd import generate
    fn = generate.ar_generate if loop == "ar" else generate.speculative_generate
    atlas = _atlas()
    tokens = [(7 * i + 3) % 990 for i in range(prompt)]
    plain = {}
    with monkeypatch.context() as m:
        m.setattr(atlas, "step_ahead", lambda g, most: 0)
        m.setattr(atlas, "verify_drafted", lambda *a: False)
        full = fn(atlas, tokens, max_gen_len=length)[0]
        for eos in ((), (full[len(full) * 2 // 3],)):
            out, st = fn(atlas, tokens, max_gen_len=length, eos_ids=eos)
            plain[eos] = (out, st["n_iters"], _history(atlas, prompt + len(out) - 1))
    for _ in range(2):
        for eos, (want, n_iters, history) in plain.items():
            out, st = fn(atlas, tokens, max_gen_len=length, eos_ids=eos)
            assert out == want and st["n_iters"] == n_iters
            assert torch.equal(_history(atlas, prompt + len(out) - 1), history)
            assert all(one is None or one.failed[0] == 0 for one in (atlas._one, atlas._block))


@pytest.mark.parametrize("loop", ["ar", "speculative"])
def test_a_step_that_gave_up_with_others_behind_it(loop):
    """What is queued behind it reads its results, which the launch behind it makes; then separate launches take over."""
    from bitmtp_amd import generate
    fn = generate.ar_generate if loop == "ar" else generate.speculative_generate
    atlas = _atlas((256,))
    prompt = list(range(3, 20))
    fn(atlas, prompt, max_gen_len=4)
    want, _ = fn(atlas, prompt, max_gen_len=12)
    one = atlas._one if loop == "ar" else atlas._block
    one.exchange[4:8].view(torch.int32).fill_(1)   # the mark of a launch that did not get the whole device
    out, _ = fn(atlas, prompt, max_gen_len=12)
    assert len(out) == 12 and atlas._separate_for > 0 and out[0] == want[0]
    atlas._separate_for = 0
    assert fn(atlas, prompt, max_gen_len=12)[0] == want


def _disturbed(one, launches):
    """``launches`` on a device that is still busy, the first one a step of ``one`` that does not get all of it."""
    one.failed[0] = 0
    torch.cuda._sleep(5000000)   # (nothing has begun when the last one is queued)
    one.exchange[4:8].view(torch.int32).fill_(1)
    return launches()


def _successors(ladder, **kw):
    """An atlas whose model has another token behind each token than itself (the tied head of ``_model`` repeats its input)."""
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 1024, 512, 8, 4)
    model.embed = torch.roll(model.embed, 37, 0)
    return GraphAtlas(model, segment_ladder=ladder, **kw)


def _random_history(atlas, sigma):
    kv = atlas.kv(sigma)
    gen = torch.Generator(device=DEV).manual_seed(1)
    return kv, (torch.randn(tuple(kv.shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)


@pytest.mark.parametrize("steps", [1, 4])
def test_steps_behind_one_that_was_done_again(steps):
    """They go on from its token and with its row in the history: to the bit what steps give that wait for each other."""
    sigma, n = 256, 20
    atlas = _successors((sigma,))
    g, (kv, hist) = atlas.get_graph(1, sigma, "ar"), _random_history(atlas, sigma)

    def step(token, at):
        atlas.replay(g, [token], [at], at)
        return int(atlas.read_outputs(g)[0][0])

    kv.copy_(hist)
    tokens, rows = [_disturbed(g.one, lambda: step(5, n))], [kv[:, :, :, sigma].clone()]
    torch.cuda.synchronize()
    assert g.one.failed[0] == 1
    g.one.failed[0] = 0
    for i in range(1, steps + 1):
        atlas.commit_kv(sigma, n + i - 1, 1)
        tokens.append(step(tokens[-1], n + i))
        rows.append(kv[:, :, :, sigma].clone())
    assert g.one.failed[0] == 0 and len(set([5] + tokens)) == steps + 2
    kv.copy_(hist)

    def queue():
        atlas.replay(g, [5], [n], n)
        assert atlas.step_ahead(g, steps) == steps
    _disturbed(g.one, queue)
    assert [atlas.read_step(g, n + i) for i in range(steps + 1)] == tokens
    torch.cuda.synchronize()
    assert g.one.failed[0] == 1
    for i, row in enumerate(rows):
        assert torch.equal(kv[:, :, :, n + i if i < steps else sigma], row), f"row of step {i}"


def test_a_verification_behind_a_draft_that_was_done_again():
    sigma, n, pending, mask = 256, 20, 5, 999
    atlas = _successors((sigma,))
    draft, verify = atlas.get_graph(9, sigma, "draft"), atlas.get_graph(9, sigma, "verify")
    kv, hist = _random_history(atlas, sigma)
    block = ([pending, pending] + [mask] * 7, [n] + [n + i for i in range(8)], n, 1)
    positions = [n + i for i in range(9)]
    assert draft.one is verify.one
    kv.copy_(hist)
    _disturbed(draft.one, lambda: atlas.replay(draft, *block))
    want = [atlas.read_outputs(draft)]
    torch.cuda.synchronize()
    assert draft.one.failed[0] == 1
    draft.one.failed[0] = 0
    atlas.commit_kv(sigma, n, 1)
    atlas.replay(verify, [pending] + [int(t) for t in want[0][0][:8]], positions, n + 1)
    want.append(atlas.read_outputs(verify))
    after = kv.clone()
    assert draft.one.failed[0] == 0
    kv.copy_(hist)

    def queue():
        atlas.replay(draft, *block)
        assert atlas.verify_drafted(verify, draft, pending, positions, n + 1, 1)
    _disturbed(draft.one, queue)
    got = [atlas.read_outputs(draft), atlas.read_outputs(verify)]
    torch.cuda.synchronize()
    assert draft.one.failed[0] == 1
    for (x, y) in zip(want, got):
        assert all(np.array_equal(a, b) for a, b in zip(x, y))
    assert torch.equal(kv, after)


def test_steps_that_have_to_wait_for_the_host():
    """After another use of the workspace, without graphs, with separate launches, in another segment."""
    atlas = _atlas()
    ar, draft, verify = atlas.get_graph(1, 64, "ar"), atlas.get_graph(9, 64, "draft"), atlas.get_graph(9, 64, "verify")
    far = atlas.get_graph(9, 256, "verify")
    positions = list(range(3, 12))
    assert not atlas.step_ahead(ar)
    atlas.replay(ar, [5], [3], 3)
    atlas.replay(draft, [5] + [999] * 8, positions, 3, 1)
    assert not atlas.step_ahead(ar) and not atlas.step_ahead(draft)
    assert not atlas.verify_drafted(far, draft, 5, positions, 4, 1) and not atlas.verify_drafted(draft, draft, 5, positions, 4, 1)
    with pytest.raises(RuntimeError):
        atlas.verify_drafted(verify, draft, 5, positions, 65, 1)
    with pytest.raises(ValueError):
        atlas.verify_drafted(verify, draft, 5, positions[:3], 4, 1)
    atlas._separate_for = 1
    assert not atlas.verify_drafted(verify, draft, 5, positions, 4, 1) and not atlas.step_ahead(ar)
    atlas.replay(ar, [5], [3], 3)
    assert atlas._separate_for == 0 and not atlas.step_ahead(ar)   # separate launches have not advanced its inputs
    atlas.replay(ar, [5], [3], 3)
    assert atlas.step_ahead(ar) == 1 and atlas.step_ahead(ar, 7) == 4
    atlas.replay(ar, [5], [61], 61)
    assert atlas.step_ahead(ar, 7) == 1   # the segment ends
    kv = atlas.kv(64)
    torch.cuda.synchronize()
    assert atlas.step_ahead(ar, 7) == 1
    atlas.commit_with_next(64, 7, 1)   # is committed before the next step's row replaces it
    row = kv[:, :, :, 64].clone()
    assert atlas.step_ahead(ar, 7) == 1 and torch.equal(atlas.kv(64)[:, :, :, 7], row)
    assert atlas.step_ahead(ar, 7) == 0
    atlas.prefill_prompt(list(range(40)), 64)
    assert not atlas.step_ahead(ar)
    eager = _atlas(use_graphs=False)
    g = eager.get_graph(1, 64, "ar")
    eager.replay(g, [5], [3], 3)
    assert not eager.step_ahead(g)


@pytest.mark.parametrize("width,role", [(1, "ar"), (9, "draft"), (9, "verify"), (32, "ar")])
def test_commits_with_the_next_replay(width, role):
    """The same history as commits of their own, at its first and last slots, one row and all of them, replay after replay."""
    sigma = 64
    atlas = _atlas((sigma, 128))
    g, other = atlas.get_graph(width, sigma, role), atlas.get_graph(9, 128, "verify")
    kv = atlas.kv(sigma)
    gen = torch.Generator(device=DEV).manual_seed(1)
    start = (torch.randn(tuple(kv.shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)
    commits = [(1, 1, 0), (5, width, 0), (sigma - width, width, 0), (sigma - 1, 1, width - 1), (7, max(1, width // 2), width // 2)]
    histories = []
    for commit in (atlas.commit_kv, atlas.commit_with_next):
        kv.copy_(start)
        for i, (at, n, first) in enumerate(commits * 3):
            atlas._separate_for = 1 if i == 7 else 0   # (separate launches for one of them)
            atlas.replay(g, [(3 * i + j) % 1000 for j in range(width)], list(range(2, 2 + width)), 2, 1 if role == "draft" else 0)
            commit(sigma, at, n, first)
            if i % 4 == 3:
                atlas.read_outputs(g)
            if i % 5 == 4:
                atlas.replay(other, list(range(9)), list(range(3, 12)), 4)   # another segment's
        histories.append(atlas.kv(sigma).clone())   # (what is owed is committed when the history is asked for)
        assert atlas._owed is None
    assert torch.equal(*histories) and not torch.equal(histories[0][:, :, :, :sigma], start[:, :, :, :sigma])
    with pytest.raises(RuntimeError):
        atlas.commit_with_next(sigma, sigma - width + 1, width)


@pytest.mark.parametrize("commit", [(64, 0, 0), (64, 0, -1), (-1, 0, 1), (0, -1, 1), (64, 90, 8), (90, 0, 8), (0, 0, 2 ** 31 - 1)])
def test_rows_outside_the_buffer_are_not_committed(commit):
    from bitmtp_amd import decode_ops
    kv = torch.arange(2 * 2 * 2 * 96 * 128, device=DEV).remainder(251).to(torch.bfloat16).view(2, 2, 2, 96, 128)
    before = kv.clone()
    inputs = torch.tensor([10, 9, 1, 2, 3, 3, 4, 5, -1, -2 ** 31, -2 ** 31 + 2] + list(commit), dtype=torch.int32).pin_memory()
    step_in = torch.zeros(11, dtype=torch.int32, device=DEV)
    drafted = torch.tensor([100, 101, 102], dtype=torch.int32, device=DEV)
    decode_ops.step_after(inputs, step_in, drafted, kv)
    assert torch.equal(kv, before) and step_in.tolist() == [10, 9, 1, 2, 3, 3, 4, 5, -1, 100, 102]
    for n in (-5, 0, 65, 2 ** 31 - 1):   # behind a step over no slots, and past the segment
        step_in[0] = n
        decode_ops.step_next(step_in, kv, 64)
        assert torch.equal(kv, before)
    step_in[0] = 64
    decode_ops.step_next(step_in, kv, 64)
    before[:, :, :, 63] = before[:, :, :, 64]
    assert torch.equal(kv, before)


@pytest.mark.parametrize("width,role", [(1, "ar"), (9, "draft"), (12, "draft"), (9, "verify"), (32, "ar")])
def test_results_in_pinned_memory_are_those_on_the_device(width, role):
    atlas = _atlas((64,))
    g = atlas.get_graph(width, 64, role)
    rows = g.logits_end - g.logits_start
    for i in range(4):
        atlas.replay(g, [(i + 7 * j) % 1000 for j in range(width)], list(range(3, 3 + width)), 3, 1 if role == "draft" else 0)
        tokens, conf, accept = atlas.read_outputs(g)
        assert g.io.arrived
        torch.cuda.synchronize()
        out = g.io.out.cpu().numpy()
        assert np.array_equal(tokens, out[:rows]) and accept == out[width]
        assert np.array_equal(conf.view(np.int32), out[width + 2: width + 2 + rows])
        if role == "draft":
            assert np.array_equal(atlas._drafted[:rows].cpu().numpy(), out[:rows])


@pytest.mark.parametrize("loop,kw", [("speculative", {}), ("hybrid", {"threshold": 2.0}), ("hybrid", {"threshold": 2.0, "hybrid_m": 9})])
def test_loops_without_graphs_keep_what_was_verified(loop, kw, monkeypatch):
    """Verifications that accept drafts: the tokens and the history of the loop whose steps are graphs."""
    from bitmtp_amd import generate
    prompt, results = list(range(3, 33)), []
    for use_graphs in (True, False):
        accepted = itertools.cycle((2, 0, 3, 7))   # (random weights agree on few)
        monkeypatch.setattr(generate, "verify_accept", lambda draft, verify, D: next(accepted))
        atlas = _successors((64, 256), use_graphs=use_graphs)
        out, st = getattr(generate, loop + "_generate")(atlas, prompt, max_gen_len=60, **kw)
        results.append((out, st["accepted_drafts"], _history(atlas, len(prompt) + len(out) - 10)))
        assert st["accepted_drafts"] > 9 and len(set(out)) > 2
    assert results[0][:2] == results[1][:2]
    assert torch.equal(results[0][2], results[1][2])


@pytest.mark.parametrize("rows", [1, 9, 32])
def test_inputs_of_a_step_are_all_that_is_written(rows):
    """``step_in`` in the middle of a larger buffer."""
    from bitmtp_amd import decode_ops
    words = 2 + 3 * rows
    inputs = torch.arange(words + 3, dtype=torch.int32)
    inputs[-3:] = 0
    memory = torch.full((words + 64,), -7, dtype=torch.int32, device=DEV)
    kv = torch.zeros(2, 1, 1, 40, 128, dtype=torch.bfloat16, device=DEV)
    decode_ops.step_after(inputs.pin_memory(), memory[32:32 + words], torch.zeros(1, dtype=torch.int32, device=DEV), kv)
    assert torch.equal(memory[32:32 + words].cpu(), inputs[:words])
    assert (memory[:32] == -7).all() and (memory[32 + words:] == -7).all()


def test_rows_are_committed_in_buffers_of_more_than_32_gib():
    """One that the graphs of a long segment have: its last planes, by both launches."""
    from bitmtp_amd import decode_ops
    slots = 240032
    kv = torch.empty(2, 36, 8, slots, 128, dtype=torch.bfloat16, device=DEV)
    rows = torch.arange(2 * 36 * 8 * 2 * 128, device=DEV).remainder(251).to(torch.bfloat16).view(2, 36, 8, 2, 128)
    kv[:, :, :, 240000:240002] = rows
    step_in = torch.zeros(5, dtype=torch.int32, device=DEV)
    inputs = torch.tensor([1, 2, 3, 4, 5, 240000, 239000, 2], dtype=torch.int32).pin_memory()
    decode_ops.step_after(inputs, step_in, torch.zeros(1, dtype=torch.int32, device=DEV), kv)
    assert torch.equal(kv[:, :, :, 239000:239002], rows) and step_in.tolist() == [1, 2, 3, 4, 5]
    step_in[0] = 777
    decode_ops.step_next(step_in, kv, 240000)
    assert torch.equal(kv[:, :, :, 776:777], rows[:, :, :, :1])
    del kv
    torch.cuda.empty_cache()
