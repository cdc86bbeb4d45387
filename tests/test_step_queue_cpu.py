"""The host side of queued steps: ``GraphAtlas`` itself over a device that does what was queued when it is waited for, no sooner.
Which rows become history, and whose results the host reads."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from bitmtp_amd import runtime as R
from bitmtp_amd.model import StepIO

SIGMA, OTHER, D = 64, 128, 8


class Device:
    """Launches in the order they were queued, on streams that an event orders where the program asks for it."""

    def __init__(self):
        self.queue, self.step = [], 0
        self.stream = SimpleNamespace(cuda_stream=1, device_index=0, wait_event=lambda e: None, synchronize=self.run)

    def run(self, until=None):
        while self.queue and (until is None or until in self.queue):
            launch = self.queue.pop(0)
            if callable(launch):
                launch()


class Event:
    def __init__(self, device):
        self.device, self.mark = device, None

    def record(self, stream):
        self.mark = object()
        self.device.queue.append(self.mark)

    def synchronize(self):
        if self.mark in self.device.queue:
            self.device.run(self.mark)


def token_of(step):
    return 100 + step


@pytest.fixture
def device(monkeypatch):
    dev = Device()
    monkeypatch.setattr(R.torch.cuda, "current_stream", lambda d=None: dev.stream)
    monkeypatch.setattr(R.torch.cuda, "synchronize", lambda d=None: dev.run())

    def commit(kv, src, dst, n):
        if min(src, dst) < 0 or max(src, dst) + n > kv.shape[3]:
            raise RuntimeError("bonsai_kv_commit failed")

        def launch():
            kv[:, :, :, dst:dst + n] = kv[:, :, :, src:src + n].clone()
        dev.queue.append(launch)
    monkeypatch.setattr(R.decode_ops, "kv_commit", commit)
    monkeypatch.setattr(R, "_whole_device", R._WholeDevice())
    dev.commit = commit
    return dev


def _atlas(dev):
    atlas = R.GraphAtlas.__new__(R.GraphAtlas)
    atlas.device, atlas.D, atlas.M_max = "cuda:0", D, 32
    atlas.segment_ladder = (SIGMA, OTHER)
    atlas.kv_buffers = {s: torch.zeros(2, 1, 1, s + 32, 1, dtype=torch.int32) for s in atlas.segment_ladder}
    atlas._last = atlas._owed = None
    atlas._last_stream = 0
    atlas.replays = atlas._separate_for = atlas._undisturbed = 0
    atlas._back_off = atlas.BACK_OFF
    atlas.dev = dev
    return atlas


def _graph(atlas, M, sigma, role, captured=True, one_launch=True):
    """As ``GraphAtlas.get_graph`` returns it.  A step leaves its number in its rows of the buffer and ``token_of`` it as its tokens."""
    dev, kv = atlas.dev, atlas.kv_buffers[sigma]
    ls, le = R.logits_rows(role, M, D)
    inputs = torch.zeros(3 * M + 5, dtype=torch.int32)
    io = StepIO(M=M, step_in=torch.zeros(3 * M + 2, dtype=torch.int32), step_in_host=inputs[:3 * M + 2], inputs_host=inputs,
                out=torch.zeros(2 * M + 2, dtype=torch.int32), out_host=torch.zeros(2 * M + 2, dtype=torch.int32), uploaded=Event(dev))
    one = SimpleNamespace(failed=np.zeros(1, dtype=np.int32)) if one_launch else None
    ring = torch.zeros(R.GraphAtlas.RING, dtype=torch.int32) if M == 1 and role == "ar" else None
    g = R.CapturedGraph(graph=None, io=io, M=M, sigma=sigma, role=role, P=M - D, logits_start=ls, logits_end=le, one=one,
                        pending=io.pending(le - ls), ring=ring)

    def layers(outs):
        dev.step += 1
        kv[:, :, :, sigma:sigma + M] = dev.step * 100 + torch.arange(M).view(1, 1, 1, M, 1)
        for out in outs:
            out[:le - ls] = token_of(dev.step)
            out[M:M + 2 + le - ls] = 1
        if ring is not None and len(outs) == 2:   # (a captured one-token step)
            ring[io.step_in[0] % len(ring)] = token_of(dev.step)
            io.step_in[0] += 1

    def replay():
        io.step_in.copy_(io.step_in_host)
        if role != "ar":                          # step_after
            src, dst, n = (int(v) for v in inputs[-3:])
            if n > 0:
                kv[:, :, :, dst:dst + n] = kv[:, :, :, src:src + n].clone()
        layers((io.out, io.out_host))

    def further(steps):
        for _ in range(steps):
            n = int(io.step_in[0])
            kv[:, :, :, n - 1] = kv[:, :, :, sigma].clone()
            layers((io.out, io.out_host))
    if captured:
        g.graph = SimpleNamespace(replay=lambda: dev.queue.append(replay))
        if ring is not None:
            g.next = {n: SimpleNamespace(replay=lambda n=n: dev.queue.append(lambda: further(n))) for n in R.GraphAtlas.AHEAD}
    g._eager = lambda one: dev.queue.append(lambda: layers((io.out,)))
    atlas._one_launch = lambda M: one
    return g


@pytest.mark.parametrize("captured,one_launch", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("M,role", [(1, "ar"), (9, "draft"), (9, "verify"), (16, "draft")])
def test_rows_left_for_the_next_replay_become_history(device, M, role, captured, one_launch):
    """With graphs and without, with steps in one launch and separate ones, by a replay of the same segment or another one: the
    history of commits of their own, by the time that the next step has run."""
    histories = []
    for name in ("commit_kv", "commit_with_next"):
        device.step = 0
        atlas = _atlas(device)
        g = _graph(atlas, M, SIGMA, role, captured, one_launch)
        other = _graph(atlas, 9, OTHER, "verify", captured, one_launch)
        seen = []
        for i in range(9):
            step = other if i % 4 == 2 else g
            atlas._separate_for = 1 if i == 5 else 0
            atlas.replay(step, [i] * step.M, list(range(step.M)), 3, 1 if role == "draft" and step is g else 0)
            device.run()
            seen.append([atlas.kv_buffers[s][:, :, :, :s].clone() for s in atlas.segment_ladder])
            rows = min(step.M, 1 + i % 3)
            getattr(atlas, name)(step.sigma, 4 + 2 * i, rows, min(i % 2, step.M - rows))
        atlas.synchronize()
        seen.append([atlas.kv_buffers[s][:, :, :, :s].clone() for s in atlas.segment_ladder])
        histories.append(seen)
    for i, (want, got) in enumerate(zip(*histories)):
        assert all(torch.equal(*pair) for pair in zip(want, got)), f"behind step {i}"
    assert (histories[0][-1][0] != 0).sum() >= 2 * 6


@pytest.mark.parametrize("sigma,cache_len,n,first_row", [(SIGMA, -1, 1, 0), (SIGMA, 60, 5, 0), (SIGMA, 3, 1, 32),
                                                         (SIGMA, 3, 9, 24), (SIGMA + 1, 3, 1, 0)])
def test_commits_that_cannot_be_are_refused_at_once(device, sigma, cache_len, n, first_row):
    """As a commit of its own refuses them; the one before is still to come."""
    atlas = _atlas(device)
    atlas.commit_with_next(SIGMA, 4, 2, 1)
    with pytest.raises((RuntimeError, KeyError)):
        atlas.commit_with_next(sigma, cache_len, n, first_row)
    atlas.kv_buffers[SIGMA][:, :, :, SIGMA:] = 7
    atlas.synchronize()
    assert atlas._owed is None and (atlas.kv_buffers[SIGMA][:, :, :, :SIGMA].flatten(0, 3) == 7).sum() == 2 * 2


@pytest.mark.parametrize("steps", [1, 4])
def test_results_behind_steps_that_nobody_has_read(device, steps):
    """A replay behind queued steps, one of which has been read: its own token, not one of theirs that is stored late."""
    atlas = _atlas(device)
    g = _graph(atlas, 1, SIGMA, "ar")
    atlas.replay(g, [5], [3], 3)
    first = g.io.uploaded.mark
    assert atlas.step_ahead(g, steps) == steps
    queued = g.io.uploaded.mark
    device.run(first)
    assert atlas.read_step(g, 3) == token_of(1)
    atlas.replay(g, [9], [20], 20)
    device.run(queued)                            # the older steps end now, if they have not by now
    tokens, _, _ = atlas.read_outputs(g)
    assert tokens.tolist() == [token_of(steps + 2)]
    assert device.step == steps + 2


def test_outputs_behind_queued_steps_are_those_of_the_last(device):
    atlas = _atlas(device)
    g = _graph(atlas, 1, SIGMA, "ar")
    atlas.replay(g, [5], [3], 3)
    first = g.io.uploaded.mark
    assert atlas.step_ahead(g) == 1
    device.run(first)
    assert atlas.read_outputs(g)[0].tolist() == [token_of(2)]
    assert atlas.read_step(g, 3) == token_of(1) and atlas.read_step(g, 4) == token_of(2)


def test_no_more_tokens_on_their_way_than_there_are_words_for(device):
    atlas = _atlas(device)
    g = _graph(atlas, 1, OTHER, "ar")
    atlas.replay(g, [5], [3], 3)
    while atlas.step_ahead(g, 7):
        pass
    assert g.at - 3 + 1 == atlas.RING
    for n in range(3, 3 + 2 * atlas.RING):        # each token read makes room for another one
        assert atlas.read_step(g, n) == token_of(n - 2)
        assert atlas.step_ahead(g) == 1
    for n in (2, g.at - atlas.RING, g.at + 1):    # not one of these steps, one whose word is taken, not queued
        with pytest.raises(ValueError):
            atlas.read_step(g, n)


class GivesUpBetween:
    """A step's mark that the device sets between two looks of the host."""

    def __init__(self, looks):
        self.looks, self.value = looks, 0

    def __getitem__(self, i):
        self.looks -= 1
        if self.looks < 0:
            self.value, self.looks = 1, 1 << 30
        return self.value

    def __setitem__(self, i, value):
        self.value = value


@pytest.mark.parametrize("looks", [0, 1, 2, 3])
@pytest.mark.parametrize("role", ["ar", "verify"])
def test_no_step_goes_as_one_launch_once_another_was_seen_to_give_up(device, role, looks):
    atlas = _atlas(device)
    draft = _graph(atlas, 9, SIGMA, "draft")
    g = _graph(atlas, 1 if role == "ar" else 9, SIGMA, role)
    queued = 0
    for i in range(6):
        if i == 1:
            g.one.failed = GivesUpBetween(looks)
        if role == "ar":
            atlas.replay(g, [5], [3], 3)
            ahead = atlas._separate_for == 0 and atlas.step_ahead(g)
        else:
            atlas.replay(draft, [5] * 9, list(range(9)), 3, 1)
            ahead = atlas.verify_drafted(g, draft, 5, list(range(9)), 4, 1)
        assert not ahead or atlas._separate_for == 0
        queued += bool(ahead)
        device.run()
    assert queued < 6 and atlas._back_off == 2 * atlas.BACK_OFF


@pytest.mark.parametrize("draft_one,verify_one", [(True, True), (True, False), (False, True), (False, False)])
def test_a_verification_on_another_stream_waits_for_its_draft(device, draft_one, verify_one):
    atlas = _atlas(device)
    draft, g = _graph(atlas, 16, SIGMA, "draft", one_launch=draft_one), _graph(atlas, 9, SIGMA, "verify", one_launch=verify_one)
    waits = []
    for other in (device.stream, SimpleNamespace(cuda_stream=2, device_index=0, wait_event=waits.append)):
        first = device.stream
        atlas.replay(draft, [5] * 16, list(range(16)), 3, 1)
        device.stream = other
        assert atlas.verify_drafted(g, draft, 5, list(range(9)), 4, 1)
        device.run()
        assert (draft.io.uploaded in waits) == (other is not first)
