"""The generation loops on a symbolic atlas (tests/symbolic_atlas.py): every replay predicts
from exactly the KV slots the real step descriptor makes visible, so the loops' bookkeeping
(pending rows, commits from draft and verify workspaces, anchors, segment migration) is
checked on the CPU against the toy model's greedy continuation.  The invariants are the
reference's: speculation with a strict verifier reproduces greedy AR token for token
(docs/testing.md:13, fast_generate.py:611-657), accounting identities
(fast_generate.py:1151-1162), confidence decoding commits the drafter's confident prefix
(fast_generate.py:354-386)."""
import pytest

from bitmtp_amd import generate as G
from symbolic_atlas import MASK, VOCAB, SymbolicAtlas, greedy

PROMPTS = [list(range(5, 5 + n)) for n in (1, 7, 31, 32, 33, 70)]


@pytest.mark.parametrize("prompt", PROMPTS, ids=lambda p: f"prompt{len(p)}")
def test_ar_loop_reproduces_the_greedy_continuation(prompt):
    atlas = SymbolicAtlas()
    out, st = G.ar_generate(atlas, prompt, max_gen_len=40)
    assert out == greedy(prompt, 40)
    assert st["decode_tokens"] == 40 and st["timed_decode_tokens"] == 39 and st["n_iters"] == 40


@pytest.mark.parametrize("wrong_every", [0, 2, 3, 5])
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("prompt", PROMPTS[1:5], ids=lambda p: f"prompt{len(p)}")
def test_speculative_and_hybrid_loops_reproduce_greedy(prompt, exact, wrong_every):
    want = greedy(prompt, 57)
    for fn, kw in ((G.speculative_generate, {}), (G.hybrid_generate, {"threshold": 0.9}),
                   (G.hybrid_generate, {"threshold": 0.9, "hybrid_m": 2})):
        atlas = SymbolicAtlas(wrong_every=wrong_every)
        out, st = fn(atlas, prompt, max_gen_len=57, exact_m1_verify=exact, **kw)
        if fn is G.speculative_generate or wrong_every == 0:
            assert out == want, (fn.__name__, kw)
        else:
            # the confidence path commits unverified drafts: with a drafter that is wrong
            # only where its confidence is low they are still the greedy tokens
            assert out == want, (fn.__name__, kw)
        assert st["draft_iters"] == st["n_conf_path"] + st["n_verify_path"]
        assert st["decode_tokens"] == 1 + st["accepted_drafts"] + st["verifier_bonus_tokens"] == 57
        assert st["drafted_tokens"] == 8 * st["draft_iters"]
        if fn is G.speculative_generate:
            assert st["n_conf_path"] == 0
        if wrong_every == 0 and not exact:
            # a perfect drafter: every verified iteration commits D drafts + 1 bonus
            assert st["committed_per_iter"] > 7.0


def test_hybrid_takes_the_confidence_path_when_the_chain_is_long_enough():
    prompt = list(range(3, 20))
    atlas = SymbolicAtlas(wrong_every=0)
    out, st = G.hybrid_generate(atlas, prompt, threshold=0.9, max_gen_len=64)
    assert out == greedy(prompt, 64)
    assert st["n_conf_path"] > 0 and st["n_verify_path"] == 0 and st["verifier_bonus_tokens"] == 0
    # pending rows of a confidence iteration: the whole committed block is re-forwarded
    widths = {m for role, m in atlas.log if role == "draft"}
    assert 16 in widths
    # a drafter that misses every second position never builds a chain of six
    atlas = SymbolicAtlas(wrong_every=2)
    out, st = G.hybrid_generate(atlas, prompt, threshold=0.9, max_gen_len=40)
    assert out == greedy(prompt, 40) and st["n_conf_path"] == 0


@pytest.mark.parametrize("wrong_every", [0, 3])
def test_confidence_loop(wrong_every):
    prompt = list(range(9, 30))
    atlas = SymbolicAtlas(wrong_every=wrong_every)
    out, st = G.confidence_generate(atlas, prompt, threshold=0.9, max_gen_len=50)
    # the drafter is wrong only where its confidence is low, so the committed prefix of every
    # block is the greedy continuation
    assert out == greedy(prompt, 50)
    assert st["n_verify_path"] == 0 and st["conf_path_frac"] == 1.0
    assert st["decode_tokens"] == 50 and st["timed_decode_tokens"] == 50 - st["untimed_output_tokens"]
    if wrong_every == 0:
        assert st["n_iters"] == 7 and st["untimed_output_tokens"] == 8
    else:
        assert st["n_iters"] > 7


def test_eos_and_length_limits():
    prompt = list(range(2, 25))
    want = greedy(prompt, 64)
    eos = want[20]
    cut = want.index(eos)
    for fn, kw in ((G.ar_generate, {}), (G.speculative_generate, {}), (G.hybrid_generate, {}),
                   (G.confidence_generate, {})):
        atlas = SymbolicAtlas(wrong_every=0)
        out, st = fn(atlas, prompt, max_gen_len=64, eos_ids=[eos], **kw)
        assert out == want[:cut], fn.__name__
        out, st = fn(SymbolicAtlas(wrong_every=3), prompt, max_gen_len=13, **kw)
        assert out == want[:13] and st["decode_tokens"] == 13, fn.__name__


def test_long_generation_migrates_between_segments():
    prompt = list(range(1, 41))
    want = greedy(prompt, 300)
    for fn in (G.ar_generate, G.speculative_generate, G.hybrid_generate, G.confidence_generate):
        atlas = SymbolicAtlas(segment_ladder=(64, 128, 512), wrong_every=4)
        # start in a segment the run outgrows: force it by asking for few tokens first
        out, st = fn(atlas, prompt, max_gen_len=300)
        assert out == want, fn.__name__
    # a run that starts in the smallest segment and has to move twice
    for fn in (G.ar_generate, G.speculative_generate, G.hybrid_generate, G.confidence_generate):
        atlas = SymbolicAtlas(segment_ladder=(64, 128, 512), wrong_every=4)
        real_select, calls = atlas.select_segment, []

        def select(needed):
            calls.append(needed)
            # the first placement pretends that the run is short; later ones ask for little
            # more than the live history, as after an under-estimated generation length
            return 64 if len(calls) == 1 else real_select(needed - 60)
        atlas.select_segment = select
        out, _ = fn(atlas, prompt, max_gen_len=300)
        assert out == want, fn.__name__
        assert len(calls) >= 3, fn.__name__
    assert MASK > VOCAB


class QueueingAtlas(SymbolicAtlas):
    """Steps queued before the results of the one in front of them are read, as ``GraphAtlas`` queues them; every third one has
    to wait for the host."""
    RING = 8

    def __init__(self, *args, refuses=3, **kw):
        super().__init__(*args, **kw)
        self.refuses, self.asked, self.ring, self.last = refuses, 0, {}, None

    def _refused(self):
        self.asked += 1
        return self.refuses and self.asked % self.refuses == 0

    owed = None

    def commit_with_next(self, *what, **more):
        self.settle()
        self.owed = what, more

    def settle(self):
        what, self.owed = self.owed, None
        if what is not None:
            super().commit_kv(*what[0], **what[1])

    def commit_kv(self, *args, **kw):
        self.settle()
        return super().commit_kv(*args, **kw)

    def migrate_segment(self, *args):
        self.settle()
        return super().migrate_segment(*args)

    def synchronize(self):
        self.settle()

    def replay(self, g, tokens, positions, cache_len, n_pend=0):
        self.settle()
        super().replay(g, tokens, positions, cache_len, n_pend)
        self.last = g
        if g.M == 1:
            g.at = cache_len
            self.ring[cache_len % self.RING] = int(g.out[0][0])

    def step_ahead(self, g, most=1):
        if self.last is not g or most < 1 or self._refused():
            return 0
        steps = 4 if most >= 4 else 1
        for _ in range(steps):
            self.commit_kv(g.sigma, g.at, 1)
            self.replay(g, [self.ring[g.at % self.RING]], [g.at + 1], g.at + 1)
        return steps

    def read_step(self, g, cache_len):
        assert 0 <= g.at - cache_len <= 4
        return self.ring[cache_len % self.RING]

    def verify_drafted(self, g, drafted, anchor, positions, cache_len, n_pend):
        if self.last is not drafted or self._refused():
            return False
        assert self.owed is None
        self.commit_kv(g.sigma, cache_len - n_pend, n_pend)
        super().replay(g, [anchor] + [int(t) for t in drafted.out[0][: g.M - 1]], positions, cache_len)
        self.last = g
        return True


@pytest.mark.parametrize("refuses", [0, 1, 3])
@pytest.mark.parametrize("prompt", PROMPTS + [list(range(5, 5 + 200))], ids=lambda p: f"prompt{len(p)}")
def test_steps_queued_before_the_results_are_read(prompt, refuses):
    """The same tokens, histories and accounting, across segments and up to the end of the longest, with and without an end-of-text
    token, behind which one step more may have run."""
    for fn, kw in ((G.ar_generate, {}), (G.speculative_generate, {}), (G.hybrid_generate, {"threshold": 0.9}),
                   (G.hybrid_generate, {"threshold": 0.9, "hybrid_m": 9})):
        ladder = (64, 128, 256)
        for length in (1, 2, 9, 45, 300):
            for eos in ((), greedy(prompt, 20)[17:18]):
                plain, queued = SymbolicAtlas(segment_ladder=ladder), QueueingAtlas(segment_ladder=ladder, refuses=refuses)
                results = []
                for atlas in (plain, queued):
                    try:
                        results.append(fn(atlas, prompt, max_gen_len=length, eos_ids=eos, **kw))
                    except (AssertionError, RuntimeError) as e:   # no room left: in both
                        results.append(type(e))
                if isinstance(results[0], type):
                    assert results[0] is results[1]
                    continue
                (want, st), (got, sq) = results
                assert got == want and {k: v for k, v in st.items() if "time" not in k and k != "ttft"} == \
                    {k: v for k, v in sq.items() if "time" not in k and k != "ttft"}
                assert len(queued.log) - len(plain.log) in ((0, 1) if eos and fn is G.ar_generate else (0,))
                assert queued.owed is None
                for s in ladder:   # history: all that was committed
                    held = len(prompt) + len(want) - 1
                    assert queued.kv[s][:min(s, held)] == plain.kv[s][:min(s, held)]
