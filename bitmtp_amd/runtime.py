"""HIP-graph atlas with shared per-segment KV history and workspace, the MI355X
counterpart of the reference ``GraphAtlas`` (src/bonsai_sft/gpu/fast_runtime.py:76-521).

Graphs are keyed by ``(M, sigma, role)``.  Each segment sigma owns one KV buffer
``[2, n_layers, n_kv, sigma + M_max, 128]``: slots ``[0, sigma)`` are history, the
captured step always writes its M new rows at slot ``sigma`` (so the graph does not
depend on ``cache_len``), and accepted rows are copied down into history afterwards.

Differences from the reference, by design:

* the additive mask tensor ``[1, 1, M, sigma+M]`` and its per-step rebuild
  (fast_runtime.py:391-465) are replaced by a ``2 + M`` word descriptor
  (``cache_len``, one hidden history slot, one workspace-visibility word per row) that
  the attention kernel evaluates, so attention reads ``cache_len + M`` slots instead
  of ``sigma + M``;
* tokens, positions and the descriptor travel in one host-to-device copy per replay and
  argmax / confidence are stored to pinned memory by its last launch;
* a greedy step can be queued behind the one before it, and a verifying block behind its draft, before the host has seen
  their results (``step_ahead``, ``verify_drafted``);
* intermediate buffers are shared by all graphs; graphs are captured on first use.
"""
from __future__ import annotations

import gc
import threading
import time
from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np

import torch

from . import contracts, decode_ops, ops
from .model import (PROMPT_BLOCK_MAX, BonsaiDecoder, PromptBuffers, StepIO, Workspace, enqueue_prompt_block,
                    enqueue_step, project_rows, rope_tables, step_one)

DEFAULT_SEGMENT_LADDER = (256, 1024, 4096)
DEFAULT_M_SET = (1, 8, 9, 10, 12, 16, 17)
ROLES = ("draft", "verify", "ar")


# ---------------------------------------------------------------------------
# Visibility descriptors (host side, pure Python: unit-tested without a GPU)
# ---------------------------------------------------------------------------
def _as_int32(mask: int) -> int:
    """A 32-bit visibility word as the signed value an int32 buffer holds (bit 31 = row 31)."""
    mask &= 0xFFFFFFFF
    return mask - (1 << 32) if mask >= (1 << 31) else mask


def draft_row_masks(M: int, D: int, n_pend: int) -> List[int]:
    """Workspace visibility of a draft step (reference template:
    ``_build_mask_template``, fast_runtime.py:345-372).

    Rows ``[0, n_pend)`` are the pending committed tokens (row r sees workspace rows
    0..r); rows ``[n_pend, P)`` are padding; rows ``[P, M)`` are the block (anchor +
    D-1 masks): block-causal among themselves, and they see the pending rows except
    the last one, which the anchor repeats.
    """
    P = M - D
    if P < 0 or not 0 <= n_pend <= P:
        raise ValueError(f"draft width {M} cannot carry {n_pend} pending rows with D={D}")
    masks = [0] * M
    for r in range(n_pend):
        masks[r] = (1 << (r + 1)) - 1
    earlier = (1 << (n_pend - 1)) - 1 if n_pend > 1 else 0
    for r in range(P, M):
        block = ((1 << (r - P + 1)) - 1) << P
        masks[r] = block | earlier
    return [_as_int32(m) for m in masks]


def causal_row_masks(M: int) -> List[int]:
    """AR-causal workspace visibility of verify / AR steps: row r sees rows 0..r
    (reference: ``_build_verify_templates``, fast_runtime.py:423-441)."""
    return [_as_int32((1 << (r + 1)) - 1) for r in range(M)]


# output projection of each role: the backbone's own ("native"), the FP8 or the raw bf16
# approximation for the acceptance-tolerant draft roles (fast_runtime.py:179-203)
DRAFT_ROLES = ("draft", "draft_fp8", "draft_bf16")
HEAD_MODE_OF_ROLE = {"ar": "native", "verify": "native", "draft": "native",
                     "draft_fp8": "fp8", "draft_bf16": "bf16_raw"}


def step_descriptor(role: str, M: int, D: int, cache_len: int, n_pend: int = 0) -> List[int]:
    """``[cache_len, hide, rowmask_0 .. rowmask_{M-1}]`` for one replay
    (reference: ``prepare_step`` / ``_prepare_verify``, fast_runtime.py:391-421,443-465)."""
    if role in DRAFT_ROLES:  # the three draft roles share the mask
        P = M - D
        n_clamp = max(0, min(n_pend, P))
        hide = cache_len - 1 if (n_clamp == 0 and cache_len > 0) else -1
        return [cache_len, hide] + draft_row_masks(M, D, n_clamp)
    if role == "ar":
        return [cache_len, -1] + causal_row_masks(M)
    if role == "verify":
        if cache_len <= 0:
            raise RuntimeError("batched verifier requires a committed anchor")
        # row 0 replays the anchor that already sits at history slot cache_len-1
        return [cache_len, cache_len - 1] + causal_row_masks(M)
    raise ValueError(f"unsupported graph role: {role!r}")


def dense_visibility(desc: Sequence[int], M: int, sigma: int) -> np.ndarray:
    """Boolean ``[M, sigma+M]`` form of a descriptor (what the reference keeps as an
    additive 0 / -inf mask); used by tests and debugging only."""
    cache_len, hide = desc[0], desc[1]
    vis = np.zeros((M, sigma + M), dtype=bool)
    vis[:, :cache_len] = True
    if hide >= 0:
        vis[:, hide] = False
    for r in range(M):
        for j in range(M):
            if (desc[2 + r] >> j) & 1:
                vis[r, sigma + j] = True
    return vis


def logits_rows(role: str, M: int, D: int) -> Tuple[int, int]:
    """Rows projected through the head (reference: ``_capture_one``, fast_runtime.py:179-203)."""
    if role == "ar":
        return 0, M
    if role in DRAFT_ROLES:
        return M - D, M
    if role == "verify":
        return 0, min(D + 1, M)
    raise ValueError(f"unsupported graph role: {role!r}")


# ---------------------------------------------------------------------------
@dataclass
class CapturedGraph:
    graph: "torch.cuda.CUDAGraph"
    io: StepIO
    M: int
    sigma: int
    role: str
    P: int
    logits_start: int
    logits_end: int
    one: Optional[decode_ops.StepOne] = None            # its layers are one launch
    pending: Optional[np.ndarray] = None                # the pinned results while they are waited for
    # of one-token steps: graphs of so many steps behind the last one, and the pinned words their tokens go to, by history length
    next: Optional[Dict[int, "torch.cuda.CUDAGraph"]] = None
    ring: Optional[torch.Tensor] = None
    at: int = 0                                         # history length of the last of them
    ahead: int = 0                                      # how many of them since the last replay
    read: int = 0                                       # history length of the last step whose token the host has read


class _WholeDevice:
    """Steps in one launch need every compute unit of a device.  Two of them on two streams would each get some and wait for
    the rest until both give up, so a step waits, on its stream, for the last one of another stream."""

    def __init__(self):
        self.lock = threading.Lock()
        self.last: Dict[int, Tuple[int, "torch.cuda.Event"]] = {}   # device: stream, what is recorded behind the step

    def launch(self, stream: "torch.cuda.Stream", done: "torch.cuda.Event", step, *args) -> None:
        """``step(*args)``, which queues a step on ``stream`` and records ``done`` behind it."""
        with self.lock:
            last = self.last.get(stream.device_index)
            if last is not None and last[0] != stream.cuda_stream:
                stream.wait_event(last[1])
            step(*args)
            self.last[stream.device_index] = (stream.cuda_stream, done)


_whole_device = _WholeDevice()


class GraphAtlas:
    """Captured decode steps keyed by ``(M, sigma, role)`` over shared KV."""

    def __init__(self, model: BonsaiDecoder,
                 segment_ladder: Tuple[int, ...] = DEFAULT_SEGMENT_LADDER,
                 m_set: Tuple[int, ...] = DEFAULT_M_SET,
                 roles: Tuple[str, ...] = ROLES,
                 threshold: float = 0.9,
                 prefill_width: int = 32,
                 use_graphs: bool = True):
        contracts.validate_graph_roles(roles)
        self.model = model
        self.args = model.args
        self.device = model.device
        self.segment_ladder = tuple(sorted(set(segment_ladder)))
        self.m_set = tuple(sorted(set(m_set)))
        self.roles = tuple(roles)
        self.D = self.args.block_size
        self.prefill_width = int(prefill_width)
        self.M_max = max(max(self.m_set), self.prefill_width)
        if self.M_max > decode_ops.MAX_WIDTH:
            raise ValueError(f"widths above {decode_ops.MAX_WIDTH} are not supported")
        self.threshold = float(threshold)
        self.use_graphs = bool(use_graphs)
        ops.init_kernels()
        self.kv_buffers: Dict[int, torch.Tensor] = {}
        max_slots = self.segment_ladder[-1] + self.M_max
        # the approximate draft projections are prepared once, like the reference does in
        # GraphAtlas.__init__ (fast_runtime.py:112-118)
        if "draft_fp8" in self.roles:
            contracts.validate_graph_roles(self.roles, torch.cuda.get_device_capability(self.device))
            model.prepare_fp8_lm_head()
        if "draft_bf16" in self.roles:
            model.prepare_raw_bf16_head()
        self.workspace = Workspace(self.args, self.M_max, max_slots, model.head_rows, self.device,
                                   logits_ld_max=model.max_logits_ld())
        self.rope = rope_tables(self.args, max_slots, self.device)
        self.graphs: Dict[Tuple[int, int, str], CapturedGraph] = {}
        self._prompt: Optional[PromptBuffers] = None   # sized by the longest block so far
        self._positions: Optional[torch.Tensor] = None
        self._drafted = torch.zeros(max(self.M_max, self.D), dtype=torch.int32, device=self.device)   # the last draft's tokens
        self._last: Optional[CapturedGraph] = None   # whose replay was the last use of the workspace, as a graph,
        self._last_stream = 0                        # .. and on which stream
        self._owed: Optional[Tuple[int, int, int, int]] = None   # segment, first row, cache_len, rows: see commit_with_next
        self.replays = 0
        # steps of one token and of up to sixteen as one launch (model.step_one), with the weights of the last capture or,
        # without graphs, of the last step
        self._one = self._block = None
        # Such a launch that does not get the whole device has its step done again behind it, the slow way.  It says so, and
        # then the separate launches stay for a while, twice as long every time until the one launch has run undisturbed again.
        self._separate_for = 0                  # replays that keep to the separate launches
        self._back_off = self.BACK_OFF
        self._undisturbed = 0                   # replays as one launch since

    #: replays with separate launches after a step that did not get the whole device
    BACK_OFF = 64
    #: tokens of one-token steps that the host has not read yet, at most
    RING = 16
    #: steps that a graph queues at once behind another (14 us pass between two graphs)
    AHEAD = (4, 1)

    def synchronize(self) -> None:
        """Wait for everything queued on the atlas's device (the loops' timing fences)."""
        self.settle()
        torch.cuda.synchronize(self.device)

    # -- KV ------------------------------------------------------------------
    def kv(self, sigma: int) -> torch.Tensor:
        """Shared buffer of segment sigma, allocated on first use
        (reference: ``_allocate_shared_kv``, fast_runtime.py:130-138)."""
        self.settle()
        buf = self.kv_buffers.get(sigma)
        if buf is None:
            if sigma not in self.segment_ladder:
                raise KeyError(f"segment {sigma} is not in the ladder {self.segment_ladder}")
            buf = torch.zeros(2, self.args.n_layers, self.args.n_kv_heads, sigma + self.M_max,
                              self.args.head_dim, device=self.device, dtype=torch.bfloat16)
            self.kv_buffers[sigma] = buf
        return buf

    def select_segment(self, needed_kv_len: int) -> int:
        """Smallest sigma >= needed_kv_len, else the largest (fast_runtime.py:377-386)."""
        for sigma in self.segment_ladder:
            if needed_kv_len <= sigma:
                return sigma
        return self.segment_ladder[-1]

    def commit_kv(self, sigma: int, cache_len: int, n_accept: int, first_row: int = 0) -> None:
        """Workspace rows ``first_row .. first_row+n_accept-1`` become history rows
        ``cache_len ..`` (``commit_kv`` with first_row 0, ``commit_kv_from_verify`` with
        first_row 1; fast_runtime.py:467-508)."""
        if n_accept <= 0:
            return
        if cache_len + n_accept > sigma:
            raise RuntimeError("KV commit would run past the history segment")
        decode_ops.kv_commit(self.kv(sigma), sigma + first_row, cache_len, n_accept)

    def commit_with_next(self, sigma: int, cache_len: int, n_accept: int, first_row: int = 0) -> None:
        """``commit_kv``, by the first launch of the next replay where that reads the segment's inputs anyway (blocks).  Whoever asks
        the atlas for the history before, or waits for it (``kv``, ``synchronize``, ``settle``), has it committed first; a tensor
        that ``kv`` returned earlier is behind until then."""
        if n_accept <= 0:
            return
        if sigma not in self.kv_buffers or not 0 <= cache_len <= sigma - n_accept or not 0 <= first_row <= self.M_max - n_accept:
            return self.commit_kv(sigma, cache_len, n_accept, first_row)   # (refuses what cannot be)
        self.settle()
        self._owed = (sigma, first_row, cache_len, n_accept)

    def settle(self) -> None:
        """Commit what ``commit_with_next`` has left for the next replay."""
        owed, self._owed = self._owed, None
        if owed is not None:
            sigma, first_row, cache_len, n_accept = owed
            decode_ops.kv_commit(self.kv_buffers[sigma], sigma + first_row, cache_len, n_accept)

    def migrate_segment(self, src_sigma: int, dst_sigma: int, cache_len: int) -> None:
        """Copy live history to another segment's buffer (fast_runtime.py:510-521)."""
        if src_sigma == dst_sigma:
            return
        self.kv(dst_sigma)[:, :, :, :cache_len].copy_(self.kv(src_sigma)[:, :, :, :cache_len])

    # -- graphs --------------------------------------------------------------
    def get_graph(self, M: int, sigma: int, role: str) -> CapturedGraph:
        key = (M, sigma, role)
        g = self.graphs.get(key)
        if g is None:
            g = self._capture_one(M, sigma, role)
            self.graphs[key] = g
        return g

    def capture_all(self) -> None:
        """Capture every (M, sigma, role) the reference captures up front
        (``_capture_all``, fast_runtime.py:154-169)."""
        for sigma in self.segment_ladder:
            for M in self.m_set:
                if M == 1:
                    if "ar" in self.roles:
                        self.get_graph(1, sigma, "ar")
                    continue
                for role in self.roles:
                    if role == "ar" or (role in DRAFT_ROLES and M < self.D) or \
                            (role == "verify" and M != self.D + 1):
                        continue
                    self.get_graph(M, sigma, role)

    def _capture_one(self, *what) -> CapturedGraph:
        """``what``: the arguments of ``_capture_one_impl``."""
        # The cyclic garbage collector must not run while a stream is capturing: if it finds
        # an unreachable atlas, it destroys that atlas's graphs in the middle of this capture,
        # which aborts the process.  Collect first, then keep the collector off until the
        # capture has ended.  (Capture keeps process-wide state tensors; they must not become
        # inference tensors, hence inference_mode(False).)
        gc.collect()
        gc_was_enabled = gc.isenabled()
        gc.disable()
        try:
            with torch.inference_mode(False):
                return self._capture_one_impl(*what)
        finally:
            if gc_was_enabled:
                gc.enable()

    def _one_launch(self, M: int) -> Optional[decode_ops.StepOne]:
        """What runs the layers of an M-row step of the model, as its weights are now, in one launch."""
        if M > decode_ops.StepBlock.MAX_ROWS:
            return None
        have = self._one if M == 1 else self._block
        one = step_one(self.model, decode_ops.StepOne if M == 1 else decode_ops.StepBlock, have)
        if have is not None and one is not have and not self.use_graphs:
            torch.cuda.synchronize(self.device)   # steps that read the old weights and their table are still queued
        if M == 1:
            self._one = one
        else:
            self._block = one
        return one

    def _capture_one_impl(self, M: int, sigma: int, role: str) -> CapturedGraph:
        self._last = None
        if role not in contracts.GRAPH_ROLES:
            raise ValueError(f"unsupported graph role: {role!r}")
        if role not in self.roles:
            raise RuntimeError(f"graph role {role!r} was not requested for this atlas")
        if role in DRAFT_ROLES and M < self.D:
            raise ValueError(f"a draft graph needs M >= D = {self.D}")
        if M > self.M_max:
            raise ValueError(f"width {M} exceeds the atlas maximum {self.M_max}")
        ls, le = logits_rows(role, M, self.D)
        io = StepIO.allocate(M, self.device)
        kv = self.kv(sigma)
        # a harmless valid descriptor for the warm-up / capture launches
        desc = step_descriptor("ar", M, self.D, 0)
        io.step_in_host[: 2 + M] = torch.tensor(desc, dtype=torch.int32)
        io.step_in.copy_(io.step_in_host)

        # the closure holds the pieces, not the atlas: no reference cycle through the graphs
        model, workspace, rope, threshold = self.model, self.workspace, self.rope, self.threshold
        if self.use_graphs:   # what is captured reads these tensors for good
            model = model.snapshot()
        head_mode = HEAD_MODE_OF_ROLE[role]
        one = self._one_launch(M)

        def run(one, also=None):
            enqueue_step(model, workspace, io, kv, sigma, rope, ls, le, threshold,
                         head_mode=head_mode, one=one, also=also)

        goes_on = M == 1 and role == "ar"
        ring = torch.zeros(self.RING, dtype=torch.int32).pin_memory() if goes_on else None
        drafted = self._drafted
        graph = graph_next = None
        if self.use_graphs:
            side = torch.cuda.Stream(device=self.device)
            side.wait_stream(torch.cuda.current_stream(self.device))
            with torch.cuda.stream(side):   # warm-up outside capture: lazy library set-up happens here
                warm = torch.cuda.Event()
                _whole_device.launch(side, warm, lambda: (run(one), warm.record(side)))
            torch.cuda.current_stream(self.device).wait_stream(side)
            torch.cuda.synchronize(self.device)
            # the graph carries its own upload of the step inputs and stores the results to the
            # pinned mirror: a replay is one launch call on the host
            also = io.also_to(**(dict(step=io.step_in, ring=ring) if goes_on else dict(tokens=drafted) if role in DRAFT_ROLES else {}))
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                if role == "ar":
                    io.step_in.copy_(io.step_in_host, non_blocking=True)
                else:
                    decode_ops.step_after(io.inputs_host, io.step_in, drafted, kv)
                run(one, also)
            if goes_on:
                graph_next = {}
                for steps in self.AHEAD:
                    graph_next[steps] = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(graph_next[steps]):
                        for _ in range(steps):
                            decode_ops.step_next(io.step_in, kv, sigma)
                            run(one, also)
        cg = CapturedGraph(graph=graph, io=io, M=M, sigma=sigma, role=role, P=M - self.D, logits_start=ls, logits_end=le, one=one,
                           pending=io.pending(le - ls), next=graph_next, ring=ring)
        cg._eager = run
        return cg

    # -- prompts -------------------------------------------------------------
    def prefill_prompt(self, prompt: Sequence[int], sigma: int) -> int:
        """Materialise a prompt's KV in segment sigma, in blocks of up to ``PROMPT_BLOCK_MAX`` rows, and return
        the token after it.  A block reads every weight once and projects its last row only; the replayed
        graphs do both for every ``prefill_width`` rows."""
        n = len(prompt)
        if n > sigma:
            raise RuntimeError("history does not fit the segment")
        kv = self.kv(sigma)
        self._last = None
        block = min(n, PROMPT_BLOCK_MAX)
        with torch.inference_mode(False), torch.cuda.device(self.device):
            if self._prompt is None or self._prompt.rows < block:
                self._prompt = None
                self._prompt = PromptBuffers(self.args, min(-(-block // 256) * 256, PROMPT_BLOCK_MAX), self.device)
            if self._positions is None:
                self._positions = torch.arange(self.rope[0].shape[0], dtype=torch.int32, device=self.device)
                self._prompt_out = torch.zeros(4, dtype=torch.int32, device=self.device)
            buffers, out = self._prompt, self._prompt_out
            tokens = torch.from_numpy(np.asarray(prompt, dtype=np.int32)).to(self.device)
            for base in range(0, n, block):
                m = min(block, n - base)
                cur = enqueue_prompt_block(self.model, buffers, tokens[base: base + m], base,
                                           self._positions[base: base + m], kv, self.rope)
            last = m - 1
            project_rows(self.model, self.workspace, buffers.proj[last: m], buffers.h[cur][last: m], 1, self.threshold,
                         out[:1], out[1:2].view(torch.float32), out[2:4])
            return int(out[0].item())

    # -- one replay ----------------------------------------------------------
    def replay(self, g: CapturedGraph, tokens: Sequence[int], positions: Sequence[int],
               cache_len: int, n_pend: int = 0) -> None:
        """Upload tokens, positions and the visibility descriptor, then replay."""
        M = g.M
        if len(tokens) != M or len(positions) != M:
            raise ValueError("tokens / positions must have exactly M entries")
        if cache_len + M > g.sigma + M or cache_len > g.sigma:
            raise RuntimeError("history does not fit the segment")
        inputs = step_descriptor(g.role, M, self.D, cache_len, n_pend) + list(positions) + list(tokens)
        if g.graph is None and g.one is not None:
            g.one = self._one_launch(M)
        separate = g.one is None or self._keeps_separate(g.one)
        # the previous upload from this pinned buffer must have left the host first (as it has where results came back), and
        # steps behind the previous replay store their results where this one's are waited for
        if not g.io.arrived or g.ahead:
            g.io.uploaded.synchronize()
        g.io.step_in_host.numpy()[:] = inputs
        owed = self._owed
        # (only the first launch of a captured block reads the words behind the inputs)
        if separate or g.graph is None or g.role == "ar" or owed is None or owed[0] != g.sigma:
            self.settle()
            g.io.inputs_host.numpy()[-1] = 0
        else:
            self._owed = None
            g.io.inputs_host.numpy()[-3:] = (owed[0] + owed[1], owed[2], owed[3])
        self._queue(g, separate)

    def _queue(self, g: CapturedGraph, separate: bool) -> None:
        stream = torch.cuda.current_stream(self.device)
        g.io.arrived = False
        g.ahead = 0
        if separate:
            self._launch(g, stream, None)
        else:
            _whole_device.launch(stream, g.io.uploaded, self._launch, g, stream, g.one)
        self.replays += 1

    # -- steps behind steps that the host has not seen the results of -----------
    def _behind(self, g: CapturedGraph) -> bool:
        """Whether a step of ``g`` can be queued without its inputs: as the graph of one launch, which separate launches do not stand
        in for."""
        return g.graph is not None and g.one is not None and self._separate_for == 0 and not self._gave_up(g.one)

    def step_ahead(self, g: CapturedGraph, most: int = 1) -> int:
        """Queue one-token steps behind the last one of ``g``, up to ``most``, each on the token of the one before it and with that
        one's row committed.  Returns how many; 0 where the step has to wait for the host (``replay``), or the host for a token: there is
        room for ``RING`` that ``read_step`` has not read."""
        most = min(most, g.sigma - g.at, self.RING - (g.at - g.read))   # (each commits a row first)
        if g.next is None or self._last is not g or most < 1 or not self._behind(g):
            return 0
        self.settle()
        self._as_one_launch()
        steps = max(n for n in self.AHEAD if n <= most)
        for _ in range(steps):
            g.at += 1
            g.ring.numpy()[g.at % self.RING] = StepIO.PENDING
        g.ahead += steps
        stream = torch.cuda.current_stream(self.device)

        def launch():
            g.next[steps].replay()
            g.io.uploaded.record(stream)

        _whole_device.launch(stream, g.io.uploaded, launch)
        self.replays += steps
        return steps

    def read_step(self, g: CapturedGraph, cache_len: int) -> int:
        """The token of the step of ``g`` over ``cache_len`` slots, once it has arrived."""
        if not g.at - g.ahead <= cache_len <= g.at or cache_len <= g.at - self.RING:
            raise ValueError(f"no step over {cache_len} slots is waited for")
        g.read = max(g.read, cache_len)
        word = cache_len % self.RING
        ring = g.ring.numpy()
        deadline = time.perf_counter() + 0.05
        while ring[word] == StepIO.PENDING:
            if time.perf_counter() > deadline:
                g.io.uploaded.synchronize()
                break
        if g.one is not None and g.one.failed[0] > 1:
            raise RuntimeError("a decode step did not end")
        return int(ring[word])

    def verify_drafted(self, g: CapturedGraph, drafted: CapturedGraph, anchor: int, positions: Sequence[int], cache_len: int,
                       n_pend: int) -> bool:
        """``replay`` the verify graph ``g`` on ``anchor`` and the tokens that the draft queued last will have, over ``cache_len`` slots,
        the last ``n_pend`` of which are the draft's first rows, committed here.  False, and nothing queued, where that has to wait
        for the host."""
        if g.role != "verify" or g.graph is None or drafted.role not in DRAFT_ROLES or self._last is not drafted or \
                drafted.sigma != g.sigma or (g.one is not None and not self._behind(g)):
            return False
        if len(positions) != g.M or g.M - 1 > drafted.logits_end - drafted.logits_start:
            raise ValueError("positions / drafted tokens must be those of the verified block")
        if cache_len > g.sigma or not 0 <= n_pend <= min(cache_len, drafted.M):
            raise RuntimeError("history does not fit the segment")
        self.settle()
        if not g.io.arrived:
            g.io.uploaded.synchronize()
        g.io.inputs_host.numpy()[:] = (step_descriptor(g.role, g.M, self.D, cache_len) + list(positions) + [int(anchor)]
                                       + [-2 ** 31 + i for i in range(g.M - 1)] + [g.sigma, cache_len - n_pend, n_pend])
        if g.one is not None:
            self._as_one_launch()
        stream = torch.cuda.current_stream(self.device)
        if stream.cuda_stream != self._last_stream:
            stream.wait_event(drafted.io.uploaded)
        self._queue(g, g.one is None)
        return True

    def _gave_up(self, one: decode_ops.StepOne) -> bool:
        """Whether a step did not get the whole device; separate launches stay for a while then."""
        failed = int(one.failed[0])   # (read once: the device may set it at any time)
        if failed == 0:
            return False
        if failed != 1:
            raise RuntimeError("a decode step did not end")
        one.failed[0] = 0
        self._separate_for, self._back_off = self._back_off, min(2 * self._back_off, 1 << 20)
        self._undisturbed = 0
        return True

    def _as_one_launch(self) -> None:
        """A step that does not keep to the separate launches."""
        self._undisturbed += 1
        if self._undisturbed == self.BACK_OFF:   # (they may still be queued: one that gives up later is seen then)
            self._back_off = self.BACK_OFF

    def _keeps_separate(self, one: decode_ops.StepOne) -> bool:
        """Whether this replay keeps to the separate launches."""
        self._gave_up(one)
        if self._separate_for > 0:
            self._separate_for -= 1
            return True
        self._as_one_launch()
        return False

    def _launch(self, g: CapturedGraph, stream: "torch.cuda.Stream", one: Optional[decode_ops.StepOne]) -> None:
        # (a step in one launch keeps to separate ones without a graph of theirs: capturing one here, in the middle of a
        # program's work, would disturb its other threads)
        if g.graph is not None and one is g.one:
            g.io.out_host.numpy()[:] = g.pending
            if g.ring is not None:
                g.at = int(g.io.step_in_host[0])
                g.read = g.at - 1
                g.ring.numpy()[g.at % self.RING] = StepIO.PENDING
            g.graph.replay()          # uploads, runs the step, downloads the results
            g.io.downloaded = True
            self._last, self._last_stream = g, stream.cuda_stream
        else:
            self._last = None
            g.io.step_in.copy_(g.io.step_in_host, non_blocking=True)
            g._eager(one)
            g.io.downloaded = False
        g.io.uploaded.record(stream)

    def read_outputs(self, g: CapturedGraph) -> Tuple[np.ndarray, np.ndarray, int]:
        """One device-to-host copy + synchronisation: (argmax tokens, confidences,
        device-side accepted-prefix length) of the projected rows; behind ``step_ahead`` those of the last step."""
        if g.io.downloaded:
            if g.ahead:   # (each stores to the same words)
                g.io.uploaded.synchronize()
            # The results themselves, as the replay's last launch writes them: the event behind it is ready 7 - 11 us later,
            # and a blocking synchronisation wakes the thread up later still.
            out = g.io.out_host.numpy()
            deadline = time.perf_counter() + 0.05
            while True:
                if not (out == StepIO.PENDING).any():
                    g.io.arrived = True
                    break
                if time.perf_counter() > deadline:  # a replay is a millisecond: stop spinning
                    g.io.uploaded.synchronize()
                    break
        else:
            stream = torch.cuda.current_stream(self.device)
            stream.wait_event(g.io.uploaded)   # (the step may be on another one)
            g.io.out_host.copy_(g.io.out, non_blocking=True)
            stream.synchronize()
        if g.one is not None and g.one.failed[0] > 1:
            raise RuntimeError("a decode step did not end")
        rows = g.logits_end - g.logits_start
        out = g.io.out_host.numpy()
        toks = out[:rows].copy()
        accept = int(out[g.M])
        conf = out[g.M + 2: g.M + 2 + rows].view(np.float32).copy()
        return toks, conf, accept
