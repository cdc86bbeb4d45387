"""Which weights a step in one launch reads: those the model has when the step is queued or captured, and memory that is
still theirs."""
import dataclasses
import gc
import weakref

import pytest
import torch

from bitmtp_amd import decode_ops
from bitmtp_amd import model as M


class Recorded(decode_ops.StepOne):
    """Without the library and the device: the addresses only."""

    @classmethod
    def exchange_bytes(cls, shape, device) -> int:
        return 256

    def __init__(self, weights, shape, device, like=None):
        self.weights, self.addresses, self.shape, self.like = weights, self.addresses_of(weights), shape, like


def _model(device, layers=3, dim=256, ffn=512, seed=0):
    args = M.ModelArgs(dim=dim, n_layers=layers, n_heads=2, n_kv_heads=1, ffn_dim=ffn, vocab_size=128, mask_token_id=127)
    return M.BonsaiDecoder.random_init(args, seed=seed, device=device)


def _other(p, seed):
    gen = torch.Generator(device=p.weight.device).manual_seed(seed)
    return M._random_packed(p.out_features, p.in_features, gen, p.weight.device, p.bits)


@pytest.fixture
def plain(monkeypatch):
    for name in ("BONSAI_ONE_LAUNCH_STEP", "BONSAI_FUSED_STEP", "BONSAI_ATTENTION_ONE_LAUNCH", "BONSAI_ROPE_IN_ATTENTION"):
        monkeypatch.delenv(name, raising=False)


def test_replaced_weights_are_read_and_old_ones_stay_allocated(plain):
    model = _model("cpu")
    one = M.step_one(model, Recorded)
    assert M.step_one(model, Recorded, one) is one          # nothing changed
    old = weakref.ref(model.layers[1].wo.weight)
    model.layers[1].wo = _other(model.layers[1].wo, 5)
    gc.collect()
    assert old() is not None                                # `one` still reads it
    two = M.step_one(model, Recorded, one)
    assert two is not one and two.like is one
    assert two.addresses[1][1] == model.layers[1].wo.weight.data_ptr() and two.addresses[0] == one.addresses[0]
    model.layers[2].q_norm = model.layers[2].q_norm.clone()
    three = M.step_one(model, Recorded, two)
    assert three.addresses[2][10] == model.layers[2].q_norm.data_ptr() != two.addresses[2][10]


@pytest.mark.parametrize("change", [
    lambda lw: dataclasses.replace(lw, wo=dataclasses.replace(lw.wo, weight=lw.wo.weight[:128])),
    lambda lw: dataclasses.replace(lw, w_down=dataclasses.replace(lw.w_down, weight_scale=lw.w_down.weight_scale[:, :2].contiguous())),
    lambda lw: dataclasses.replace(lw, input_layernorm=lw.input_layernorm[:128]),
    lambda lw: dataclasses.replace(lw, k_norm=lw.k_norm.float()),
    lambda lw: dataclasses.replace(lw, w_gu=dataclasses.replace(lw.w_gu, weight=lw.w_gu.weight.t().contiguous().t())),
    lambda lw: dataclasses.replace(lw, wqkv=dataclasses.replace(lw.wqkv, bits=1)),
])
def test_tensors_that_the_launch_cannot_read_keep_the_separate_launches(change, plain):
    model = _model("cpu")
    assert M.step_one(model, Recorded) is not None
    model.layers[1] = change(model.layers[1])
    assert M.step_one(model, Recorded) is None


def test_a_snapshot_keeps_what_the_model_had():
    model = _model("cpu")
    before, weight = model.snapshot(), model.layers[0].wo.weight
    model.layers[0].wo = _other(model.layers[0].wo, 1)
    model.layers[1].w_gu.weight = model.layers[1].w_gu.weight.clone()
    model.layers[2] = model.layers[0]
    assert before.layers[0].wo.weight is weight and before.layers[2] is not model.layers[2]
    assert before.layers[1].w_gu.weight is not model.layers[1].w_gu.weight and before.head.weight is model.head.weight


@pytest.mark.parametrize("use_graphs", [False, True])
def test_old_weights_are_dropped_when_no_step_reads_them(use_graphs, plain, monkeypatch):
    """Without graphs the step before may still be queued, on whatever stream; a graph holds what it reads."""
    from bitmtp_amd import runtime
    atlas = runtime.GraphAtlas.__new__(runtime.GraphAtlas)
    atlas.model, atlas.device, atlas.use_graphs, atlas._one, atlas._block = _model("cpu"), torch.device("cpu"), use_graphs, None, None
    waits = []
    monkeypatch.setattr(torch.cuda, "synchronize", waits.append)
    monkeypatch.setattr(decode_ops, "StepOne", Recorded)
    first = atlas._one_launch(1)
    assert atlas._one_launch(1) is first and not waits
    atlas.model.layers[1].wo = _other(atlas.model.layers[1].wo, 5)
    assert atlas._one_launch(1) is not first and atlas._one is not first
    assert waits == ([] if use_graphs else [atlas.device])


@pytest.mark.gpu
@pytest.mark.parametrize("width", [1, 9])
def test_steps_follow_replaced_weights(width, plain, monkeypatch):
    """Without graphs every step, with graphs every capture, reads the weights of that moment; a graph captured before goes
    on with its own, also where it keeps to separate launches."""
    from bitmtp_amd.runtime import GraphAtlas
    model = _model("cuda:0", dim=1024, ffn=512)
    role = "ar" if width == 1 else "verify"

    def rows(atlas, g):
        """Keys and values of layer 0: one projection of the embedding."""
        atlas.kv(g.sigma).zero_()
        atlas.replay(g, list(range(width)), list(range(4, 4 + width)), 5)
        atlas.read_outputs(g)
        return atlas.kv(g.sigma)[:, 0, :, g.sigma:g.sigma + width].float()

    def separate():
        monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", "0")
        atlas = GraphAtlas(model, segment_ladder=(64,))
        out = rows(atlas, atlas.get_graph(width, 64, role))
        monkeypatch.delenv("BONSAI_ONE_LAUNCH_STEP")
        return out

    def same(x, y):
        # exact integer sums, scaled in another order: one bf16 step, and a key's norm and rotation (four roundings) make it two
        return bool(((x - y).abs() <= 2.0 ** -6 * y.abs().clamp(min=2.0 ** -3)).all())

    eager, graphs = GraphAtlas(model, segment_ladder=(64,), use_graphs=False), GraphAtlas(model, segment_ladder=(64, 256))
    ge, g = eager.get_graph(width, 64, role), graphs.get_graph(width, 64, role)
    assert ge.one is not None and g.one is not None
    first = separate()
    assert same(rows(eager, ge), first) and same(rows(graphs, g), first)
    for i, lw in enumerate(model.layers):
        lw.wqkv = _other(lw.wqkv, 30 + i)
    second = separate()
    assert not same(second, first)
    assert same(rows(eager, ge), second)
    assert same(rows(graphs, g), first)                     # captured before
    late = graphs.get_graph(width, 256, role)
    assert late.one is not g.one and late.one.exchange.data_ptr() == g.one.exchange.data_ptr()
    assert same(rows(graphs, late), second)
    graphs._separate_for = 1
    assert same(rows(graphs, g), first) and graphs._separate_for == 0
