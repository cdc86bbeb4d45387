"""All layers of a step of 2 to 16 rows as one launch (``decode_ops.StepBlock``) against the separate launches of the same
step: shapes at the edges of what the launch takes, block widths, roles, histories at the edges of the attention's parts,
and what happens after a launch that did not get the whole device."""
import numpy as np
import pytest
import torch

from test_step_one_gpu import BAD_ARGUMENTS, DEV, _model, _refused

pytestmark = pytest.mark.gpu


def _pair(model, sigma, width, role, monkeypatch):
    """Atlases whose step is one launch / separate launches."""
    from bitmtp_amd.runtime import GraphAtlas
    atlases = []
    for flag in ("1", "0"):
        monkeypatch.setenv("BONSAI_ONE_LAUNCH_STEP", flag)
        a = GraphAtlas(model, segment_ladder=(sigma,))
        g = a.get_graph(width, sigma, role)
        assert (g.one is not None) == (flag == "1")
        atlases.append((a, g))
    return atlases


def _compare(model, sigma, width, role, lengths, monkeypatch):
    (a1, g1), (a0, g0) = _pair(model, sigma, width, role, monkeypatch)
    gen = torch.Generator(device=DEV).manual_seed(1)
    hist = (torch.randn(tuple(a1.kv(sigma).shape), generator=gen, device=DEV) * 0.5).to(torch.bfloat16)
    rows = slice(sigma, sigma + width)
    for n in lengths:
        tokens = [(7 * n + 13 * i) % 1000 for i in range(width)]
        positions = [max(n - 1, 0) + i for i in range(width)]
        outs = []
        for a, g in ((a1, g1), (a0, g0), (a1, g1)):
            a.kv(sigma).copy_(hist)
            a.replay(g, tokens, positions, n, width - 8 if role == "draft" else 0)
            a.read_outputs(g)
            outs.append((a.kv(sigma)[:, :, :, rows].clone(), a.workspace.logits[:g.logits_end - g.logits_start, :1000].clone()))
        assert a1._block.failed[0] == 0
        assert torch.equal(outs[0][0], outs[2][0]) and torch.equal(outs[0][1], outs[2][1])   # other set, same bits
        after = a1.kv(sigma)
        assert torch.equal(after[:, :, :, :sigma], hist[:, :, :, :sigma])
        assert torch.equal(after[:, :, :, sigma + width:], hist[:, :, :, sigma + width:])
        # Layer 0 sees no attention: projections are exact integer sums, scaled in another order, so values and keys before
        # their norm differ by one bf16 step at most, and a key's norm and rotation (four roundings) can make it two.
        first = (outs[0][0][:, 0].float() - outs[1][0][:, 0].float()).abs()
        assert bool((first <= 2.0 ** -6 * outs[1][0][:, 0].float().abs().clamp(min=2.0 ** -3)).all())
        # Behind the attention (another split of the slots, bf16 probabilities) int8 roundings of a row move by whole steps.
        # If every value of a normal row moved by one, 1 / 127 of its maximum of about 3.5 rms, a product of it would change
        # by 2.8e-2; the row itself differs by less than a bf16 step, 4e-3, a layer.
        for x, y in ((outs[0][0].transpose(0, 3), outs[1][0].transpose(0, 3)), (outs[0][1], outs[1][1])):
            x, y = x.float().flatten(1), y.float().flatten(1)
            assert float(((x - y).norm(dim=1) / y.norm(dim=1)).max()) <= 4e-2, f"history of {n}"


CASES = [
    # bits, dim, ffn, heads, kv heads, width, role
    (2, 128, 128, 1, 1, 2, "ar"),          # one group of K, workgroups without rows
    (1, 256, 256, 2, 1, 16, "draft"),
    (2, 384, 640, 3, 1, 3, "ar"),          # odd numbers of groups, three query heads on one key head
    (1, 384, 640, 3, 1, 9, "verify"),
    (2, 1024, 512, 8, 4, 8, "draft"),      # half of a load's lanes
    (2, 1280, 2304, 8, 8, 9, "draft"),     # row counts that leave workgroups idle
    (1, 1024, 1024, 8, 2, 16, "draft"),
    (2, 2048, 6144, 16, 8, 9, "verify"),   # the smaller build at its largest
    (1, 2048, 6144, 16, 8, 16, "ar"),
    (2, 2560, 9728, 32, 8, 9, "draft"),    # the larger build at its largest
    (2, 2560, 9728, 32, 8, 16, "verify"),
    (1, 2560, 9728, 32, 8, 5, "ar"),
]


@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv,width,role", CASES)
def test_one_launch_against_the_separate_launches(bits, dim, ffn, n_heads, n_kv, width, role, monkeypatch):
    print(f"[case] {bits} bits, {dim} x {ffn}, {n_heads} / {n_kv} heads, {width} rows, {role}", flush=True)
    lengths = [1, 7, 64 - width, 65 - width, 64, 127, 255, 256] + ([0] if role == "ar" else [])
    _compare(_model(bits, dim, ffn, n_heads, n_kv), 256, width, role, lengths, monkeypatch)


@pytest.mark.parametrize("n_heads,n_kv,width", [(16, 8, 9), (32, 8, 16), (8, 1, 2)])
def test_long_histories(n_heads, n_kv, width, monkeypatch):
    """As many parts as there are workgroups for, with up to several passes each."""
    print(f"[case] long histories, {n_heads} / {n_kv} heads, {width} rows", flush=True)
    _compare(_model(2, 1024, 1024, n_heads, n_kv), 4096, width, "verify", (300, 447, 448, 512, 960 - width, 961 - width, 2047, 4096), monkeypatch)


def test_shapes_and_widths_that_keep_the_separate_launches():
    from bitmtp_amd import decode_ops
    from bitmtp_amd.runtime import GraphAtlas
    assert decode_ops.StepBlock.exchange_bytes((2, 3, 2048, 6144, 16, 8), torch.device(DEV)) > 0
    assert decode_ops.StepBlock.exchange_bytes((2, 2, 2048, 6144, 16, 8), torch.device(DEV)) > 0
    for shape in ((2, 1, 2048, 6144, 16, 8),        # one layer
                  (2, 3, 1088, 6144, 16, 8),        # half a group of K
                  (2, 3, 8192, 28672, 64, 8),       # more rows than the LDS has room for
                  (2, 3, 2048, 6144, 15, 8),
                  (3, 3, 2048, 6144, 16, 8)):
        assert decode_ops.StepBlock.exchange_bytes(shape, torch.device(DEV)) == 0, shape
    atlas = GraphAtlas(_model(2, 256, 256, 2, 1), segment_ladder=(64,))
    assert atlas.get_graph(16, 64, "ar").one is not None and atlas.get_graph(17, 64, "ar").one is None


def test_argument_checks():
    from bitmtp_amd import decode_ops
    _refused(9, [(0, {}), (1, {}), (17, {})] + [(9, bad) for bad in BAD_ARGUMENTS + [dict(sigma=88), dict(dim=2000)]])
    assert decode_ops.decode_lib().bonsai_decode_step_block(None, 9, None) != 0


def test_steps_are_repeated_after_a_launch_that_gave_up():
    """Marks of launches that gave up, for a block and a one-token step behind it, with nothing read in between."""
    from bitmtp_amd.runtime import GraphAtlas
    model = _model(2, 1024, 1024, 8, 4)
    atlas = GraphAtlas(model, segment_ladder=(256,))
    sigma = 256
    verify, ar = atlas.get_graph(9, sigma, "verify"), atlas.get_graph(1, sigma, "ar")
    assert verify.one is not None and ar.one is not None and verify.one is not ar.one
    results = []
    for lost in (False, True):
        atlas.kv(sigma).zero_()
        for n in range(1, 28, 9):
            if lost and n == 10:
                for one in (atlas._one, atlas._block):
                    one.exchange[4:8].view(torch.int32).fill_(1)
            atlas.replay(verify, list(range(n, n + 9)), list(range(n - 1, n + 8)), n)
            atlas.commit_kv(sigma, n, 4)
            atlas.replay(ar, [n], [n + 4], n + 4)
            atlas.commit_kv(sigma, n + 4, 1)
            toks, conf, accept = atlas.read_outputs(verify)
        results.append((toks, accept, atlas.kv(sigma)[:, :, :, :24].float().clone()))
    assert atlas._separate_for > 0
    (t0, c0, k0), (t1, c1, k1) = results
    assert np.array_equal(t0, t1) and c0 == c1
    assert float((k0 - k1).norm() / k0.norm()) <= 4e-2   # other launches, as in the comparison above
