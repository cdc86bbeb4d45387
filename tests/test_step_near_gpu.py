"""Hand-overs between workgroups of a die in the steps of one launch: the exchange memory knows whether a kv head's workgroups
share one, and results do not depend on it."""
import pytest
import torch

from test_step_one_gpu import DEV, _model

pytestmark = pytest.mark.gpu

SHARED, DIE_OF = 16, 24   # control words: whether the dies are shared, a word of dies for each number modulo eight


@pytest.mark.parametrize("width", [1, 9])
@pytest.mark.parametrize("bits,dim,ffn,n_heads,n_kv", [
    (2, 2048, 6144, 16, 8),    # a workgroup's rows within a head
    (2, 2304, 6400, 24, 8),    # .. and in two of them
    (1, 2560, 9728, 32, 8),
    (2, 1024, 512, 8, 4),      # heads that two dies share
])
def test_the_same_results_near_and_past_the_l2(bits, dim, ffn, n_heads, n_kv, width):
    print(f"[case] {bits} bits, {dim} x {ffn}, {n_heads} / {n_kv} heads, {width} rows", flush=True)
    from bitmtp_amd.runtime import GraphAtlas, step_descriptor
    sigma = 1024
    model = _model(bits, dim, ffn, n_heads, n_kv)
    atlas = GraphAtlas(model, segment_ladder=(sigma,))
    g = atlas.get_graph(width, sigma, "ar")
    control = g.one.exchange[:256].view(torch.int32)
    words = control.tolist()
    assert words[SHARED] == (n_kv % 8 == 0)
    assert all(w and w & (w - 1) == 0 for w in words[DIE_OF:DIE_OF + 8])
    kv = atlas.kv(sigma)
    hist = (torch.randn(tuple(kv.shape), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV) * 0.5).to(torch.bfloat16)
    h = atlas.workspace.h[0][:width]
    for n in (0, 24, 127, 300, 1000):   # one part of a head's slots, and several
        inputs = step_descriptor("ar", width, model.args.block_size, n) + [n + i for i in range(width)] + list(range(width))
        outs = []
        # as found, every workgroup elsewhere than expected, heads that share no die
        for shared, dies in ((words[SHARED], words[DIE_OF:DIE_OF + 8]), (words[SHARED], [0] * 8), (0, words[DIE_OF:DIE_OF + 8])):
            control[SHARED:DIE_OF + 8] = torch.tensor([shared] + [0] * 7 + dies, dtype=torch.int32, device=DEV)
            kv.copy_(hist)
            g.io.step_in.copy_(torch.tensor(inputs, dtype=torch.int32))
            g.one.enqueue(model.embed, g.io.step_in, kv, *atlas.rope, sigma, 1e-6, h, width)
            torch.cuda.synchronize()
            assert g.one.failed[0] == 0
            outs.append((h.clone(), kv.clone()))
        for other in outs[1:]:
            assert torch.equal(outs[0][0], other[0]) and torch.equal(outs[0][1], other[1]), f"history of {n}"
