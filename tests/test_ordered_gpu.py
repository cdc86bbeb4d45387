"""Activations in operand order (bonsai_*_quant_ordered, t2g128_gemv_ordered): the quantisers' bytes are those of the other order, moved; the
products are the same bits, on every tile, and what the wide kernel does not take is refused.  Sizes sit on the edges of tiles, slices and
scale groups."""
import ctypes

import pytest
import torch

from bitmtp_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
p = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())   # noqa: E731


def _ordered(q):
    m, k = q.shape
    return q.view(m, k // 16, 4, 4).transpose(2, 3).reshape(m, k).contiguous()


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("m,k", [(1, 128), (3, 384), (5, 2048), (2, 8192), (2, 8320), (1, 9728), (1, 40960), (1, 65536)])
def test_quantisers(m, k):
    gen = torch.Generator(device=DEV).manual_seed(k + m)
    x, r = ((torch.randn(m, k, generator=gen, device=DEV) * 3).to(torch.bfloat16) for _ in range(2))
    w = (1 + 0.1 * torch.randn(k, generator=gen, device=DEV)).to(torch.bfloat16)
    lib = ops.actq_lib()
    q, s, h = torch.empty(m, k, dtype=torch.int8, device=DEV), torch.empty(m, device=DEV), torch.empty_like(x)
    eps = ctypes.c_float(1e-6)
    assert lib.bonsai_act_quant_ordered(p(x), p(q), p(s), m, k, _stream()) == 0
    want, scale = ops.quant_input(x)
    assert torch.equal(q, _ordered(want)) and torch.equal(s.view(-1), scale.view(-1))
    assert lib.bonsai_norm_quant_ordered(p(x), None, p(w), eps, None, p(q), p(s), m, k, _stream()) == 0
    want, scale = ops.fused_norm_quant(x, w, 1e-6)
    assert torch.equal(q, _ordered(want)) and torch.equal(s.view(-1), scale.view(-1))
    assert lib.bonsai_norm_quant_ordered(p(x), p(r), p(w), eps, p(h), p(q), p(s), m, k, _stream()) == 0
    rows, want, scale = ops.fused_add_norm_quant(x, r, w, 1e-6)
    assert torch.equal(h, rows) and torch.equal(q, _ordered(want)) and torch.equal(s.view(-1), scale.view(-1))
    for rc in (lib.bonsai_act_quant_ordered(p(x), p(q), p(s), m, k - 64, _stream()),
               lib.bonsai_norm_quant_ordered(p(x), p(r), p(w), eps, None, p(q), p(s), m, k, _stream())):
        assert rc != 0


@pytest.mark.parametrize("variant", [0, 1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (17, 32, 256), (33, 80, 384), (64, 256, 512), (129, 272, 640), (128, 128, 2048),
                                   (257, 1008, 1152), (40, 144, 9728)])
def test_products(m, n, k, variant):
    print(f"[case] ordered variant {variant} {m}x{n}x{k}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, device=DEV, dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k // 4), generator=gen, device=DEV, dtype=torch.int8)
    ws = torch.exp(torch.randn(n, k // 128, generator=gen, device=DEV) * 0.5 - 4).to(torch.bfloat16)
    s = torch.rand(m, generator=gen, device=DEV) * 40 + 1
    s[0] = 1e-30   # (infinite results)
    lib = ops.t2_lib()
    tune, plain, silu, ordered = (getattr(lib, "t2g128_" + f) for f in ("set_mfma_tuning", "gemv_ex", "gemv_silu", "gemv_ordered"))
    order = _ordered(a)
    tune(0, variant, 0, 0, 7 if variant else 0)
    try:
        for pairs in (0, 1):
            want, got = (torch.full((m, n // (1 + pairs)), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
            args = [p(b), p(want), p(s), p(ws), m, n, k]
            rc = silu(p(a), *args, _stream()) if pairs else plain(p(a), *args, 0, 0, _stream())
            args[1] = p(got)
            answer = ordered(p(order), *args, pairs, 1, _stream())
            wide = answer == 0
            assert answer in (0, -1) and (got == 7.0).all()
            if pairs and rc == -1 and wide:   # (the other order may leave a block to two launches that this one takes)
                whole = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
                assert plain(p(a), p(b), p(whole), p(s), p(ws), m, n, k, 0, 0, _stream()) == 0
                gate, up = whole.chunk(2, dim=1)
                want = None   # the same but for the device's exponential: see the forced tiles
            else:
                assert rc == 0 or not wide
            assert ordered(p(order), *args, pairs, 0, _stream()) == (0 if wide else -1)
            assert wide or variant == 0
            if wide:
                assert ops.last_kernel(2).startswith("gemv_wide_ordered_kernel<")
                if want is None:
                    torch.testing.assert_close(got[1:].float(), (torch.nn.functional.silu(gate) * up)[1:].float(), rtol=2 ** -6, atol=1e-3)
                else:
                    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
            else:
                assert (got == 7.0).all()
    finally:
        tune(0, 0, 0, 0, 0)
