"""The Python extension behind the operator layer (csrc/py_ops.cpp): it declines everything but plain contiguous GPU
tensors, and what it takes gives the bits of the checked ctypes path."""
import pytest
import torch

from bitmtp_amd import ops

DEV = "cuda:0"


def test_declines_what_is_not_a_plain_gpu_tensor():
    from bitmtp_amd import build
    build.build_torch_ops(verbose=False)
    if ops._native is None:
        ops._load_native()
    n = ops._native
    a, b = torch.zeros(2, 256, dtype=torch.int8), torch.zeros(8, 64, dtype=torch.int8)
    s, ws = torch.ones(2, 1), torch.ones(8, 2, dtype=torch.bfloat16)
    assert n.linear(2, a, b, s, ws, False) is None and n.linear(2, None, b, s, 3, False) is None
    assert n.grouped(2, [(a, b, s, ws)]) is None and n.grouped(2, []) is None and n.grouped(2, "x") is None
    x, w = torch.zeros(2, 256, dtype=torch.bfloat16), torch.zeros(256, dtype=torch.bfloat16)
    assert n.quant_input(x) is None and n.quant_input(7) is None and n.norm_quant(x, w, 1e-6) is None
    assert n.add_norm_quant(x, x, w, 1e-6) is None and n.silu_mul_quant(x) is None


def _without_extension(monkeypatch, tmp_path, broken=False):
    so = tmp_path / "_bonsai_py.so"
    if broken:
        so.write_bytes(b"not a library")
    monkeypatch.setattr(ops, "_native", None)
    monkeypatch.setattr(ops, "_native_missing", False)
    monkeypatch.setattr(ops, "py_ops_lib_path", lambda: str(so))


@pytest.mark.parametrize("broken", [False, True])
def test_only_the_prompt_path_needs_the_extension(monkeypatch, tmp_path, broken):
    _without_extension(monkeypatch, tmp_path, broken)
    with pytest.warns(RuntimeWarning, match="_bonsai_py.so"):
        ops._offer_native()
    import warnings
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        ops._offer_native()      # said once
    with pytest.raises((RuntimeError, ImportError)):
        ops.native()


@pytest.mark.gpu
def test_operators_run_without_the_extension(monkeypatch, tmp_path):
    x = torch.randn(3, 512, device=DEV).to(torch.bfloat16)
    b = torch.randint(-128, 128, (48, 128), device=DEV, dtype=torch.int8)
    ws = torch.rand(48, 4, device=DEV).to(torch.bfloat16)
    want = ops.t2g128_int8xint2_linear(*ops.quant_input(x)[:1], b, ops.quant_input(x)[1], ws)
    _without_extension(monkeypatch, tmp_path)
    with pytest.warns(RuntimeWarning, match="slower host path"):
        q, s = ops.quant_input(x)
    _same(ops.t2g128_int8xint2_linear(q, b, s, ws), want)
    assert ops._native is None


def _same(got, want):
    got, want = (g if isinstance(g, (tuple, list)) else (g,) for g in (got, want))
    assert len(got) == len(want)
    for g, t in zip(got, want):
        assert g.shape == t.shape and g.dtype == t.dtype
        assert torch.equal(g.view(torch.uint8), t.view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1,), (2, 3), (9,)])
@pytest.mark.parametrize("bits", [2, 1])
def test_same_bits_as_the_checked_path(bits, shape, monkeypatch):
    gen = torch.Generator(device=DEV).manual_seed(3)
    n, k = 384, 1024
    x = torch.randn(*shape, k, generator=gen, device=DEV)
    b = torch.randint(-128, 128, (n, k * bits // 8), generator=gen, device=DEV, dtype=torch.int8)
    ws = torch.rand(n, k // 128, generator=gen, device=DEV).to(torch.bfloat16)
    w = torch.rand(k, generator=gen, device=DEV).to(torch.bfloat16)
    xb = x.to(torch.bfloat16)
    linear = ops.t2g128_int8xint2_linear if bits == 2 else ops.q1g128_int8xint1_linear

    def everything():
        out = [ops.quant_input(t) for t in (x, xb, x.half())]
        q, s = out[1]
        out.append(linear(q, b, s, ws))
        q2, s2 = q.view(-1, k), s.view(-1, 1)
        out.append(ops.packed_gemv_ex(q2, b, s2, ws.half(), bits=bits))
        out.append(ops.packed_gemv_grouped([(q2, b, s2, ws), (q2[:1], b[:77], s2[:1], ws[:77])], bits=bits))
        out.append(ops.fused_norm_quant(xb, w, 1e-6))
        out.append(ops.fused_add_norm_quant(xb, xb, w, 1e-6))
        out.append(ops.silu_mul_quant(xb))
        return out

    everything()  # (the first accepted call of a process loads the extension)
    fast = everything()
    monkeypatch.setattr(ops, "_native", None)
    monkeypatch.setattr(ops, "_load_native", lambda: None)
    for got, want in zip(fast, everything()):
        _same(got, want)


@pytest.mark.gpu
def test_refused_operands_raise_the_operator_messages():
    x = torch.zeros(2, 256, dtype=torch.bfloat16, device=DEV)
    q, s = ops.quant_input(x)
    b = torch.zeros(8, 64, dtype=torch.int8, device=DEV)
    ws = torch.ones(8, 2, dtype=torch.bfloat16, device=DEV)
    ops.t2g128_int8xint2_linear(q, b, s, ws)
    with pytest.raises(RuntimeError, match="invalid weight scale shape"):
        ops.t2g128_int8xint2_linear(q, b, s, ws[:, :1])
    with pytest.raises(RuntimeError, match="contiguous CUDA tensors"):
        ops.t2g128_int8xint2_linear(q, b, s, ws.t().contiguous().t())
    with pytest.raises(RuntimeError, match="activation scales"):
        ops.t2g128_int8xint2_linear(q, b, s.view(-1), ws)
