"""gate|up of a wide block with silu(gate) * up behind it (``*_gemv_silu``) against the projection and the activation as two
launches: every tile of the wide kernel, ragged tokens and rows, the same bits."""
import ctypes
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(oracle, bits, M, F, K, seed):
    import bitmtp_amd as ops
    p = oracle.synth_problem(seed, M, 2 * F, K, bits)
    A, B = torch.from_numpy(p["A"]).to(DEV), torch.from_numpy(p["B"].view(np.int8)).to(DEV)
    s = torch.from_numpy(p["s"]).reshape(M, 1).to(DEV)
    ws = torch.from_numpy(p["ws"].view(np.int16).copy()).view(torch.bfloat16).to(DEV)
    lib, name = (ops.ops.t2_lib(), "t2g128") if bits == 2 else (ops.ops.q1_lib(), "q1g128")
    out = torch.full((M, F), 7.0, dtype=torch.bfloat16, device=DEV)
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = getattr(lib, name + "_gemv_silu")(vp(A), vp(B), vp(out), vp(s), vp(ws), M, 2 * F, K, stream)
    gu = ops.packed_gemv_ex(A, B, s, ws, bits=bits, out_kind=ops.ops.OUT_BF16)
    torch.cuda.synchronize()
    return lib, name, rc, out, gu


def _same(out, gu):
    import bitmtp_amd as ops
    q, s = ops.quant_input(out)
    q0, s0 = ops.silu_mul_quant(gu)
    assert torch.equal(s, s0) and torch.equal(q, q0)
    g, u = gu.float().chunk(2, dim=1)
    want = (torch.nn.functional.silu(g).to(torch.bfloat16).float() * u).to(torch.bfloat16)
    # (the hardware's exponential: the neighbouring bf16 silu, times up)
    assert float((out.float() - want.float()).abs().max()) <= 2.0 ** -7 * float(want.float().abs().max())


@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("tile", range(1, 7))
def test_every_tile(oracle, bits, tile):
    lib = __import__("bitmtp_amd").ops.t2_lib() if bits == 2 else __import__("bitmtp_amd").ops.q1_lib()
    tuning = getattr(lib, ("t2g128" if bits == 2 else "q1g128") + "_set_mfma_tuning")
    tuning(0, tile, 0, 0, 7)
    try:
        for M, F, K in ((33, 136, 384), (64, 128, 512), (130, 1000, 640)):
            print(f"[case] {bits} bits, tile {tile}, {M} x {2 * F} x {K}", flush=True)
            _, _, rc, out, gu = _run(oracle, bits, M, F, K, 7 + M)
            assert rc == 0
            _same(out, gu)
    finally:
        tuning(0, 0, 0, 0, 0)


@pytest.mark.parametrize("bits,M,F,K", [(2, 256, 6144, 2048), (2, 301, 9728, 2560), (1, 77, 6144, 2048)])
def test_default_tile(oracle, bits, M, F, K):
    print(f"[case] {bits} bits, {M} x {2 * F} x {K}", flush=True)
    _, _, rc, out, gu = _run(oracle, bits, M, F, K, 11 + M)
    assert rc == 0
    _same(out, gu)


def test_what_is_not_taken(oracle):
    """Blocks of other kernels and rows that do not come in whole pieces: nothing is launched."""
    for M, F, K in ((9, 512, 512), (64, 132, 512)):
        _, _, rc, out, _ = _run(oracle, 2, M, F, K, 5)
        assert rc == -1 and bool((out == 7.0).all())
