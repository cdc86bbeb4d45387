"""Blocks of more than 16 tokens (gemv_wide_kernel, every tile) and rows that are no whole number of 512-wide K tiles
(gemv_mxl_ragged_kernel) against a float64 product of the unpacked operands: int32 group sums exactly, the scaled value to fp32
summation order, bf16 to its own rounding.  Sizes sit on the edges of tiles, slices and scale groups."""
import pytest
import torch

from bitmtp_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(m, n, k, bits, seed, scale_dtype=torch.bfloat16):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randint(-128, 128, (m, k), generator=gen, device=DEV, dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k * bits // 8), generator=gen, device=DEV, dtype=torch.int8)
    ws = torch.exp(torch.randn(n, k // 128, generator=gen, device=DEV) * 0.5 - 4).to(scale_dtype)
    s = torch.rand(m, 1, generator=gen, device=DEV) * 40 + 1
    shifts = torch.arange(0, 8, bits, device=DEV, dtype=torch.uint8)
    codes = ((b.view(torch.uint8).unsqueeze(-1) >> shifts) & ((1 << bits) - 1)).view(n, k).double()
    w = codes - 2 if bits == 2 else 2 * codes - 1
    groups = torch.stack([a[:, g:g + 128].double() @ w[:, g:g + 128].T for g in range(0, k, 128)], dim=-1)
    return a, b, s, ws, groups, (groups * ws.double()).sum(-1) / s.double()


def _check(m, n, k, bits, scale_dtype, family):
    a, b, s, ws, groups, want = _problem(m, n, k, bits, m + n + k, scale_dtype)
    g = ops.packed_gemv_ex(a, b, None, None, bits=bits, out_kind=ops.OUT_G32)
    assert ops.last_kernel(bits).startswith(family), ops.last_kernel(bits)
    assert torch.equal(g.double(), groups)
    y32 = ops.packed_gemv_ex(a, b, s, ws, bits=bits, out_kind=ops.OUT_F32)
    assert ops.last_kernel(bits).startswith(family)
    scale = (groups.abs() * ws.double()).sum(-1) / s.double()
    assert ((y32.double() - want).abs() <= 1e-6 * scale + 1e-30).all()
    y = ops.packed_gemv_ex(a, b, s, ws, bits=bits)
    assert torch.equal(y.view(torch.int16), y32.to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("variant", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (17, 16, 256), (32, 64, 384), (33, 65, 512), (128, 128, 2048),
                                   (129, 131, 640), (257, 1000, 1152), (40, 136, 9728)])
def test_wide_kernel(m, n, k, variant, bits, scale_dtype):
    print(f"[case] wide variant {variant} bits {bits} {m}x{n}x{k} {scale_dtype}", flush=True)
    lib = ops.t2_lib() if bits == 2 else ops.q1_lib()
    tune = lib.t2g128_set_mfma_tuning if bits == 2 else lib.q1g128_set_mfma_tuning
    tune(0, variant, 0, 0, 7)
    try:
        _check(m, n, k, bits, scale_dtype, "gemv_wide_kernel<")
    finally:
        tune(0, 0, 0, 0, 0)


@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k,family", [(49, 12288, 2048, "gemv_wide_kernel<"), (32, 2048, 2048, "gemv_mxl_kernel<"),
                                          (600, 700, 1664, "gemv_wide_kernel<"), (9, 20000, 896, "gemv_mxl_ragged_kernel<"),
                                          (5, 33000, 384, "gemv_wide_kernel<")])
def test_built_in_choice(m, n, k, family, bits):
    print(f"[case] choice bits {bits} {m}x{n}x{k}", flush=True)
    _check(m, n, k, bits, torch.bfloat16, family)


@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k,family", [
    (192, 1086, 1152, "gemv_mxl_ragged_kernel<"), (193, 1086, 1152, "gemv_wide_kernel<"),   # a table holds twelve token tiles
    (16, 2048, 512, "gemv_mxl_kernel<"), (33, 4096, 512, "gemv_mfma_direct_kernel<"), (64, 1000, 1024, "gemv_mxl_kernel<"),
    (65, 1000, 1024, "gemv_mfma_direct_kernel<"), (16, 12000, 1536, "gemv_mxl_kernel<"), (17, 20000, 1536, "gemv_mfma_kernel<"),
    (80, 12288, 1024, "gemv_wide_kernel<")])
def test_built_in_choice_is_among_kernels_that_run(m, n, k, family, bits):
    """Where the lean kernel does not take the rows, the choice is between the wide kernel and what does."""
    print(f"[case] choice bits {bits} {m}x{n}x{k}", flush=True)
    _check(m, n, k, bits, torch.bfloat16, family)


@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k", [(3, 1, 512), (4, 17, 512), (8, 100, 1024), (9, 48, 1536), (16, 333, 1024), (33, 1000, 512),
                                   (64, 700, 1536)])
def test_lean_kernel_rows_of_one_to_three_tiles(m, n, k, bits, scale_dtype):
    """Fewer K tiles than waves: some slices are empty."""
    print(f"[case] lean short rows bits {bits} {m}x{n}x{k} {scale_dtype}", flush=True)
    _check(m, n, k, bits, scale_dtype, "gemv_mxl_kernel<")


@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k", [(2, 40, 512), (5, 333, 1024), (16, 100, 2048), (17, 100, 2048), (200, 300, 512),
                                   (70, 1000, 2176)])
def test_scales_on_any_16_bit_address(m, n, k, bits):
    """Scales that do not start on 8 bytes keep the kernels with wide scale loads out, alone and in a grouped call."""
    print(f"[case] unaligned scales bits {bits} {m}x{n}x{k}", flush=True)
    a, b, s, ws, groups, want = _problem(m, n, k, bits, m + n + k)
    flat = torch.empty(ws.numel() + 1, dtype=ws.dtype, device=DEV)
    odd = flat[1:].view(ws.shape)
    odd.copy_(ws)
    assert odd.data_ptr() % 8 == 2 and odd.is_contiguous()
    scale = (groups.abs() * ws.double()).sum(-1) / s.double()
    for y in (ops.packed_gemv_ex(a, b, s, odd, bits=bits, out_kind=ops.OUT_F32),
              ops.packed_gemv_grouped([(a, b, s, odd), (a, b, s, ws)], bits=bits, out_kind=ops.OUT_F32)[0]):
        assert ((y.double() - want).abs() <= 1e-6 * scale + 1e-30).all()


@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k", [(600, 600, 23936), (300, 4100, 24064), (130, 1100, 32512), (70, 520, 56704), (33, 40, 65536)])
def test_rows_too_long_for_some_tiles(m, n, k, bits):
    """Rows whose staged scales leave no room for the tile that would be fastest take another one that fits."""
    print(f"[case] long rows bits {bits} {m}x{n}x{k}", flush=True)
    lib = ops.t2_lib() if bits == 2 else ops.q1_lib()
    tune = lib.t2g128_set_mfma_tuning if bits == 2 else lib.q1g128_set_mfma_tuning
    tune(0, 0, 0, 0, 7)   # the wide kernel, the tile its own choice
    try:
        _check(m, n, k, bits, torch.bfloat16, "gemv_wide_kernel<")
    finally:
        tune(0, 0, 0, 0, 0)


@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits", [2, 1])
@pytest.mark.parametrize("m,n,k", [(3, 16, 640), (4, 17, 768), (8, 100, 896), (9, 48, 640), (16, 333, 896), (16, 40, 1920),
                                   (20, 1000, 2176), (5, 2048, 6272), (12, 2500, 9600)])
def test_lean_kernel_rows_of_any_length(m, n, k, bits, scale_dtype):
    print(f"[case] lean bits {bits} {m}x{n}x{k} {scale_dtype}", flush=True)
    _check(m, n, k, bits, scale_dtype, "gemv_mxl_ragged_kernel<")
