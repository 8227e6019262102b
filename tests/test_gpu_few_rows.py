"""The few-row matvec kernel (decode batches of up to 32 rows, two passes up to
64): ring and one-tile forms, one and two column tiles, K slices through the
workspace, tile and K remainders, types, groups and scale layouts, with the
bound of test_gpu_gemm_rows.  (fp16 rows start where the v_dot2 kernel, exact
in W, ends.)"""

import pytest
import torch

import mk.quant_ops as qo
from mk import _lib
from tests.test_gpu_gemm_rows import HALF_ULP, _check, _check_rows, _rounded, _weight

pytestmark = pytest.mark.gpu

CASES = [  # M, N, K
    (5, 1, 32), (8, 15, 96), (9, 33, 544), (16, 100, 512), (16, 3000, 512), (17, 257, 1056), (32, 600, 2080),
    # several tiles per workgroup (ring refills, turns of one tile and of two, a last partial turn); K slices of 4096
    # and less, the last partly past K
    (6, 9000, 1024), (31, 17000, 512), (7, 1000, 4128), (16, 515, 14336), (32, 4096, 8224), (20, 5000, 4608),
    (40, 4096, 14336), (33, 700, 5120), (28, 700, 4128), (9, 25000, 512), (20, 25000, 512),
    # rows that go to the K-split and MFMA kernels in fp16
    (7, 3072, 8192), (12, 4096, 6144), (8, 3000, 5056), (5, 2100, 11008)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", CASES)
def test_few_rows(dev, M, N, K, bits, dtype):
    gen = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).to(dtype)
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    for g, zeros in ((64, "whole"), (32, "whole"), (128, "whole"), (256, "whole"), (128, "none"), (64, "affine")):
        codes, packed, s, z = _weight(gen, dev, N, K, bits, g, torch.float16, zeros)
        got = fn(x, packed, s, z, group_size=g)
        _check_rows(got, x, codes, s, z, g, bits, f"M{M} N{N} K{K} q{bits} g{g} {zeros}")
        res = torch.randn((M, N), generator=gen, device=dev).to(dtype)
        mm, out = qo.q_matvec_residual(x, packed, s, z, res, bits=bits, group_size=g, want_mm=True)
        assert torch.equal(mm, got)
        assert torch.equal(out, (res.float() + mm.float()).to(dtype))


@pytest.mark.parametrize("g", [32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(5, 7, 64), (8, 300, 1024), (12, 14336, 512), (32, 9000, 1024), (24, 100, 4096),
                                   (16, 3000, 1056)])
def test_few_rows_gate_up(dev, M, N, K, bits, dtype, g):
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).to(dtype)
    for zeros in ("whole", "affine"):
        cg, gw, gs, gz = _weight(gen, dev, N, K, bits, g, torch.float16, zeros)
        cu, uw, us, uz = _weight(gen, dev, N, K, bits, g, torch.float16, zeros)
        gate, up, mlp = qo.q_gate_up_swiglu(x, gw, uw, gs, us, gz, uz, bits=bits, group_size=g, return_gate_up=True)
        _check_rows(gate, x, cg, gs, gz, g, bits, ("gate", zeros))
        _check_rows(up, x, cu, us, uz, g, bits, ("up", zeros))
        gf = gate.double()
        want = gf / (1 + torch.exp(-gf)) * up.double()
        # silu in fp32 (a few 2^-24), the product rounded once
        assert bool(((mlp.double() - want).abs() <= 1.01 * HALF_ULP[dtype] * want.abs() + 2.0 ** -24).all())


@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_few_rows_bf16_small(dev, M):
    gen = torch.Generator(device=dev).manual_seed(M)
    for N, K, bits in ((70, 1024, 4), (4096, 4608, 4), (33, 96, 8)):
        x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
        codes, packed, s, z = _weight(gen, dev, N, K, bits, 32, torch.float16, "whole")
        fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
        _check(fn(x, packed, s, z, group_size=32), x, _rounded(codes, s, z, 32, torch.bfloat16), torch.bfloat16,
               (M, N, K))


@pytest.mark.parametrize("bits", [4, 8])
def test_few_rows_unaligned_scales_and_no_workspace(dev, bits):
    """Scales 2 bytes off (one value per load) give the aligned result; a call
    without a workspace (whole rows, other kernels) agrees within the bound."""
    gen = torch.Generator(device=dev).manual_seed(5)
    M, N, K, g = 8, 130, 14336, 64
    x = torch.randn((M, K), generator=gen, device=dev).half()
    codes, packed, s, z = _weight(gen, dev, N, K, bits, g, torch.float16, "whole")
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    want = fn(x, packed, s, z, group_size=g)
    off = lambda t: torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)[1:].reshape(t.shape).copy_(t)
    assert torch.equal(fn(x, packed, off(s), off(z), group_size=g), want)
    y = torch.empty_like(want)
    _lib.launch(f"mk_q{bits}_matvec", dev, x.data_ptr(), packed.data_ptr(), s.data_ptr(), z.data_ptr(), None, None,
                y.data_ptr(), M, N, K, g, _lib.DT_F16, _lib.DT_F16)
    _check(y, x, _rounded(codes, s, z, g, torch.float16), torch.float16, "no workspace")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,K,g", [(6, 96, 32), (16, 544, 64), (8, 1056, 128), (16, 4608, 32), (7, 4608, 64),
                                   (5, 4608, 128)])
def test_few_rows_infinite_weights_before_k_ends(dev, M, K, g, bits):
    """Rows whose first weights are infinite in fp16 give the saturated sum, also
    where blocks (or whole waves) past K re-read them against zero activations."""
    N, top = 70, 15 if bits == 4 else 255
    codes = torch.full((N, K), top, dtype=torch.uint8, device=dev)
    s = torch.full((N, -(-K // g)), 1e-3, device=dev).half()
    s[:, 0] = 2 * 65504.0 / top
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4) if bits == 4 else codes).contiguous()
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    x = torch.full((M, K), 0.01, device=dev).half()
    x[1::2] = -0.01
    got = fn(x, packed, s, None, group_size=g)
    assert bool((got[0::2] == 65504.0).all()) and bool((got[1::2] == -65504.0).all())
