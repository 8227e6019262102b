"""The matrix-product kernel (33 and more activation rows): every workgroup
shape, tile edges in rows, output rows and K, types, group sizes and scale
layouts, against a float64 product of the weights as the reference rounds
them (to the activation type, ops/quant_ops.py:509-526).

Bound: fp32 accumulation of K products, each partial sum within 2^-24 of it
(K * 2^-24 * sum |x||w| over any order), then one rounding to the type."""

import pytest
import torch

import mk.quant_ops as qo

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _weight(gen, dev, N, K, bits, g, sdt, zeros):
    top = 16 if bits == 4 else 256
    codes = torch.randint(0, top, (N, K), generator=gen, device=dev, dtype=torch.uint8)
    G = -(-K // g)
    # fp16 scales and zero points in eighths: (q - z) * s is then exact in
    # fp32 (22 bits), and the rounded weight does not depend on whether that
    # product is rounded first
    s = (torch.rand((N, G), generator=gen, device=dev) * 0.01 + 0.001).half().to(sdt)
    z = None
    if zeros == "affine":  # fractional zero points
        z = (torch.randint(0, 8 * top, (N, G), generator=gen, device=dev) / 8).to(sdt)
    elif zeros == "whole":
        z = torch.randint(0, top, (N, G), generator=gen, device=dev).to(sdt)
    packed = codes
    if bits == 4:
        packed = codes[:, 0::2] | (codes[:, 1::2] << 4)
    return codes, packed.contiguous(), s, z


def _rounded(codes, s, z, g, dtype):
    K = codes.shape[1]
    full = s.float().repeat_interleave(g, 1)[:, :K]
    zero = 0.0 if z is None else z.float().repeat_interleave(g, 1)[:, :K]
    return ((codes.float() - zero) * full).to(dtype).double()


def _check(got, x, W, dtype, what, slack=None):
    ref = x.double() @ W.t()
    bound = x.shape[1] * 2.0 ** -24 * (x.double().abs() @ W.abs().t())
    if slack is not None:
        bound += x.double().abs() @ slack.t()
    lim = bound + 1.01 * HALF_ULP[dtype] * ref.abs() + 2.0 ** -24
    err = (got.double() - ref).abs()
    assert bool((err <= lim).all()), (what, float((err - lim).max()), float(err.max()))


def _weights(codes, s, z, g, dtype):
    """(W, slack): the weights as the reference rounds them, None; for fp16 with
    fp16 fractional zero points the unrounded ones and how far a kernel's may be
    off: the zero point's fractional part times the scale, at most s / 2, is rounded
    to fp16 (by 2^-12 s), then the weight (by 2^-11 of it)."""
    if dtype != torch.float16 or z is None or s.dtype != torch.float16 or bool((z == z.round()).all()):
        return _rounded(codes, s, z, g, dtype), None
    full = s.double().repeat_interleave(g, 1)[:, : codes.shape[1]]
    W = (codes.double() - z.double().repeat_interleave(g, 1)[:, : codes.shape[1]]) * full
    return W, 2.0 ** -12 * full + 2.0 ** -11 * W.abs()


def _check_rows(got, x, codes, s, z, g, bits, what):
    """_check, with the rows past the last pass of 32 (q4 1-4, q8 1-2; fp16 with
    fp16 scales in whole vectors) held to the weights that are not rounded: the
    v_dot2 kernel takes those.  It sums x * (c + offset), offset 64 (q8: 1024),
    and subtracts the offset's part, so that its sums are K * 2^-24 of that."""
    (M, K), dtype, G = x.shape, x.dtype, s.shape[1]
    dot = (dtype == torch.float16 and s.dtype == torch.float16 and M > 32 and 0 < M % 32 <= (4 if bits == 4 else 2)
           and K % 128 == 0 and K <= 16384 and G % 8 == 0 and g <= 256)
    m = M - M % 32 if dot else M
    W, slack = _weights(codes, s, z, g, dtype)
    _check(got[:m], x[:m], W, dtype, what, slack)
    if dot:
        full = s.double().repeat_interleave(g, 1)[:, :K]
        W = (codes.double() - (0.0 if z is None else z.double().repeat_interleave(g, 1)[:, :K])) * full
        xd = x[m:].double()
        ref, top = xd @ W.t(), 80 if bits == 4 else 1280
        bound = K * 2.0 ** -24 * (xd.abs() @ (top * full).t()) + 1.01 * HALF_ULP[dtype] * ref.abs() + 2.0 ** -24
        assert bool(((got[m:].double() - ref).abs() <= bound).all()), (what, "rows past the last pass")


CASES = [  # M, N, K: the smallest; ragged N and K, one past a column tile; tiles of 64 and 128 rows and one more
    (33, 4, 32), (40, 101, 96), (64, 257, 2080), (65, 515, 1024), (128, 64, 4096), (129, 1030, 512),
    # many tiles of output rows (8 x 8), few of them over a long K (8 x 1 x 4, 4 x 2 x 4, 4 x 1 x 4), and between (8 x 2 x 2)
    (509, 14336, 256), (500, 4096, 1056), (256, 2048, 14336), (72, 1024, 7168), (130, 6144, 4096)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", CASES)
def test_product_rows(dev, M, N, K, bits, dtype):
    gen = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).to(dtype)
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    for g, sdt, zeros in ((64, torch.float16, "whole"), (32, torch.float16, "none"), (128, torch.float32, "affine"),
                          (64, torch.float16, "affine")):
        codes, packed, s, z = _weight(gen, dev, N, K, bits, g, sdt, zeros)
        got = fn(x, packed, s, z, group_size=g)
        _check_rows(got, x, codes, s, z, g, bits, f"M{M} N{N} K{K} q{bits} g{g} {sdt} {zeros}")
        res = torch.randn((M, N), generator=gen, device=dev).to(dtype)
        mm, out = qo.q_matvec_residual(x, packed, s, z, res, bits=bits, group_size=g, want_mm=True)
        assert torch.equal(mm, got)
        assert torch.equal(out, (res.float() + mm.float()).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(33, 7, 64), (65, 260, 160), (200, 1024, 1024), (509, 14336, 128)])
def test_product_gate_up(dev, M, N, K, bits, dtype):
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).to(dtype)
    cg, gw, gs, gz = _weight(gen, dev, N, K, bits, 32, torch.float16, "whole")
    cu, uw, us, uz = _weight(gen, dev, N, K, bits, 32, torch.float16, "whole")
    gate, up, mlp = qo.q_gate_up_swiglu(x, gw, uw, gs, us, gz, uz, bits=bits, group_size=32, return_gate_up=True)
    _check_rows(gate, x, cg, gs, gz, 32, bits, "gate")
    _check_rows(up, x, cu, us, uz, 32, bits, "up")
    gf = gate.double()
    want = gf / (1 + torch.exp(-gf)) * up.double()
    # silu in fp32 (a few 2^-24), the product rounded once
    assert bool(((mlp.double() - want).abs() <= 1.01 * HALF_ULP[dtype] * want.abs() + 2.0 ** -24).all())


@pytest.mark.parametrize("bits", [4, 8])
def test_product_unaligned_scales_and_saturation(dev, bits):
    """Scales 2 bytes off (copied one by one) give the aligned result; sums
    past fp16 saturate."""
    gen = torch.Generator(device=dev).manual_seed(3)
    M, N, K, g = 70, 130, 1024, 64
    x = torch.randn((M, K), generator=gen, device=dev).half()
    _, packed, s, z = _weight(gen, dev, N, K, bits, g, torch.float16, "whole")
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    want = fn(x, packed, s, z, group_size=g)
    off = lambda t: torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)[1:].reshape(t.shape).copy_(t)
    assert torch.equal(fn(x, packed, off(s), off(z), group_size=g), want)
    big = fn(torch.full((40, K), 200.0, device=dev).half(), packed, s * 400, None, group_size=g)
    assert bool((big == 65504.0).all())


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K,g", [(96, 32), (96, 64), (1056, 128), (2080, 32)])
def test_product_past_k_with_large_weights(dev, bits, K, g):
    """The last stage past K adds nothing, also where the last group's scale
    would make an infinite fp16 weight of other codes than its own (they re-read
    the row's first ones), and where the row's own first weights are infinite:
    those give the saturated sum, as in the reference."""
    gen = torch.Generator(device=dev).manual_seed(K + g)
    M, N, top = 70, 70, 15 if bits == 4 else 255
    codes = torch.full((N, K), top, dtype=torch.uint8, device=dev)
    codes[:, (K - 1) // g * g:] = 2
    s = torch.full((N, -(-K // g)), 1e-3, device=dev).half()
    s[:, -1] = 2 * 65504.0 / top  # top * s is past fp16, the group's own 2 * s is not
    packed = codes[:, 0::2] | (codes[:, 1::2] << 4) if bits == 4 else codes
    x = (torch.randn((M, K), generator=gen, device=dev) * 0.01).half()
    x[:, (K - 1) // g * g:] *= 0.01
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    _check(fn(x, packed.contiguous(), s, None, group_size=g), x, _rounded(codes, s, None, g, torch.float16),
           torch.float16, (K, g))
    s[:] = 1e-3
    s[:, 0] = 2 * 65504.0 / top
    got = fn(x.abs() + 1e-3, packed.contiguous(), s, None, group_size=g)
    assert bool((got == 65504.0).all())
