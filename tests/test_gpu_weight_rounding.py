"""The weights that the few-row and product kernels multiply with, read back one
by one: an activation row with a single 1 gives a column of W, exactly.

Layouts that the MFMA kernel of 16 rows does not take (q4: K % 64 = 32, q8: K %
32 = 16), bf16 activations and fp32 scales: (q - z) * s in fp32, rounded once,
for zero points whole, fractional and far from the codes.  fp16 weights
elsewhere: the same for whole zero points; a fractional one's addend is rounded
to fp16 first (|addend| <= s / 2, so by 2^-12 s at most)."""

import pytest
import torch

import mk.quant_ops as qo
from tests.test_gpu_gemm_rows import _rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,K,g", [(4, 96, 32), (4, 224, 64), (4, 1056, 128), (4, 2080, 256), (8, 80, 32), (8, 1040, 64),
                                      (4, 128, 32), (4, 1024, 64), (4, 2048, 128), (8, 96, 32), (8, 1024, 128)])
@pytest.mark.parametrize("dtype,sdt", [(torch.float16, torch.float16), (torch.bfloat16, torch.float16),
                                       (torch.float16, torch.float32)])
@pytest.mark.parametrize("M", [8, 24, 40, 80])
def test_weights_as_rounded(dev, M, bits, K, g, dtype, sdt):
    gen = torch.Generator(device=dev).manual_seed(M + K)
    N, top, G = 70, 1 << bits, -(-K // g)
    codes = torch.randint(0, top, (N, K), generator=gen, device=dev, dtype=torch.uint8)
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4) if bits == 4 else codes).contiguous()
    s = (torch.rand((N, G), generator=gen, device=dev) * 0.01 + 0.001).half()
    cols = torch.randperm(K, generator=gen, device=dev)[:M]
    cols[0] = K - 1
    x = torch.zeros((M, K), device=dev, dtype=dtype)
    x[torch.arange(len(cols), device=dev), cols] = 1
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    generic_layout = K % (64 if bits == 4 else 32) != 0
    for z in (None, torch.randint(0, top, (N, G), generator=gen, device=dev).half(),
              (torch.randint(0, 8 * top, (N, G), generator=gen, device=dev) / 8).half(),  # (q - z) * s: 22 bits, exact
              torch.randint(1100, 2000, (N, G), generator=gen, device=dev).half()):
        exact = generic_layout or dtype == torch.bfloat16 or sdt == torch.float32
        if z is not None and not exact and bool((z > 1000).all()):
            continue  # the exponent trick's range ends at 1024, as in the MFMA kernel
        W = _rounded(codes, s, z, g, dtype)
        got = fn(x, packed, s.to(sdt), None if z is None else z.to(sdt), group_size=g)[: len(cols)].double().t()
        want = W[:, cols]
        if exact or z is None or bool((z == z.round()).all()):
            assert torch.equal(got, want), (M, bits, K, g, float((got - want).abs().max()))
        else:
            full = s.double().repeat_interleave(g, 1)[:, :K][:, cols]
            true = (codes[:, cols].double() - z.double().repeat_interleave(g, 1)[:, :K][:, cols]) * full
            assert bool(((got - true).abs() <= 2.0 ** -11 * true.abs() + 2.0 ** -12 * full + 2.0 ** -24).all())
