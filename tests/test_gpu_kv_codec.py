"""The vectorised KV quantizer and the KV dequantizer: bytes equal to the
row-per-thread kernel (reached through a source 8 bytes off a 16-byte
boundary) and to the tensor ops, at chunk, group and block edges."""

import pytest
import torch

import mk.paged_quantized_kv_ops as pq

pytestmark = pytest.mark.gpu

# (rows, D, g): one chunk; part of a block, one group per row; a block and a
# few lanes; groups of 1, 2, 16 and 64 lanes; then what the row-per-thread
# kernel and the value-per-thread kernel keep: ragged, odd and non-power-of-two groups
CASES = [(1, 8, 8), (3, 64, 64), (257, 128, 64), (65, 128, 8), (70, 96, 16), (33, 256, 128), (9, 512, 512),
         (5, 1024, 512), (7, 80, 64), (5, 15, 5), (6, 96, 24), (4, 130, 32)]


def _rows(rows, D, dtype, dev, special):
    g = torch.Generator().manual_seed(rows * 1000 + D)
    x = torch.randn(rows, D, generator=g) * torch.rand(rows, 1, generator=g) * 4
    if special:
        x[0, : D // 2] = 0.0
        x[-1, 0], x[-1, D - 1], x[rows // 2, 1] = float("inf"), float("nan"), float("-inf")
    return x.to(dtype).to(dev)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows,D,g", CASES)
def test_quantize_rows_same_bytes_on_both_kernels(dev, rows, D, g, bits, dtype):
    for special in (False, True):
        x = _rows(rows, D, dtype, dev, special)
        off = torch.empty(rows * D + 4, dtype=dtype, device=dev)[4:].reshape(rows, D)
        off.copy_(x)
        assert x.data_ptr() % 16 == 0 and off.data_ptr() % 16 == 8
        codes, scales = pq._hip_quantize_rows(x, g, bits)
        codes2, scales2 = pq._hip_quantize_rows(off, g, bits)
        assert torch.equal(codes, codes2) and torch.equal(scales.view(torch.int16), scales2.view(torch.int16))
        if not special:
            want, want_s = pq._quantize_last_dim(x.cpu().float(), g, bits)
            want = pq._pack_last_dim(want) if bits == 4 else want
            assert torch.equal(codes.cpu(), want) and torch.equal(scales.cpu(), want_s)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows,D,g", CASES)
def test_dequantize_equals_tensor_ops(dev, rows, D, g, bits):
    gen = torch.Generator().manual_seed(7)
    codes = torch.randint(0, 256, (rows, D if bits == 8 else (D + 1) // 2), generator=gen, dtype=torch.uint8)
    scales = (torch.randn(rows, -(-D // g), generator=gen) * 0.1).half()  # negative ones too: |s| counts
    scales[0, 0], scales[-1, -1] = 6e4, 6e-8  # a product past fp16, a subnormal scale
    flat = codes if bits == 8 else torch.stack((codes & 15, codes >> 4), -1).reshape(rows, -1)[:, :D]
    want = pq._dequant_last_dim(flat, scales, g, bits, D).half()
    got = pq._hip_dequantize(codes.to(dev), scales.to(dev), g, bits, D)
    assert torch.equal(got.cpu(), want)
    shifted = torch.empty(codes.numel() + 1, dtype=torch.uint8, device=dev)[1:].reshape(codes.shape)
    shifted.copy_(codes)
    assert torch.equal(pq._hip_dequantize(shifted, scales.to(dev), g, bits, D).cpu(), want)


def test_dequantize_leaves_other_forms_to_the_tensor_ops(dev):
    codes, scales = torch.zeros(2, 64, dtype=torch.uint8, device=dev), torch.ones(2, 1, dtype=torch.float16, device=dev)
    assert pq._hip_dequantize(codes.cpu(), scales.cpu(), 64, 8, 64) is None
    assert pq._hip_dequantize(codes, scales.float(), 64, 8, 64) is None
    assert pq._hip_dequantize(codes.int(), scales, 64, 8, 64) is None
    assert pq._hip_dequantize(codes, scales, 32, 8, 64) is None  # two groups per row expected
    assert pq._hip_dequantize(codes[:0], scales[:0], 64, 8, 64).shape == (0, 64)


@pytest.mark.parametrize("bits", [8, 4])
def test_dequantize_under_transforms(dev, bits):
    """Forward-mode, jvp, vmap and reverse-mode of both dequantizers over the
    scales: the tensor ops' values and tangents."""
    import dataclasses

    import torch.autograd.forward_ad as fwAD

    import mk.quantized_kv_cache_ops as qc

    gen = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(3, 16, 2, 64, generator=gen, device=dev).half()
    table = torch.arange(3, dtype=torch.int32, device=dev).reshape(1, 3)
    paged = pq.quantize_kv_pages(x, x, table, torch.tensor([48], dtype=torch.int32, device=dev),
                                 pq.PagedQuantizedKVConfig(bits=bits, page_size=16, group_size=32))
    flat = qc.quantize_kv_cache(x, x, qc.QuantizedKVCacheConfig(bits=bits, group_size=32))
    for cache, fn in ((paged, pq.dequantize_kv_pages), (flat, qc.dequantize_kv_cache)):
        f = lambda s: fn(dataclasses.replace(cache, k_scales=s))[0]
        s, t = cache.k_scales, torch.randn(cache.k_scales.shape, generator=gen, device=dev).half()
        off = fn(dataclasses.replace(cache, k_scales=torch.ones_like(s)))[0].float()  # code - 128 | 8
        want_t = (off * t.float().repeat_interleave(32, dim=-1)).half()  # scales are positive
        with fwAD.dual_level():
            out = fwAD.unpack_dual(f(fwAD.make_dual(s, t)))
            assert torch.equal(out.primal, f(s)) and torch.equal(out.tangent, want_t)
        val, tan = torch.func.jvp(f, (s,), (t,))
        assert torch.equal(val, f(s)) and torch.equal(tan, want_t)
        sg = s.clone().requires_grad_(True)
        f(sg).float().sum().backward()
        want_g = off.half().float().unflatten(-1, (-1, 32)).sum(-1)
        assert torch.allclose(sg.grad.float(), want_g, rtol=2e-3, atol=1e-2)
    rows = torch.stack([paged.k_scales, paged.k_scales * 2])
    got = torch.func.vmap(lambda s: pq.dequantize_kv_pages(
        dataclasses.replace(paged, k_scales=s, v_scales=s))[0])(rows)
    for i in range(2):
        assert torch.equal(got[i], pq.dequantize_kv_pages(dataclasses.replace(paged, k_scales=rows[i]))[0])
