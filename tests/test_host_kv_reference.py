"""What must not reach the KV dequantize kernel: the reference backends, which
the kernels are compared with, and everything under MLX_METAL_CI_SAFE_MODE=1."""

import torch

import mk.paged_quantized_kv_ops as pq
import mk.quantized_kv_cache_ops as qc
import mk.speculative_verify_ops as sv


def test_reference_and_ci_safe_dequantize_use_tensor_ops(monkeypatch):
    gen = torch.Generator().manual_seed(1)
    x = torch.randn(3, 16, 2, 64, generator=gen).half()
    table = torch.arange(3, dtype=torch.int32).reshape(1, 3)
    paged = pq.quantize_kv_pages(x, x, table, torch.tensor([40], dtype=torch.int32),
                                 pq.PagedQuantizedKVConfig(bits=8, page_size=16, group_size=32))
    flat = qc.quantize_kv_cache(x, x, qc.QuantizedKVCacheConfig(bits=8, group_size=32))
    want = pq.dequantize_kv_pages(paged)[0], qc.dequantize_kv_cache(flat)[0]

    def kernel(*args):
        raise AssertionError("the kernel's wrapper was called")

    monkeypatch.setattr(pq, "_hip_dequantize", kernel)
    monkeypatch.setattr(qc, "_hip_dequantize", kernel)
    q = torch.randn(1, 1, 4, 64, generator=gen).half()
    pq.paged_quantized_kv_gqa_decode_attention(q, paged, backend="reference")
    sv.paged_quantized_verify_attention(torch.cat([q, q], 1), paged, backend="reference")
    qc.reference_quantized_kv_gqa_decode_attention(q.expand(3, -1, -1, -1), flat, torch.tensor([16, 3, 9]))
    monkeypatch.setenv("MLX_METAL_CI_SAFE_MODE", "1")
    assert torch.equal(pq.dequantize_kv_pages(paged)[0], want[0])
    assert torch.equal(qc.dequantize_kv_cache(flat)[0], want[1])
