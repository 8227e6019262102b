"""Gate/up pairs of which only one matrix has zero points (the two arguments are
independent, ops/quant_ops.py:634-738): the products, the fused front and the
whole block against the reference's values, at the row counts and sizes of
every kernel that a pair with both zero points takes."""

import pytest
import torch

import mk.quant_ops as qo
from mk.mlp_block_ops import quantized_mlp_block
from tests.test_gpu_gemm_rows import _check, _rounded, _weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(1, 300, 512), (2, 64, 512), (4, 300, 1024), (8, 300, 512), (20, 100, 512),
                                   (40, 300, 512), (8, 34, 96)])
def test_one_zero_point_tensor(dev, M, N, K, bits, dtype, first):
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    g = 64 if K % 64 == 0 else 32
    x = torch.randn((M, K), generator=gen, device=dev).to(dtype)
    for sdt in (torch.float16, torch.float32):
        cg, gw, gs, gz = _weight(gen, dev, N, K, bits, g, sdt, "whole" if first else "none")
        cu, uw, us, uz = _weight(gen, dev, N, K, bits, g, sdt, "none" if first else "whole")
        gate, up, mlp = qo.q_gate_up_swiglu(x, gw, uw, gs, us, gz, uz, bits=bits, group_size=g, return_gate_up=True)
        _check(gate, x, _rounded(cg, gs, gz, g, dtype), dtype, ("gate", sdt))
        _check(up, x, _rounded(cu, us, uz, g, dtype), dtype, ("up", sdt))
        # the front: the same products of the normalised rows that it returns
        nw = torch.ones(K, device=dev, dtype=dtype)
        z, normed, gate, up, mlp = qo.q_rmsnorm_gate_up_swiglu(x, x, nw, gw, uw, gs, us, gz, uz, bits=bits, group_size=g,
                                                               return_gate_up=True)
        _check(gate, normed, _rounded(cg, gs, gz, g, dtype), dtype, ("front gate", sdt))
        _check(up, normed, _rounded(cu, us, uz, g, dtype), dtype, ("front up", sdt))
        # the block: equal to its two calls
        _, dw, ds, dz = _weight(gen, dev, K, N, bits, g, sdt, "whole")
        out = quantized_mlp_block(x[:, None], x[:, None], nw, gw, gs, uw, us, dw, ds, gate_zeros=gz, up_zeros=uz,
                                  down_zeros=dz, bits=bits, group_size=g)
        _, want = qo.q_matvec_residual(mlp, dw, ds, dz, z, bits=bits, group_size=g)
        assert torch.equal(out[:, 0], want)
