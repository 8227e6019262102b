"""Rows past the last whole pass of a batch (1-4, q8 1-2, after passes of 32 or
16): the same bits as when these rows are called alone, that is from the v_dot2
kernel, which does not round W."""

import pytest
import torch

import mk.quant_ops as qo
from tests.test_gpu_gemm_rows import _check, _rounded, _weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,M,K,g,tail", [
    (4, 33, 4096, 64, 1), (4, 36, 1024, 32, 4), (4, 66, 14336, 64, 2), (4, 131, 2048, 128, 3), (4, 35, 5120, 64, 3),
    (4, 19, 960, 128, 3), (8, 33, 1024, 64, 1), (8, 66, 4096, 32, 2), (8, 17, 992, 128, 1)])
def test_tail_rows_alone(dev, bits, M, K, g, tail):
    gen = torch.Generator(device=dev).manual_seed(M + K)
    N = 300
    x = torch.randn((M, K), generator=gen, device=dev).half()
    res = torch.randn((M, N), generator=gen, device=dev).half()
    codes, packed, s, z = _weight(gen, dev, N, K, bits, g, torch.float16, "whole")
    fn = qo.q4_matvec_decode if bits == 4 else qo.q8_matvec_decode
    got, alone = fn(x, packed, s, z, group_size=g), fn(x[M - tail:], packed, s, z, group_size=g)
    assert torch.equal(got[M - tail:], alone)
    _check(got[: M - tail], x[: M - tail], _rounded(codes, s, z, g, torch.float16), torch.float16, (M, K))
    mm, out = qo.q_matvec_residual(x, packed, s, z, res, bits=bits, group_size=g, want_mm=True)
    assert torch.equal(mm, got) and torch.equal(out, (res.float() + mm.float()).half())


@pytest.mark.parametrize("bits,M,N,K,g,tail", [
    (4, 34, 300, 4096, 64, 2), (4, 20, 4096, 4096, 32, 4), (4, 33, 64, 8192, 64, 1), (8, 34, 300, 1024, 64, 2)])
def test_tail_rows_gate_up(dev, bits, M, N, K, g, tail):
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).half()
    cg, gw, gs, gz = _weight(gen, dev, N, K, bits, g, torch.float16, "whole")
    cu, uw, us, uz = _weight(gen, dev, N, K, bits, g, torch.float16, "whole")
    call = lambda v: qo.q_gate_up_swiglu(v, gw, uw, gs, us, gz, uz, bits=bits, group_size=g, return_gate_up=True)
    for a, b in zip(call(x), call(x[M - tail:])):
        assert torch.equal(a[M - tail:], b)
    gate, up, _ = call(x)
    _check(gate[: M - tail], x[: M - tail], _rounded(cg, gs, gz, g, torch.float16), torch.float16, "gate")
    _check(up[: M - tail], x[: M - tail], _rounded(cu, us, uz, g, torch.float16), torch.float16, "up")
