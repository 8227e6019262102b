"""The MLP block in one library call against its two calls (norm + gate/up,
then down + residual): the same kernels on the same values, so the outputs are equal
bit for bit.  One row to
more than the workspace's 68, both weight types, hidden sizes with and without
a workspace for the down projection, inputs that are views."""

import pytest
import torch

from mk.mlp_block_ops import quantized_mlp_block
from mk.quant_ops import q_matvec_residual, q_rmsnorm_gate_up_swiglu

pytestmark = pytest.mark.gpu


def _linear(g, bits, n, k, gs, scale_dtype, zeros):
    cols = k if bits == 8 else (k + 1) // 2
    w = torch.randint(0, 256, (n, cols), generator=g, dtype=torch.uint8).cuda()
    groups = -(-k // gs)
    s = (torch.rand(n, groups, generator=g) * 0.01 + 0.001).to(scale_dtype).cuda()
    z = torch.full((n, groups), 7.0 if bits == 4 else 127.0).to(scale_dtype).cuda() if zeros else None
    return w, s, z


@pytest.mark.parametrize("shape,hidden,bits,gs,dtype,scale_dtype,zeros", [
    ((1, 1, 256), 512, 4, 32, torch.float16, torch.float16, True),
    ((1, 1, 96), 160, 8, 32, torch.bfloat16, torch.float32, False),
    ((4, 1, 512), 6144, 4, 64, torch.bfloat16, torch.float16, True),
    ((2, 16, 256), 8192, 8, 128, torch.float16, torch.float16, False),
    ((64, 1, 128), 4128, 4, 32, torch.float16, torch.float32, True),
    ((5, 13, 256), 512, 4, 32, torch.float16, torch.float16, True),
    ((66, 1, 128), 8192, 4, 64, torch.float16, torch.float16, True),  # two rows past the last pass, K slices
    ((3, 1, 33), 65, 4, 32, torch.float16, torch.float16, True),  # odd sizes
])
def test_block_equals_its_two_calls(shape, hidden, bits, gs, dtype, scale_dtype, zeros):
    g = torch.Generator().manual_seed(3)
    d = shape[2]
    gate, up = (_linear(g, bits, hidden, d, gs, scale_dtype, zeros) for _ in range(2))
    down = _linear(g, bits, d, hidden, gs, scale_dtype, zeros)
    x = torch.randn(shape[1], shape[0], d, generator=g).to(dtype).cuda().transpose(0, 1)
    r = torch.randn(shape, generator=g).to(dtype).cuda()
    nw = (torch.rand(d, generator=g) + 0.5).cuda()
    one = quantized_mlp_block(x, r, nw, gate[0], gate[1], up[0], up[1], down[0], down[1], gate_zeros=gate[2],
                              up_zeros=up[2], down_zeros=down[2], bits=bits, group_size=gs)
    z, _, mlp = q_rmsnorm_gate_up_swiglu(x, r, nw, gate[0], up[0], gate[1], up[1], gate[2], up[2], bits=bits,
                                         group_size=gs)
    _, two = q_matvec_residual(mlp, *down, z, bits=bits, group_size=gs)
    assert one.shape == x.shape and one.dtype == dtype
    assert torch.isfinite(one).all()
    assert torch.equal(one, two.reshape(shape))
