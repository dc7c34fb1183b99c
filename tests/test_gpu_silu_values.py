"""silu of every number of 16 bits (csrc/common.h: silu_of_dtype), against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_of_every_number(dtype):
    from minivllm_amd import hip_ops as H

    a = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dtype).view(64, 1024)
    y = H.silu_and_mul(torch.cat((a, torch.ones_like(a)), 1).to("cuda:0")).cpu()
    x = a.double()
    want = x / (1 + torch.exp(-x))
    finite = torch.isfinite(x)
    up = y.double()
    # half the distance to a neighbour, and the few ulp of fp32 by which exponential and quotient are off; below the exponential's range (fp32 overflows
    # at 88.7) a zero, and the dtype's own denormal numbers
    off = (up - want).abs()
    tiny = torch.finfo(dtype).smallest_normal * torch.finfo(dtype).eps
    assert (off <= (0.5 * torch.finfo(dtype).eps * 2.0 ** torch.floor(torch.log2(want.abs().clamp_min(1e-300)))) * (1 + 2**-12) + 4 * tiny)[finite & (x > -88.7)].all()
    assert (up[finite & (x < -88.75)] == 0).all()
    assert y[x == torch.inf] == torch.inf and torch.isnan(y[torch.isnan(x)]).all() and torch.isnan(y[x == -torch.inf]).all()
