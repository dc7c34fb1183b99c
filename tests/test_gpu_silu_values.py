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


def test_silu_of_bf16_has_the_divisions_bits():
    """Every bf16 gate above fp32's last exponential: x / (1 + exp(-x)) of 64 bits, rounded once, to the bit, as fp32's division gives it too; below, a zero."""
    from minivllm_amd import hip_ops as H

    a = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(64, 1024)
    y = H.silu_and_mul(torch.cat((a, torch.ones_like(a)), 1).to("cuda:0")).cpu()
    x = a.double()
    exact = x / (1 + torch.exp(-x))
    ulp = 2.0 ** (torch.floor(torch.log2(exact.abs().clamp_min(1e-300))).clamp_min(-126) - 7)
    want = (torch.round(exact / ulp) * ulp).to(torch.bfloat16)      # (half to even; a number of bf16 already)
    there = torch.isfinite(x) & (x > -88.75)
    assert torch.equal(y.view(torch.int16)[there], want.view(torch.int16)[there])
    below = y[torch.isfinite(x) & (x < -88.75)]
    assert (below == 0).all() and below.signbit().all()
    wide = a.to("cuda:0").float()
    division = (wide / (1 + torch.exp(-wide))).bfloat16().cpu()
    assert torch.equal(y.view(torch.int16)[torch.isfinite(x)], division.view(torch.int16)[torch.isfinite(x)])


@pytest.mark.parametrize("rows, cols", [(153593, 1024), (65537, 2400), (19200, 8200)])
def test_results_that_go_past_the_last_cache(rows, cols):
    """More rows than a grid has, rows that the workgroups' vectors leave ragged, results of more than 300 MB: each row is that of a few rows alone."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device="cuda:0").manual_seed(cols)
    x = torch.randn(rows, 2 * cols, device="cuda:0", generator=g, dtype=torch.bfloat16)
    y = H.silu_and_mul(x)
    for at in (0, 40000 if rows > 65536 else 7000, rows - 64):
        assert torch.equal(y[at:at + 64], H.silu_and_mul(x[at:at + 64]))


@pytest.mark.parametrize("rows", [7918, 7919])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_sides_of_the_last_caches_line(dtype, act, rows):
    """Results of 299.997 and 300.035 MB (rows that lie apart, of which a few are asked for again)."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device="cuda:0").manual_seed(rows)
    x = torch.randn(rows, 2 * 18944 + 8, device="cuda:0", generator=g, dtype=dtype)[:, :2 * 18944]
    y = H.act_and_mul(x, act)
    for at in (0, 4000, rows - 16):
        assert torch.equal(y[at:at + 16], H.act_and_mul(x[at:at + 16], act))
