"""State space recurrence of four heads a workgroup, chunks of all sequences dealt out evenly (csrc/ssm_heads.hip), against token by token."""
import pytest
import torch

from test_gpu_ssm_segments import H, _case  # noqa: F401

pytestmark = pytest.mark.gpu


# a row of workgroups that ends with a sequence, within one and behind several; sequences of one token, none, and one of several rows; states that
# sequences come with, a sequence without a slot (the last)
SPANS = [[(1900, 5), (1700, 0), (1500, 64), (1301, 1)], [(1, 3)] * 40 + [(0, 0), (3000, 2), (0, 9), (65, 0), (1500, 0), (64, 3)], [(64, 0)] * 70 + [(2049, 7)] * 2]


@pytest.mark.parametrize("spans", SPANS, ids=["long", "ragged", "short"])
@pytest.mark.parametrize("heads, groups, n", [(64, 1, 128), (32, 2, 64), (24, 2, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_heads(H, spans, heads, groups, n, dtype):  # noqa: F811
    case = _case(spans, heads, groups, 64, n, dtype, H)
    states = [case[6].clone() for _ in range(2)]
    got, want = (H.ssm_prefill(*case[:6], s, *case[7:], flags=f) for s, f in zip(states, (0, H.MV_SSM_SCAN)))
    # fp32 sums in another order, rounded once: a unit of the 16-bit result.  Weighted numbers are sums of two parts, off by 2^-17 of themselves at most
    unit = 2 ** -7 if dtype == torch.bfloat16 else 2 ** -10
    torch.testing.assert_close(got.float(), want.float(), rtol=unit, atol=unit * want.float().abs().max().item() * 2 ** -4)
    assert ((states[0] - states[1]).norm() / states[1].norm()).item() < 2 ** -17
    for (tokens, before), slot in zip(spans, case[7].tolist()):
        for side in (0, 1):   # (what is not written: the other half, both without a token)
            if slot >= 0 and not (tokens and side == (tokens + before) & 1):
                assert torch.equal(states[0][side, slot], case[6][side, slot])
