"""Norm and gate behind the gated delta rule in the call itself (csrc/delta_scalar.hip where a workgroup has a head's columns) against the two calls.  The same
rounding points and orders of sums, so the same bits."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = (1, 63, 64, 65, 200, 2)


def _compare(heads, groups, p, p_true, n, dtype=torch.bfloat16, lens=LENS, gate_kind="silu", channel=False, out_scale=1.0, flags=0, skew=0):
    from minivllm_amd import hip_ops as H

    gen = torch.Generator(device=DEV).manual_seed(p * 1000 + n)
    rand = lambda *shape: torch.empty(shape, device=DEV).normal_(0, 1, generator=gen).to(dtype)
    t, width = sum(lens), heads * p + 2 * groups * n
    s = H.DeltaShape(heads, groups, p, n, heads * p, heads * p + groups * n, p_true, n ** -0.5, channel, 1e-6)
    x, beta, gate = rand(t, width), rand(t, heads), rand(t, heads * p + skew)[:, skew:]
    a, bias = rand(t, heads * (n if channel else 1)), rand(heads * (n if channel else 1))
    a_log, norm = rand(heads), rand(p)
    slots = torch.arange(len(lens), dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, *itertools.accumulate(lens)], dtype=torch.int32, device=DEV)
    first = torch.empty(2, len(lens), heads, n, p, device=DEV).normal_(0, 0.1, generator=gen)
    outs, states = [], []
    for fused in (True, False):
        state = first.clone()
        out = torch.full((t, heads * p + skew), 7.0, dtype=dtype, device=DEV)
        rest = dict(gate=gate, norm_w=norm, gate_kind=gate_kind, out_scale=out_scale, out=out[:, skew:]) if fused else {}
        o = H.delta_prefill(s, x, beta, a, bias, a_log, state, slots, cu, cu, max(lens), flags=flags, **rest)
        if not fused:
            H.head_norm_gate(o, gate, norm, heads, p, p_true, 1e-6, gate_kind, out_scale, out=out[:, skew:])
        outs.append(out), states.append(state)
    assert torch.equal(*outs), float((outs[0].float() - outs[1].float()).abs().max())
    assert torch.equal(*states)


# heads enough for workgroups of eight waves (more than 256 of four) or not; columns of a part of a workgroup, of all of it, of two; padded ones
@pytest.mark.parametrize("heads, p, p_true", [(3, 16, 16), (3, 48, 41), (2, 64, 64), (4, 128, 128), (32, 80, 80), (32, 128, 128), (32, 112, 100), (4, 144, 144)])
@pytest.mark.parametrize("n", [32, 128])
def test_in_the_call_or_behind_it(heads, p, p_true, n):
    _compare(heads, heads, p, p_true, n)


def test_gates_scales_strides_and_shared_keys():
    _compare(32, 16, 128, 128, 128, gate_kind="sigmoid", out_scale=0.5, skew=8)
    _compare(2, 1, 64, 64, 160, gate_kind="sigmoid", out_scale=2.0, skew=24, lens=(700, 1), flags=4)


# in the walk, whatever the rule on sizes says: every number of key channels, both numbers of waves, columns that fill a workgroup or not, more chunks than
# are under way, keys that two heads share
@pytest.mark.parametrize("heads, groups, p, p_true, n", [(*h, n) for n in (32, 64, 96, 128, 160) for h in (
    (3, 3, 16, 16), (2, 1, 48, 41), (4, 2, 64, 64), (32, 16, 80, 80), (32, 32, 112, 100), (32, 16, 128, 128)) if h[2] <= 64 or n <= 128])
@pytest.mark.parametrize("gate_kind, skew", [("silu", 0), ("sigmoid", 24)])
def test_in_the_walk(heads, groups, p, p_true, n, gate_kind, skew):
    from minivllm_amd import hip_ops as H

    lens = (1, 63, 450, 64, 65, 2)
    # eight waves have all columns of up to 128 where workgroups of four would be more than 256, up to 128 key channels; four have 64
    assert p <= 64 or (n <= 128 and -(-p // 64) * heads * len(lens) > 256)
    _compare(heads, groups, p, p_true, n, lens=lens, gate_kind=gate_kind, skew=skew, out_scale=0.5, flags=H.MV_DELTA_NORM_WALK)


@pytest.mark.parametrize("dtype, channel, flags", [(torch.float16, False, 0), (torch.float32, False, 0), (torch.bfloat16, True, 0), (torch.float16, True, 0), (torch.bfloat16, False, 1)])
def test_other_forms_norm_behind(dtype, channel, flags):
    _compare(2, 2, 64, 60, 64, dtype=dtype, channel=channel, flags=flags)
