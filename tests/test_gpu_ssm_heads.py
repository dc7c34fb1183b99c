"""State space recurrence of four heads a workgroup, chunks of all sequences dealt out evenly (csrc/ssm_heads.hip), against token by token."""
import pytest
import torch

from test_gpu_ssm_segments import DEV, H, _case  # noqa: F401

pytestmark = pytest.mark.gpu


def _scratch(H, case):
    """Bytes without and with what the kernel of four heads needs."""
    (x, _, _, _, _, (heads, _, p, n, _, _), _, slots, _, _, longest) = case
    of = (slots.numel(), x.shape[0], longest, heads, p, n)
    return [H._lib.mv_ssm_prefill_workspace_bytes(*of, H._dt(x) | f) for f in (0, H.MV_SSM_SHARED)]


# a row of workgroups that ends with a sequence, within one and behind several; sequences of one token, none, and one of several rows; states that
# sequences come with, a sequence without a slot (the last)
LONG = [(1900, 5), (1700, 0), (1500, 64), (1301, 1)]
RAGGED = [(1, 3)] * 40 + [(0, 0), (3000, 2), (0, 9), (65, 0), (1500, 0), (64, 3)]
SHORT = [(64, 0)] * 70 + [(2049, 7)] * 2
FOUR = [(1900, 5), (1899, 0), (1857, 64), (1856, 1)]
MANY = [(1900, 0), (1300, 2), (960, 7), (1700, 0), (1500, 1), (1000, 0), (1200, 3), (1850, 64)]
CASES = {"long": (LONG, [(64, 1, 128), (64, 1, 64)]), "ragged": (RAGGED, [(64, 1, 128), (32, 2, 64), (24, 2, 128), (64, 4, 64)]),
         "short": (SHORT, [(32, 2, 64), (24, 2, 128), (32, 1, 128)]), "four": (FOUR, [(32, 2, 64), (32, 8, 128), (64, 1, 64)]),
         "many": (MANY, [(32, 1, 64), (24, 2, 128)])}


@pytest.mark.parametrize("spans, heads, groups, n", [pytest.param(s, *shape, id=f"{k}-{shape}") for k, (s, shapes) in CASES.items() for shape in shapes])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_heads(H, spans, heads, groups, n, dtype):  # noqa: F811
    case = _case(spans, heads, groups, 64, n, dtype, H)
    assert _scratch(H, case)[1] > _scratch(H, case)[0]      # (this kernel's: it is what runs)
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


# heads that share with fewer than three others, columns other than 64, and sizes at which a head a workgroup is as fast: the other kernel's, whatever the scratch memory
@pytest.mark.parametrize("spans, heads, groups, p, n", [(LONG, 64, 32, 64, 128), (LONG, 6, 1, 64, 64), (FOUR, 32, 1, 32, 64), (FOUR, 32, 1, 64, 96), (LONG, 32, 2, 64, 64),
                                                        (SHORT, 64, 1, 64, 128), ([(320, 1)] * 3, 32, 1, 64, 64)], ids=str)
def test_what_stays_with_a_head_a_workgroup(H, monkeypatch, spans, heads, groups, p, n):  # noqa: F811
    case = _case(spans, heads, groups, p, n, torch.bfloat16, H)
    without = _scratch(H, case)[0]
    runs = []
    for more in (0, 1 << 27):
        monkeypatch.setattr(H._lib, "mv_ssm_prefill_workspace_bytes", lambda *a: without + more if without else 0)
        state = case[6].clone()
        runs.append((H.ssm_prefill(*case[:6], state, *case[7:]), state))
    assert all(torch.equal(a, b) for a, b in zip(*runs))
    monkeypatch.undo()
    state = case[6].clone()
    got = H.ssm_prefill(*case[:6], state, *case[7:])
    assert torch.equal(got, runs[0][0]) and torch.equal(state, runs[0][1])


@pytest.mark.parametrize("spans, heads, groups, n", [(FOUR, 32, 2, 64), (RAGGED, 64, 1, 128)], ids=["four", "ragged"])
@pytest.mark.parametrize("whole", [False, True])
def test_a_sequence_alone_and_among_others(H, monkeypatch, spans, heads, groups, n, whole):  # noqa: F811
    """The same bits without scratch memory; with it, where a sequence is cut goes by the others: fp32 sums in another order."""
    case = _case(spans, heads, groups, 64, n, torch.bfloat16, H)
    x, dt, bias, a_log, d, shape, state, slots, _, _, _ = case
    if whole:
        monkeypatch.setattr(H._lib, "mv_ssm_prefill_workspace_bytes", lambda *a: 0)
    else:
        assert _scratch(H, case)[1] > _scratch(H, case)[0]
    left = state.clone()
    out = H.ssm_prefill(*case[:6], left, *case[7:])
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    begin = 0
    for (t, before), slot in zip(spans, slots.tolist()):
        rows, begin = slice(begin, begin + t), begin + t
        if t < 64:
            continue
        kept = state[:, max(slot, 0):max(slot, 0) + 1].contiguous()
        alone = H.ssm_prefill(x[rows], dt[rows], bias, a_log, d, shape, kept, ints(min(slot, 0)), ints(0, t), ints(0, t + before), t)
        side = (t + before) & 1
        if whole:
            assert torch.equal(out[rows], alone) and (slot < 0 or torch.equal(left[side, slot], kept[side, 0]))
        else:
            torch.testing.assert_close(out[rows].float(), alone.float(), rtol=2 ** -7, atol=2 ** -11 * alone.float().abs().max().item())
            # (each within 2^-17 of token by token)
            assert slot < 0 or ((left[side, slot] - kept[side, 0]).norm() / kept[side, 0].norm()).item() < 2 ** -16
