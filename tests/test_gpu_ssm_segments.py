"""State space recurrence of few long sequences, cut into segments (csrc/ssm_chunk.hip), against the same kernel on whole sequences."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


def _case(spans, heads, groups, p, n, dtype, H):
    """spans: (tokens, tokens before) of the sequences; the last of several has no slot.  -> arguments of ssm_prefill, with the states"""
    g = torch.Generator(device=DEV).manual_seed(len(spans) * 1000 + p)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    up = lambda v: -(-v // 64) * 64
    total, b_off = sum(a for a, _ in spans), up(heads * p)
    c_off = b_off + up(groups * n)
    shape, channels = (heads, groups, p, n, b_off, c_off), c_off + groups * n
    x, dt = rand(total, channels).to(dtype), (rand(total, heads) - 2).to(dtype)
    bias, a_log, d = (rand(heads).to(dtype) for _ in range(3))
    cu = lambda v: ints([0, *torch.tensor(v).cumsum(0).tolist()])
    cq, ck, longest = cu([a for a, _ in spans]), cu([a + b for a, b in spans]), max(a for a, _ in spans)
    slots = ints([*range(len(spans))][::-1][:-1] + [-1] if len(spans) > 1 else [0])
    return x, dt, bias, a_log, d, shape, rand(2, len(spans), heads, n, p), slots, cq, ck, longest


def _both(H, monkeypatch, case, dtype):
    def run():
        state = case[6].clone()
        return H.ssm_prefill(*case[:6], state, *case[7:]), state

    (x, _, _, _, _, (heads, _, p, n, _, _), _, slots, _, _, longest) = case
    assert H._lib.mv_ssm_prefill_workspace_bytes(slots.numel(), x.shape[0], longest, heads, p, n, H._dt(x)) > 0
    got, state = run()
    monkeypatch.setattr(H._lib, "mv_ssm_prefill_workspace_bytes", lambda *a: 0)
    want, kept = run()
    # fp32 sums in another order, rounded once: a unit of the 16-bit result
    torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7 if dtype == torch.bfloat16 else 2 ** -10, atol=1e-3)
    torch.testing.assert_close(state, kept, rtol=1e-4, atol=1e-5)
    assert torch.isfinite(got).all()


# around the lengths at which a sequence gets one more segment (four chunks of 64 tokens and up; from 449 tokens on), beside short ones and empty slots
@pytest.mark.parametrize("spans", [[(449, 7)], [(512, 0), (1, 0)], [(576, 3), (64, 0)], [(513, 7), (70, 0), (512, 3)], [(2500, 0), (33, 5)],
                                   [(1000, 2), (999, 1), (40, 0)]], ids=str)
@pytest.mark.parametrize("heads, groups, p, n", [(4, 2, 64, 128), (3, 1, 48, 32), (2, 1, 80, 160), (6, 1, 32, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_segments_are_whole_sequences(H, monkeypatch, spans, heads, groups, p, n, dtype):
    _both(H, monkeypatch, _case(spans, heads, groups, p, n, dtype, H), dtype)


@pytest.mark.parametrize("spans", [[(4000, 5), (3500, 0), (2000, 64)], [(2500, 0), (2400, 3), (900, 1)]], ids=str)
def test_segments_sized_by_the_work_of_many_heads(H, monkeypatch, spans):
    """Ten and six chunks where the longest sequence alone would take eight and five: the workgroups of all heads even out at about four a CU."""
    _both(H, monkeypatch, _case(spans, 64, 8, 64, 128, torch.bfloat16, H), torch.bfloat16)


def _call(H, entry, case, *rest):
    x, dt, bias, a_log, d, shape, state, slots, cq, ck, longest = case
    state, out = state.clone(), torch.full((x.shape[0], shape[0] * shape[2]), 7.0, dtype=x.dtype, device=DEV)
    a = H._ssm_args(shape, x, slots, out, ssm_state=state, dt=dt, dt_bias=bias, a_log=a_log, d=d)
    a.cu_q, a.cu_k, a.max_q = cq.data_ptr(), ck.data_ptr(), longest
    H._check(entry(ctypes.byref(a), *rest, H._dt(x), 0, H._stream()), "ssm_prefill")
    return out, state


@pytest.mark.parametrize("spans", [[(900, 0), (400, 3)], [(470, 1)]], ids=str)
def test_calls_that_cannot_be_cut_are_whole_sequences(H, spans):
    """The entry point without scratch memory, too little of it, and a number of rows that no bound can be."""
    case = _case(spans, 4, 2, 64, 128, torch.bfloat16, H)
    want = _call(H, H._lib.mv_ssm_prefill, case)
    rows, longest = case[0].shape[0], case[-1]
    need = H._lib.mv_ssm_prefill_workspace_bytes(len(spans), rows, longest, 4, 64, 128, H._dt(case[0]))
    ws = torch.zeros(2 * need, dtype=torch.uint8, device=DEV)
    for size, total in ((need - 1, rows), (2 * need, 0), (2 * need, -5), (2 * need, longest - 1)):
        for got, kept in zip(_call(H, H._lib.mv_ssm_prefill_ws, case, ws.data_ptr(), size, total), want):
            assert torch.equal(got, kept), (size, total)


def test_states_that_never_decay_and_vanish_at_once(H, monkeypatch):
    heads, p, n, total = 2, 64, 64, 1500
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(total, heads * p + 2 * n, generator=g, device=DEV).bfloat16()
    for a in (-20.0, 9.0):
        dt = torch.full((total, heads), -1.0, device=DEV).bfloat16()
        vec = lambda v: torch.full((heads,), v, device=DEV).bfloat16()
        cu = torch.tensor([0, total], dtype=torch.int32, device=DEV)
        args = (x, dt, vec(0.0), vec(a), vec(0.5), (heads, 1, p, n, heads * p, heads * p + n))
        with monkeypatch.context() as m:
            got = [H.ssm_prefill(*args, torch.zeros(2, 1, heads, n, p, device=DEV), cu[:1], cu, cu, total)]
            m.setattr(H._lib, "mv_ssm_prefill_workspace_bytes", lambda *a: 0)
            got.append(H.ssm_prefill(*args, torch.zeros(2, 1, heads, n, p, device=DEV), cu[:1], cu, cu, total))
        assert torch.isfinite(got[0]).all()
        torch.testing.assert_close(got[0].float(), got[1].float(), rtol=2 ** -6, atol=1e-2)
