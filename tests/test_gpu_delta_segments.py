"""Gated delta rule of few long sequences, cut into segments (csrc/delta_chunk.hip), against the same kernel on whole sequences."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


def _both(H, monkeypatch, spans, heads, groups, p, n, dtype, channel, skew=0, speed=None, equal_keys=False):
    """spans: (tokens, tokens before) of the sequences; the last of several has no slot."""
    g = torch.Generator(device=DEV).manual_seed(len(spans) * 1000 + p + n)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    cu = lambda v: torch.tensor([0, *torch.tensor(v).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    total, longest = sum(t for t, _ in spans), max(t for t, _ in spans)
    s = H.DeltaShape(heads, groups, p, n, heads * p, heads * p + groups * n, p, n ** -0.5, channel)
    width = heads * (n if channel else 1)
    x, beta, a = rand(total, s.channels).to(dtype), rand(total, heads + -heads % 8).to(dtype)[:, :heads], rand(total, width + -width % 8).to(dtype)[:, :width]
    if equal_keys:
        x[:, s.k_off:s.k_off + groups * n] = x[:1, s.k_off:s.k_off + groups * n]
    # steps between 0.002 and 0.1 without `speed`
    bias = (rand(width) - 4 if speed is None else torch.full((width,), speed, device=DEV)).to(dtype)
    a_log = rand(heads).to(dtype)
    cq, ck = cu([t for t, _ in spans]), cu([t + b for t, b in spans])
    slots = torch.tensor([*range(len(spans))][::-1][:-1] + [-1] if len(spans) > 1 else [0], dtype=torch.int32, device=DEV)
    state = rand(2, len(spans), heads, n, p) * 0.3

    def run():
        left, out = state.clone(), torch.full((total, heads * p + 8 + skew), 7.0, dtype=dtype, device=DEV)
        H.delta_prefill(s, x, beta, a, bias, a_log, left, slots, cq, ck, longest, out=out[:, skew:skew + heads * p])
        assert (out[:, skew + heads * p:] == 7).all() and (out[:, :skew] == 7).all()
        return out[:, skew:skew + heads * p].double(), left.double()

    assert H._lib.mv_delta_prefill_segments_bytes(len(spans), total, longest, heads, p, n, channel, H._dt(x)) > 0
    got, left = run()
    with monkeypatch.context() as m:
        m.setattr(H._lib, "mv_delta_prefill_segments_bytes", lambda *a: 0)
        want, kept = run()
    assert torch.isfinite(got).all()
    # operands are sums of two bf16 numbers (2^-17 of them): a few of those where the state goes from segment to segment; results rounded once more
    unit = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11
    assert (got - want).norm() <= max(unit, 2 ** -12) * want.norm()
    assert ((got - want).abs() <= 2 * unit * want.abs() + 2 ** -10 * want.abs().max()).all()
    assert (left - kept).norm() <= 2 ** -14 * kept.norm()
    untouched = [(h, int(slots[i])) for i, (t, b) in enumerate(spans) for h in (0, 1) if slots[i] >= 0 and (t == 0 or h != (b + t) & 1)]
    for h, i in untouched:
        assert torch.equal(left[h, i], state[h, i].double())


# around the lengths at which a sequence gets one more segment (two chunks of 64 tokens and up; from 577 tokens on), beside short ones and empty ones
@pytest.mark.parametrize("spans", [[(577, 7)], [(640, 0), (1, 0)], [(768, 3), (64, 0)], [(641, 7), (0, 5), (70, 0), (640, 3)], [(2500, 0), (33, 5)],
                                   [(1000, 2), (999, 1), (40, 0)]], ids=str)
@pytest.mark.parametrize("heads, p, n", [(4, 128, 128), (3, 48, 32), (2, 144, 160), (5, 16, 96), (2, 208, 64)])
@pytest.mark.parametrize("dtype, skew", [(torch.bfloat16, 0), (torch.bfloat16, 1), (torch.float16, 0)])
def test_segments_are_whole_sequences(H, monkeypatch, spans, heads, p, n, dtype, skew):
    if n == 32:     # cut from 897 tokens on
        spans = [(t + 320 if t > 500 else t, b) for t, b in spans]
    _both(H, monkeypatch, spans, heads, heads, p, n, dtype, True, skew)


@pytest.mark.parametrize("heads, groups, p, n", [(4, 2, 128, 128), (6, 6, 64, 64)])
def test_one_decay_per_head_in_fp16(H, monkeypatch, heads, groups, p, n):
    _both(H, monkeypatch, [(1000, 2), (577, 1), (40, 0)], heads, groups, p, n, torch.float16, False)


@pytest.mark.parametrize("spans", [[(4000, 5), (3500, 0), (2000, 64)], [(4011, 3)]], ids=str)
def test_segments_sized_by_the_work_of_many_heads(H, monkeypatch, spans):
    _both(H, monkeypatch, spans, 8, 8, 128, 128, torch.bfloat16, True)


@pytest.mark.parametrize("speed", [-20.0, 9.0])
@pytest.mark.parametrize("equal_keys", [False, True])
def test_states_that_never_decay_and_vanish_at_once(H, monkeypatch, speed, equal_keys):
    _both(H, monkeypatch, [(1500, 3)], 4, 4, 64, 64, torch.bfloat16, True, speed=speed, equal_keys=equal_keys)


def test_less_scratch_is_whole_sequences(H, monkeypatch):
    """A workspace of the size asked for before there were segments."""
    s = H.DeltaShape(2, 2, 64, 64, 128, 256, 64, 0.125, True)
    g = torch.Generator(device=DEV).manual_seed(0)
    rand = lambda *sh: torch.randn(*sh, generator=g, device=DEV).bfloat16()
    t = 1500
    args = s, rand(t, s.channels), rand(t, 8)[:, :2], rand(t, 128), rand(128), rand(2)
    cu = torch.tensor([0, t], dtype=torch.int32, device=DEV)
    outs = []
    for less in (0, 1):
        need = H._lib.mv_delta_prefill_segments_bytes(1, t, t, 2, 64, 64, 1, H._dt(args[1]))
        with monkeypatch.context() as m:
            m.setattr(H._lib, "mv_delta_prefill_segments_bytes", lambda *a: need - 1 if less else 0)
            outs.append(H.delta_prefill(*args, torch.zeros(2, 1, 2, 64, 64, device=DEV), cu[:1], cu, cu, t))
    assert torch.equal(*outs)
