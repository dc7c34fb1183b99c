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


def _call(H, s, ins, spans, state):
    """ins: the rows of all sequences -> their outputs and the states left (sequence i at slot i)."""
    cu = lambda v: torch.tensor([0, *torch.tensor(v).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    x, beta, a, bias, a_log = ins
    left, slots = state.clone(), torch.arange(len(spans), dtype=torch.int32, device=DEV)
    out = H.delta_prefill(s, x, beta, a, bias, a_log, left, slots, cu([t for t, _ in spans]), cu([t + b for t, b in spans]), max(t for t, _ in spans))
    return out.double(), [left[(t + b) & 1, i].double() for i, (t, b) in enumerate(spans)]


def _inputs(H, seed, tokens, heads, p, n, speed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    s = H.DeltaShape(heads, heads, p, n, heads * p, heads * (p + n), p, n ** -0.5, True)
    bias = torch.full((heads * n,), speed, device=DEV).bfloat16() if speed is not None else rand(heads * n) - 4
    return s, (rand(tokens, s.channels), rand(tokens, heads + 8)[:, :heads], rand(tokens, heads * n), bias, rand(heads)), rand


# nothing decays: what a segment makes of the state ahead of it is then all but the state itself; segments of two chunks and more
@pytest.mark.parametrize("tokens", [700, 1500])
@pytest.mark.parametrize("heads, p, n", [(4, 128, 128), (2, 144, 160), (3, 48, 96)])
@pytest.mark.parametrize("speed", [-20.0, None])
def test_segments_keep_the_state_as_exactly_as_whole_sequences(H, monkeypatch, tokens, heads, p, n, speed):
    """The kept state against the recurrence in 64 bits."""
    ratios = []
    for seed in range(4):
        s, ins, rand = _inputs(H, seed, tokens, heads, p, n, speed)
        x, beta, a, bias, a_log = (t.double() for t in ins)
        state = rand(2, 1, heads, n, p).float() * 0.3
        v, k, q = (t.unflatten(1, (heads, -1)) for t in x.split([heads * p, heads * n, heads * n], 1))
        k = k / (k.square().sum(-1, keepdim=True) + 1e-6).sqrt()
        decay = (-a_log.exp()[:, None] * torch.nn.functional.softplus((a + bias).unflatten(1, (heads, n)), threshold=60.0)).exp()
        want = state[1, 0].double()
        for t in range(tokens):
            want = want * decay[t][:, :, None]
            u = beta[t].sigmoid()[:, None] * (v[t] - (k[t][:, None] @ want)[:, 0])
            want = want + k[t][:, :, None] * u[:, None]
        got = _call(H, s, ins, [(tokens, 1)], state)[1][0]
        with monkeypatch.context() as m:
            m.setattr(H._lib, "mv_delta_prefill_segments_bytes", lambda *a: 0)
            whole = _call(H, s, ins, [(tokens, 1)], state)[1][0]
        assert not torch.equal(got, whole)
        error, other = ((t - want).norm() / want.norm() for t in (got, whole))
        # operands are sums of two bf16 numbers, 2^-17 of them off at most; a few such roundings of a state live at a time
        assert error <= 2 ** -16
        ratios.append(float(error / other))
    # four draws scatter by 1 % around 1; with the diagonal in two bf16 numbers and the product of the rests left out 1.05 to 1.09 (700 tokens that do not decay)
    assert sum(ratios) / len(ratios) <= 1.02, ratios


def test_a_sequence_alone_and_among_others(H):
    """Its segments depend on the others: the last bits may, the rest does not."""
    lens, heads, p, n = [2500, 700, 1900, 130], 4, 128, 128
    s, ins, rand = _inputs(H, 0, sum(lens), heads, p, n, None)
    state = rand(2, len(lens), heads, n, p).float() * 0.3
    out, states = _call(H, s, ins, [(t, 3) for t in lens], state)
    at = 0
    for i, t in enumerate(lens):
        rows = [r[at:at + t] for r in ins[:3]] + list(ins[3:])
        alone, kept = _call(H, s, rows, [(t, 3)], state[:, i:i + 1].contiguous())
        got = out[at:at + t]
        # (each 2^-17 of its operands off; results rounded once to 8 bits, which may fall either way)
        assert (got - alone).norm() <= 2 ** -10 * alone.norm()
        assert ((got - alone).abs() <= 2 ** -7 * alone.abs() + 2 ** -14 * alone.abs().max()).all()
        assert (states[i] - kept[0]).norm() <= 2 ** -15 * kept[0].norm()
        at += t
