"""The gated delta rule's prompts from projected channels (the convolution along with the preparation of a chunk, csrc/delta_chunk.h, or ahead of it), against the
convolution and the rule in calls of their own: the same bits, the kept inputs among them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# (tokens, tokens before): fewer than the taps, around a chunk of 64 and two, halves of the kept inputs that are the same and the other
SPANS = [(1, 0), (2, 5), (1, 1), (3, 2), (63, 5), (64, 0), (65, 64), (128, 7), (129, 0), (200, 1), (0, 3), (16, 900)]


# with two heads to a group, one, four (which goes the other way), gaps between the channels, a decay per channel (values that fit the
# decays' place in LDS and a wave's tile each, just or not), other numbers of taps, which go the other way too; the last sequence has no slot
@pytest.mark.parametrize("heads, groups, p, n, gap, channel", [(8, 4, 128, 128, 0, False), (3, 3, 64, 32, 0, False), (4, 2, 48, 96, 0, False), (8, 2, 64, 64, 0, False),
                                                               (4, 2, 64, 64, 32, False), (2, 2, 64, 64, 0, True), (2, 1, 16, 160, 0, False),
                                                               (2, 2, 128, 128, 0, True), (2, 2, 80, 32, 0, True), (2, 2, 144, 96, 0, True), (2, 2, 48, 160, 0, True),
                                                               (4, 2, 32, 64, 0, True)])
@pytest.mark.parametrize("taps", [4, 2, 1, 6])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_with_the_convolution(heads, groups, p, n, gap, channel, taps, dtype):
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(heads * p + n + taps)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    total, slots = sum(t for t, _ in SPANS), len(SPANS) - 1
    k_off = heads * p + gap
    s = H.DeltaShape(heads, groups, p, n, k_off, k_off + groups * n, p, n ** -0.5, channel)
    assert s.channels % 32 == 0      # (other rows have no convolution)
    width = heads * (n if channel else 1)
    z = torch.nn.functional.pad(rand(total, s.channels), (8, 24)).to(dtype)[:, 8:8 + s.channels]      # rows that are apart
    beta, a, gate = (torch.nn.functional.pad(rand(total, c), (0, -c % 8)).to(dtype)[:, :c] for c in (heads, width, heads * p))
    bias, a_log, w, norm = rand(width).to(dtype), rand(heads).to(dtype), rand(taps, s.channels).to(dtype), rand(p).to(dtype)
    state, kept = rand(2, slots, heads, n, p) * 0.1, rand(2, slots, taps - 1, s.channels).to(dtype)
    cu = lambda v: ints([0] + torch.tensor(v).cumsum(0).tolist())
    at = ints([*range(slots)][::-1] + [-1])
    cq, ck, longest = cu([t for t, _ in SPANS]), cu([t + b for t, b in SPANS]), max(t for t, _ in SPANS)

    def run(together):
        left, inputs = state.clone(), kept.clone()
        x = z if together else H.causal_conv(z, w, None, s.conv, inputs, at, cq, ck, longest)
        out = torch.full((total, heads * p), 7.0, dtype=dtype, device=DEV)
        H.delta_prefill(s, x, beta, a, bias, a_log, left, at, cq, ck, longest, out=out, gate=gate, norm_w=norm, conv=(w, inputs) if together else None)
        return out, left, inputs

    for got, want in zip(run(True), run(False)):
        assert torch.isfinite(want).all() and torch.equal(got, want)
    with pytest.raises(H.MvHipError):
        H.delta_prefill(s, z, beta, a, bias, a_log, state, at, cq, ck, longest, gate=gate, norm_w=norm, conv=(w[:, :-8], kept))


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("taps", [1, 2, 3, 4])
def test_infinite_inputs(channel, taps):
    """Infinities and NaN among the queries' inputs, which no state carries on: they reach as many tokens as there are taps, in either form."""
    from minivllm_amd import hip_ops as H

    heads, p, n, tokens = 2, 64, 64, 200
    g = torch.Generator(device=DEV).manual_seed(taps)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    s = H.DeltaShape(heads, heads, p, n, heads * p, heads * (p + n), p, n ** -0.5, channel)
    z, beta, a = rand(tokens, s.channels), rand(tokens, 8)[:, :heads], rand(tokens, heads * n if channel else 8)[:, :heads * (n if channel else 1)]
    struck = {5: float("inf"), 28: float("nan"), 61: float("-inf"), 110: float("inf"), 199: float("nan")}      # ends of runs of 8 and 32 tokens, of a chunk
    for t, v in struck.items():
        z[t, s.q_off + 3::n] = v
    width = heads * (n if channel else 1)
    bias, a_log, w = rand(width), rand(heads), rand(taps, s.channels)
    cu, at = ints([0, tokens]), ints([0])

    def run(together):
        state, kept = torch.zeros(2, 1, heads, n, p, device=DEV), torch.zeros(2, 1, taps - 1, s.channels, device=DEV).bfloat16()
        x = z if together else H.causal_conv(z, w, None, s.conv, kept, at, cu, cu, tokens)
        out = H.delta_prefill(s, x, beta, a, bias, a_log, state, at, cu, cu, tokens, conv=(w, kept) if together else None)
        return out, state, kept

    got, want = run(True), run(False)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)
    reached = {t + i for t in struck for i in range(taps)}
    assert torch.isfinite(got[0][[t for t in range(tokens) if t not in reached]]).all() and torch.isfinite(got[1]).all()
    assert all(not torch.isfinite(got[0][t]).any() for t, v in struck.items() if v != v)
