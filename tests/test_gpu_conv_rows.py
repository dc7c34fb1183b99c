"""The causal convolution's two forms, by 8 tokens a workgroup (few of them) and by 32: the same bits, the kept inputs among them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SPANS = [(1, 0), (2, 5), (7, 1), (8, 2), (9, 3), (31, 0), (32, 7), (33, 1), (0, 3), (320, 0)]      # (tokens, tokens before)


@pytest.mark.parametrize("taps", [1, 2, 4, 8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_of_a_workgroup(taps, dtype):
    from minivllm_amd import hip_ops as H

    times, channels = 18, 96      # all at once: 180 sequences x 10 workgroups of 32 tokens
    shape = (2, 1, 16, 32, 32, 64)
    g = torch.Generator(device=DEV).manual_seed(taps)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    total, n = sum(t for t, _ in SPANS), len(SPANS)
    x, w, b, kept = rand(times * total, channels), rand(taps, channels), rand(channels), rand(2, times * n, taps - 1, channels)
    cu = lambda v: ints([0] + torch.tensor(v).cumsum(0).tolist())
    tokens, ends = [t for t, _ in SPANS], [t + c for t, c in SPANS]

    all_kept = kept.clone()
    out = H.causal_conv(x, w, b, shape, all_kept, ints(range(times * n)), cu(tokens * times), cu(ends * times), max(tokens))
    assert torch.isfinite(out).all()
    for i in range(times):
        part = kept.clone()
        got = H.causal_conv(x[i * total:(i + 1) * total], w, b, shape, part, ints(range(i * n, (i + 1) * n)), cu(tokens), cu(ends), max(tokens))
        assert torch.equal(got, out[i * total:(i + 1) * total])
        assert torch.equal(part[:, i * n:(i + 1) * n], all_kept[:, i * n:(i + 1) * n])


@pytest.mark.parametrize("taps", range(1, 9))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_infinite_inputs_reach_their_taps(taps, dtype):
    """An infinity or NaN reaches the tokens that have a tap for it and no other, wherever a workgroup's tokens begin, in either form."""
    from minivllm_amd import hip_ops as H

    tokens, channels, struck = 99, 96, {0: float("inf"), 6: float("nan"), 31: float("-inf"), 61: float("nan"), 98: float("inf")}
    g = torch.Generator(device=DEV).manual_seed(taps)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    x, w = (torch.randn(n, channels, generator=g, device=DEV).to(dtype) for n in (tokens, taps))
    for t, v in struck.items():
        x[t] = v
    for times in (1, 450):      # 4 workgroups of 32 tokens, 1800
        cu = ints(range(0, tokens * times + 1, tokens))
        kept = torch.zeros(2, times, taps - 1, channels, dtype=dtype, device=DEV)
        out = H.causal_conv(x.repeat(times, 1), w, None, (2, 1, 16, 32, 32, 64), kept, ints(range(times)), cu, cu, tokens).view(times, tokens, channels)
        reached = torch.zeros(tokens, dtype=torch.bool, device=DEV)
        for t in struck:
            reached[t:t + taps] = True
        assert torch.isfinite(out[:, ~reached]).all()
        assert all(not torch.isfinite(out[:, t]).any(0).all() for t in struck)
