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
