"""The gated delta rule's walk over chunks (csrc/delta_scalar.hip): eight waves to a workgroup for many heads and sequences, four for few."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


# tokens of a sequence around a chunk of 64 and two of them; tokens before it
SPANS = [(1, 0), (63, 5), (64, 0), (65, 64), (129, 0), (200, 1), (16, 900)]


# columns: workgroups of eight full, ragged, with one wave, only of four; key channels of every kernel (the largest has no workgroups of eight)
@pytest.mark.parametrize("heads, groups, p, n", [(8, 4, 128, 128), (6, 6, 208, 32), (12, 3, 80, 64), (16, 2, 144, 96), (9, 9, 64, 128), (4, 2, 256, 160), (5, 1, 16, 32)])
@pytest.mark.parametrize("skew", [0, 1])
def test_many_sequences_are_as_each_alone(H, heads, groups, p, n, skew):
    g = torch.Generator(device=DEV).manual_seed(heads * p + n)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    spans = SPANS * (1 + 256 // (heads * len(SPANS) * -(-p // 128)))
    total, slots = sum(t for t, _ in spans), len(spans) - 1
    s = H.DeltaShape(heads, groups, p, n, heads * p, heads * p + groups * n, p, n ** -0.5, False)
    x, beta, a = (rand(total, c).bfloat16() for c in (s.channels, heads, heads))
    if beta.shape[1] % 8:
        beta, a = (torch.nn.functional.pad(t, (0, 8 - heads % 8))[:, :heads] for t in (beta, a))
    bias, a_log = (rand(heads).bfloat16() for _ in range(2))
    state = rand(2, slots, heads, n, p) * 0.1

    def run(first, last, rows, flags=0):
        left = state.clone()
        cu = lambda v: ints([0] + torch.tensor(v).cumsum(0).tolist())
        part = spans[first:last]
        out = torch.full((rows.stop - rows.start, heads * p + 8 + skew), 7.0, dtype=torch.bfloat16, device=DEV)   # skewed: rows at odd places
        at = [i if i < slots else -1 for i in range(first, last)]
        H.delta_prefill(s, x[rows], beta[rows], a[rows], bias, a_log, left, ints(at), cu([t for t, _ in part]), cu([t + b for t, b in part]),
                        max(t for t, _ in part), out=out[:, skew:skew + heads * p], flags=flags)
        assert (out[:, skew + heads * p:] == 7).all() and (out[:, :skew] == 7).all()
        return out[:, skew:skew + heads * p], left

    out, left = run(0, len(spans), slice(0, total))
    begin = 0
    for i, (t, before) in enumerate(spans):
        if i < len(SPANS) or i >= slots - 1:
            alone, state_alone = run(i, i + 1, slice(begin, begin + t))
            assert torch.equal(out[begin:begin + t], alone), f"sequence {i}: {t} tokens behind {before}"
            if i < slots:
                half = (before + t) & 1
                assert torch.equal(left[half, i], state_alone[half, i])
                assert torch.equal(left[1 - half, i], state[1 - half, i])
        begin += t
    # token by token: the operands are the same 16-bit rows, the sums run in another order; outputs of size sqrt(n) at most, rounded to 8 bits
    scan, _ = run(0, len(spans), slice(0, total), flags=H.MV_DELTA_SCAN)
    assert (out.double() - scan.double()).abs().max() <= 2**-6 * max(1.0, scan.double().abs().max().item())


# one decay per channel (csrc/delta_chunk.hip): two column tiles a wave for many heads and sequences, one for few; groups of operands refilled a chunk ahead
@pytest.mark.parametrize("heads, p, n", [(8, 128, 128), (6, 208, 32), (12, 80, 64), (16, 144, 96), (9, 64, 128), (4, 256, 160), (5, 16, 32)])
@pytest.mark.parametrize("dtype, skew", [(torch.bfloat16, 0), (torch.bfloat16, 1), (torch.float16, 0)])
def test_many_sequences_with_channel_decay_are_as_each_alone(H, heads, p, n, dtype, skew):
    g = torch.Generator(device=DEV).manual_seed(heads * p + n)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    spans = SPANS * (1 + 256 // (heads * len(SPANS) * -(-p // 128)))
    total, slots = sum(t for t, _ in spans), len(spans) - 1
    s = H.DeltaShape(heads, heads, p, n, heads * p, heads * (p + n), p, n ** -0.5, True)
    x, beta, a = (rand(total, c).to(dtype) for c in (s.channels, heads + -heads % 8, heads * n))
    beta, bias, a_log = beta[:, :heads], rand(heads * n).to(dtype), rand(heads).to(dtype)
    state = rand(2, slots, heads, n, p) * 0.1

    def run(first, last, rows, flags=0):
        left, part = state.clone(), spans[first:last]
        cu = lambda v: ints([0] + torch.tensor(v).cumsum(0).tolist())
        out = torch.full((rows.stop - rows.start, heads * p + 8 + skew), 7.0, dtype=dtype, device=DEV)
        at = [i if i < slots else -1 for i in range(first, last)]
        H.delta_prefill(s, x[rows], beta[rows], a[rows], bias, a_log, left, ints(at), cu([t for t, _ in part]), cu([t + b for t, b in part]),
                        max(t for t, _ in part), out=out[:, skew:skew + heads * p], flags=flags)
        assert (out[:, skew + heads * p:] == 7).all() and (out[:, :skew] == 7).all()
        return out[:, skew:skew + heads * p], left

    out, left = run(0, len(spans), slice(0, total))
    begin = 0
    for i, (t, before) in enumerate(spans):
        if i < len(SPANS) or i >= slots - 1:
            alone, state_alone = run(i, i + 1, slice(begin, begin + t))
            assert torch.equal(out[begin:begin + t], alone), f"sequence {i}: {t} tokens behind {before}"
            if i < slots:
                assert torch.equal(left[(before + t) & 1, i], state_alone[(before + t) & 1, i])
        begin += t
    scan, _ = run(0, len(spans), slice(0, total), flags=H.MV_DELTA_SCAN)   # (bounds as above)
    assert (out.double() - scan.double()).abs().max() <= 2**-6 * max(1.0, scan.double().abs().max().item())


@pytest.mark.parametrize("n", [32, 64, 96, 128, 160])
def test_heads_that_share_keys_are_as_those_with_their_own(H, n):
    """Prepared two at a time, or one: the same bits."""
    g = torch.Generator(device=DEV).manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    heads, groups, p, lens = 8, 2, 48, [130, 64, 1, 63]
    total, cu = sum(lens), torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    v, k, q = rand(total, heads * p), rand(total, groups, n), rand(total, groups, n)
    beta, a, bias, a_log = rand(total, heads), rand(total, heads), rand(heads), rand(heads)
    state = torch.randn(2, len(lens), heads, n, p, generator=g, device=DEV)
    results = []
    for times in (1, heads // groups):
        many = groups * times
        s = H.DeltaShape(heads, many, p, n, heads * p, heads * p + many * n, p, n ** -0.5, False)
        x = torch.cat([v, *(t.repeat_interleave(times, 1).flatten(1) for t in (k, q))], 1)
        left = state.clone()
        results.append((H.delta_prefill(s, x, beta, a, bias, a_log, left, torch.arange(len(lens), dtype=torch.int32, device=DEV), cu, cu, max(lens)), left))
    assert all(torch.equal(*pair) for pair in zip(*results))
