"""State space recurrence of few long sequences, cut into segments (csrc/ssm_chunk.hip), against the same kernel on whole sequences."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


# around the lengths at which a sequence gets one more segment (four chunks of 64 tokens and up), beside short ones and empty slots
@pytest.mark.parametrize("spans", [[(256, 0)], [(257, 0), (1, 0)], [(513, 7), (70, 0), (512, 3)], [(2500, 0), (33, 5)], [(1000, 2), (999, 1), (40, 0)]], ids=str)
@pytest.mark.parametrize("heads, groups, p, n", [(4, 2, 64, 128), (3, 1, 48, 32), (2, 1, 80, 160), (6, 1, 32, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_segments_are_whole_sequences(H, monkeypatch, spans, heads, groups, p, n, dtype):
    """spans: (tokens, tokens before) of the sequences; the last one has no slot."""
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
    old = rand(2, len(spans), heads, n, p)

    def run():
        state = old.clone()
        return H.ssm_prefill(x, dt, bias, a_log, d, shape, state, slots, cq, ck, longest), state

    got, state = run()
    asked = H._lib.mv_ssm_prefill_workspace_bytes(len(spans), total, longest, heads, p, n, H._dt(x))
    assert asked > 0 or longest <= 5 * 64
    monkeypatch.setattr(H._lib, "mv_ssm_prefill_workspace_bytes", lambda *a: 0)
    want, kept = run()
    # fp32 sums in another order, rounded once: a unit of the 16-bit result
    torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7 if dtype == torch.bfloat16 else 2 ** -10, atol=1e-3)
    torch.testing.assert_close(state, kept, rtol=1e-4, atol=1e-5)
    assert torch.isfinite(got).all()


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
