"""Sampling of rows that stay on their CU (csrc/sampler.hip, RowOnChip) against the form that reads memory in every pass, which a call that
asks for the mask takes.  Same order of the elements, so the same tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PARAMS = [(0.0, -1, 1.0, 0.0), (1.0, -1, 1.0, 0.0), (0.6, 40, 0.95, 0.0), (0.7, 3, 1.0, 0.0), (1.3, 2000, 1.0, 0.0), (0.8, -1, 0.9, 0.0),
          (2.0, -1, 0.999, 0.0), (0.7, -1, 1.0, 0.05), (0.9, 50, 0.8, 0.02), (1e-3, -1, 0.5, 0.0), (1.0, 1, 1.0, 0.0)]


def _both(H, logits, seed=3):
    rows, vocab = logits.shape
    t, k, p, m = (torch.tensor(v, device=DEV) for v in zip(*(PARAMS[i % len(PARAMS)] for i in range(rows))))
    for offset in range(3):
        got = H.sample(logits, t, k, p, m, seed=seed, offset=offset)
        want, mask = H.sample(logits, t, k, p, m, seed=seed, offset=offset, return_mask=True)
        assert torch.equal(got, want), (got != want).nonzero().flatten().tolist()
        assert 0 <= int(got.min()) and int(got.max()) < vocab
    return got


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


# one vector; a partial and a full vector per thread; the LDS alone, its last row of vectors, one behind; the registers' last; memory again
@pytest.mark.parametrize("vocab", [8, 512, 8192, 8200, 50272, 9 * 8192, 9 * 8192 + 8, 18992 * 8, 19 * 8192, 19 * 8192 + 8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_on_chip_draw_what_rows_in_memory_draw(H, vocab, dtype):
    g = torch.Generator(device=DEV).manual_seed(vocab)
    logits = torch.empty(2 * len(PARAMS), vocab, device=DEV).normal_(0, 2.5, generator=g)
    logits[len(PARAMS):] *= 0.05            # flat: thresholds far below the maximum
    _both(H, logits.to(dtype).contiguous())


@pytest.mark.parametrize("vocab", [4096, 100_000])
def test_unusual_rows(H, vocab):
    g = torch.Generator(device=DEV).manual_seed(7)
    n = len(PARAMS)
    base = torch.empty(n, vocab, device=DEV).normal_(0, 2.0, generator=g)
    kinds = {
        "all negative": -base.abs() - 1, "below a maximum of zero": -base.abs() * (torch.arange(vocab, device=DEV) != 77),
        "equal": torch.full_like(base, 1.5), "few values": base.round(), "all but one masked": torch.full_like(base, -float("inf")).index_fill_(
            1, torch.tensor([vocab - 1], device=DEV), 0.25), "all masked": torch.full_like(base, -float("inf")),
        "infinite": base.index_fill(1, torch.tensor([5, vocab // 2], device=DEV), float("inf")),
        "tiny": base * 1e-38, "one far ahead": base.index_fill(1, torch.tensor([vocab // 3], device=DEV), 60.0),
    }
    for name, logits in kinds.items():
        got = _both(H, logits.to(torch.bfloat16).contiguous())
        if name == "all but one masked":
            assert (got == vocab - 1).all()
        if name == "one far ahead":
            assert (got[[0, 2, 3]] == vocab // 3).all()


def test_rows_with_nan_end_and_name_a_word(H):
    logits = torch.randn(len(PARAMS), 40_000, device=DEV)
    logits[:, 17] = float("nan")
    logits[:, 123] = -float("nan")
    _both(H, logits.bfloat16())
    _both(H, torch.full_like(logits, float("nan")).bfloat16())


@pytest.mark.parametrize("vocab", [8, 4096, 32_000, 50_272, 19 * 8192, 19 * 8192 + 8, 4099])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_greedy_rows_name_the_first_of_the_largest(H, vocab, dtype):
    g = torch.Generator(device=DEV).manual_seed(vocab)
    x = torch.empty(40, vocab, device=DEV).normal_(0, 3, generator=g).round()            # many ties
    x[1], x[2, vocab // 2:] = -float("inf"), -float("inf")
    x[3], x[3, -1], x[4] = float("nan"), -float("inf"), float("nan")
    x[5, ::3], x[6, 1::2], x[7] = float("nan"), float("inf"), -x[7].abs() * 1e-30 + 0.0  # (the last: zeros of both signs, tiny values)
    x[8, :7], x[9] = -float("inf"), -x[9].abs() - 1
    x = x.to(dtype)
    t = torch.zeros(40, device=DEV)
    t[30:] = 0.7                                                                         # beside sampled rows
    got, stats = H.sample(x, t, None, None, None, return_stats=True)
    top = x.double().nan_to_num(-float("inf"), float("inf"), -float("inf")).amax(1, keepdim=True)
    is_top = x.double() == top
    want = torch.where(is_top.any(1), is_top.double().argmax(1), 0)
    assert torch.equal(got[:30], want[:30])
    assert torch.equal(stats[:30, 0].double(), top[:30, 0]) and (stats[:30, 1] == 1).all()
    assert torch.equal(got, H.sample(x, t, None, None, None, return_mask=True)[0])
