"""The router's workgroups (csrc/moe.hip): one tile of 16 tokens over 16 or eight waves, or two tiles (long rows of inputs); choices out of registers
(up to 64 outputs in up to 8 groups) or LDS."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


def _choose(scores, corr, top, groups, keep):
    """fp64 scores [T, R] -> ids [T, top], falling choice score, the lowest id first among equals."""
    choice = scores + corr
    if keep < groups:
        best = choice.unflatten(1, (groups, -1)).amax(2)
        kept = torch.zeros_like(best).scatter(1, best.sort(dim=1, descending=True, stable=True).indices[:, :keep], 1.0)
        choice = choice.masked_fill(kept.repeat_interleave(choice.shape[1] // groups, 1) == 0, -torch.inf)
    return choice.sort(dim=1, descending=True, stable=True).indices[:, :top]


# rows around a tile, two tiles and the line between the two workgroups; steps of K that the waves share unevenly; outputs around 64, groups around 8
@pytest.mark.parametrize("rows", [1, 15, 17, 33, 4096, 4097])
@pytest.mark.parametrize("k, outputs, top, groups, keep", [(32, 1, 1, 1, 1), (544, 17, 17, 1, 1), (96, 63, 5, 3, 2), (2048, 64, 64, 8, 8), (160, 64, 3, 16, 5),
                                                           (1056, 72, 9, 8, 3), (64, 512, 6, 1, 1), (2080, 96, 8, 4, 2)])
@pytest.mark.parametrize("dtype, sigmoid", [(torch.bfloat16, True), (torch.float16, False), (torch.float32, True)])
def test_choices_at_the_edges_of_the_tiles(H, rows, k, outputs, top, groups, keep, dtype, sigmoid):
    """Logits are multiples of 1/8 below 16 in size, exact in any order; corrections of r/16 (8 bits hold them) order what would tie."""
    g = torch.Generator().manual_seed(rows + outputs)
    x = (torch.rand(rows, k, generator=g) < 16 / k).double() * torch.randint(-1, 2, (rows, k), generator=g)
    w = torch.randint(-4, 5, (outputs, k), generator=g).double() / 8
    corr = torch.arange(outputs).double().remainder(128) / 16
    ids, weights = H.moe_route(x.to(DEV, dtype), w.to(DEV, dtype), corr.to(DEV, dtype), top, groups, keep, 1.5, sigmoid=sigmoid)
    logits = x @ w.T
    scores = logits.sigmoid() if sigmoid else logits.softmax(1)
    ids, weights = ids.cpu().long(), weights.cpu().double()
    assert ids.min() >= 0 and ids.max() < outputs and (ids.sort(1).values.diff(dim=1) > 0).all()
    # choices: as good as the best ones, up to what single precision makes of a choice score (sizes below 9, an exponential of a few ulp)
    if keep == groups:
        best, got = (scores + corr).gather(1, _choose(scores, corr, top, groups, keep)), (scores + corr).gather(1, ids)
        assert (got - best).abs().max() < 9 * 2**-21
    else:
        assert (ids == _choose(scores, corr, top, groups, keep)).double().mean() > 0.99   # (groups that tie in single precision)
    want = scores.gather(1, ids)
    want = want / want.sum(1, keepdim=True) * 1.5
    # a score is off by a few ulp and its logit's share of one; the sum of ``top`` of them by half an ulp each
    assert ((weights - want).abs() <= (32 + top) * 2**-23 * want + 1e-30).all()


@pytest.mark.parametrize("rows", [24, 5000])
@pytest.mark.parametrize("outputs, groups", [(34, 2), (64, 8), (96, 8), (64, 16)])
def test_equal_and_undefined_scores(H, rows, outputs, groups):
    x, w = torch.ones(rows, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(outputs, 64, device=DEV, dtype=torch.bfloat16)
    ids, weights = H.moe_route(x, w, None, 8, groups, groups)
    assert torch.equal(ids, torch.arange(8, device=DEV, dtype=torch.int32).expand(rows, 8)) and torch.allclose(weights, torch.full_like(weights, 1 / 8))
    x[1::3] = float("nan")
    ids, _ = H.moe_route(x, w, None, 8, groups, groups)
    assert ids.min() >= 0 and ids.max() < outputs
    assert torch.equal(ids[::3], torch.arange(8, device=DEV, dtype=torch.int32).expand(len(ids[::3]), 8))


@pytest.mark.parametrize("outputs, top, groups, keep", [(1, 1, 1, 1), (16, 16, 1, 1), (34, 4, 2, 1), (49, 20, 7, 6), (64, 33, 8, 5)])
@pytest.mark.parametrize("dtype, sigmoid", [(torch.bfloat16, False), (torch.float16, True), (torch.float32, False)])
def test_four_tokens_choose_as_one(H, outputs, top, groups, keep, dtype, sigmoid):
    """Many tokens choose four at once, few one by one: with exact logits the bits are the same, NaN among them or not."""
    g = torch.Generator().manual_seed(outputs)
    x = torch.randint(-1, 2, (4099, 64), generator=g).to(DEV, dtype)
    x[5::7] = float("nan")
    w = (torch.randint(-4, 5, (outputs, 64), generator=g) / 8).to(DEV, dtype)
    corr = torch.randn(outputs, generator=g).to(DEV, dtype)
    ids, weights = H.moe_route(x, w, corr, top, groups, keep, 1.5, sigmoid=sigmoid)
    for rows in (slice(0, 37), slice(4060, 4099)):
        few, few_weights = H.moe_route(x[rows], w, corr, top, groups, keep, 1.5, sigmoid=sigmoid)
        assert torch.equal(few, ids[rows]) and torch.equal(few_weights.view(torch.int32), weights[rows].view(torch.int32))
