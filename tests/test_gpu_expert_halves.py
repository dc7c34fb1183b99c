"""Products of very many rows per expert (csrc/moe.hip: halves of a tile of 256 rows, dealt to the XCDs), against the kernel of few rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


# rows around a half and a whole tile, experts without any, more tiles than a wave looks at at a time, fewer halves than a run of eight
@pytest.mark.parametrize("counts", [[1], [128, 0, 129], [0, 127, 256, 257, 0, 1, 385], [3] * 50 + [0] * 20 + [300] + [130] * 40, [0, 0, 900, 0]], ids=lambda c: str(sum(c)))
# two stages of 32 inputs, four, more; outputs that leave the last 256 of a workgroup ragged
@pytest.mark.parametrize("k, n", [(64, 16), (128, 272), (448, 528)])
@pytest.mark.parametrize("dtype, act, scaled", [(torch.bfloat16, None, True), (torch.float16, None, False), (torch.bfloat16, 0, True), (torch.float16, 1, False),
                                                (torch.bfloat16, 2, False), (torch.bfloat16, 3, True)])
def test_halves_are_as_few_rows(H, counts, k, n, dtype, act, scaled):
    g = torch.Generator().manual_seed(len(counts) + k)
    experts, rows = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(rows, generator=g)].int().to(DEV)[:, None]
    x = torch.randn(rows, k + 64, generator=g).to(DEV, dtype)[:, :k]
    w = (torch.randn(experts * n * (1 if act is None else 2), k, generator=g) * k ** -0.5).to(DEV, dtype)
    scale = (torch.rand(rows, generator=g) + 0.5).to(DEV)
    packed, glu = H.pack_weight(w), None if act is None else H.GateAct(act, 3.0, 1.7)
    out = []
    for tile in (16, 256):
        groups = H.moe_group(ids, experts, tile)
        out.append(H.moe_linear(x, packed, n, groups, glu, gather=True, experts=experts, in_scale=scale if scaled else None).double())
    # Sums of k products of size 1 / sqrt(k) in another order differ by less than 2^-12, which rounds to the next value; gated, both factors and their
    # product may be rounded to the next value
    eps = torch.finfo(dtype).eps
    assert ((out[0] - out[1]).abs() <= 4 * eps * out[0].abs() + 2**-11).all()
    assert torch.isfinite(out[1]).all()


@pytest.mark.parametrize("counts", [[1] * 700 + [300], [0] * 600 + [257] * 3 + [0] * 100 + [5], [130] * 515])
def test_more_tiles_than_are_held(H, counts):
    """Tiles that a workgroup looks for among more than 512: each place's result is its expert's."""
    experts, rows, k, n = len(counts), sum(counts), 64, 32
    ids = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts)).int().to(DEV)[:, None]
    x = torch.ones(rows, k, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(experts, n, k, dtype=torch.bfloat16, device=DEV)
    w[:, :, 0], w[:, :, 1] = (torch.arange(experts, device=DEV) // 16)[:, None].bfloat16(), (torch.arange(experts, device=DEV) % 16 / 16)[:, None].bfloat16()
    groups = H.moe_group(ids, experts, 256)
    got = H.moe_linear(x, H.pack_weight(w.view(-1, k)), n, groups, None, gather=True, experts=experts)
    want = (ids.float() / 16).bfloat16().expand(rows, n)      # (exact sums, rounded once)
    assert torch.equal(got[groups.place.long()], want)
