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


@pytest.mark.parametrize("k", [64, 256])
@pytest.mark.parametrize("counts", [[1] * 700 + [300], [0] * 600 + [257] * 3 + [0] * 100 + [5], [130] * 515])
def test_tiles_beyond_those_held(H, counts, k):
    """The same with the expert's number, the token's and a digit from each stage of 32 inputs in the outputs, all of them exact, tokens in any order: a
    neighbour's tile, the other half of one's own, another row or stage is another result."""
    experts, rows, n = len(counts), sum(counts), 32
    e = torch.arange(experts, device=DEV)
    g = torch.Generator().manual_seed(rows)
    ids = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(rows, generator=g)].to(DEV)
    t = torch.arange(rows, device=DEV)
    x, w = torch.zeros(rows, k, device=DEV), torch.zeros(experts, n, k, device=DEV)
    x[:, 0], w[:, 0, 0], w[:, 1, 0] = 1.0, (e // 32).float(), (e % 32).float()
    for digit in range(3):
        x[:, 1 + digit], w[:, 2 + digit, 1 + digit] = (t >> 8 * digit & 255).float(), 1.0
    w[:, 5, 1], w[:, 5, 0] = 1.0 / 256, (e % 256).float() / 256         # (the expert and the token in one sum: 9 bits, rounded once)
    for stage in range(k // 32):
        x[:, 32 * stage + 5 + stage], w[:, 8 + stage, 32 * stage + 5 + stage] = ((t * 7 + stage) % 251).float(), 1.0
    groups = H.moe_group(ids.int()[:, None].contiguous(), experts, 256)
    got = H.moe_linear(x.bfloat16(), H.pack_weight(w.bfloat16().view(-1, k)), n, groups, None, gather=True, experts=experts)[groups.place.long()]
    want = torch.zeros(rows, n, device=DEV)
    want[:, 0], want[:, 1] = (ids // 32).float(), (ids % 32).float()
    for digit in range(3):
        want[:, 2 + digit] = (t >> 8 * digit & 255).float()
    want[:, 5] = ((t & 255) + ids % 256).float() / 256
    for stage in range(k // 32):
        want[:, 8 + stage] = ((t * 7 + stage) % 251).float()
    assert torch.equal(got, want.bfloat16())
