"""Pairs of (token, choice) sorted by expert where several workgroups place an expert's pairs (csrc/moe.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# pairs: below, at and behind 2048, where a second part comes in; runs of a wave that no number of parts divides; more experts than parts have room for
@pytest.mark.parametrize("pairs, top, experts, outputs, tile_m", [(2047, 1, 3, 3, 64), (2048, 4, 32, 34, 64), (3075, 3, 32, 32, 256), (8200, 8, 32, 34, 256), (9216, 4, 1, 2, 256),
                                                                  (36004, 4, 40, 42, 256), (70000, 8, 300, 300, 64)])
@pytest.mark.parametrize("weighed", [False, True])
def test_groups_in_parts(pairs, top, experts, outputs, tile_m, weighed):
    from minivllm_amd import hip_ops as H

    gen = torch.Generator().manual_seed(pairs)
    ids = torch.randint(0, outputs, (pairs // top, top), generator=gen, dtype=torch.int32)
    weights = torch.rand(ids.shape, generator=gen) if weighed else None
    g = H.moe_group(ids.to(DEV), experts, tile_m, weights.to(DEV) if weighed else None)
    flat = ids.flatten().long()
    order = torch.sort(flat, stable=True).indices
    order = order[flat[order] < experts]                       # places in the order of the pairs
    place = torch.full_like(flat, -1)
    place[order] = torch.arange(len(order))
    assert torch.equal(g.place.cpu().long(), place)
    assert torch.equal(g.tokens.cpu().long()[:len(order)], order // top)
    if weighed:
        assert torch.equal(g.weights.cpu()[:len(order)], weights.flatten()[order])
    seen = torch.zeros(len(order), dtype=torch.int32)
    for e, first, n in g.tiles.cpu().tolist():
        if e >= 0:
            assert 0 < n <= tile_m and bool((flat[order[first:first + n]] == e).all())
            seen[first:first + n] += 1
    assert bool((seen == 1).all())
