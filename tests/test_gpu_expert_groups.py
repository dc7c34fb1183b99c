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


# inputs: quarters that are empty, that end within a trip of 64 inputs, whole ones
@pytest.mark.parametrize("k", [64, 128, 192, 320, 768, 2048])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gated, weighed", [(True, False), (False, False), (True, True)])
def test_sums_by_quarters_are_those_of_small_tiles(k, dtype, gated, weighed):
    from minivllm_amd import hip_ops as H

    gen = torch.Generator(device=DEV).manual_seed(k)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    experts, tokens, top, n = 5, 97, 2, 144
    ids = torch.randint(0, experts + 1, (tokens, top), generator=gen, device=DEV, dtype=torch.int32)
    scale = torch.rand(ids.shape, generator=gen, device=DEV) if weighed else None
    x = rand(tokens, k).to(dtype)
    w = H.pack_weight((rand(experts * n * (2 if gated else 1), k) * k ** -0.5).to(dtype))
    outs = []
    for tile, quarters in ((16, False), (32, False), (64, True)):
        g = H.moe_group(ids, experts, tile, scale)
        y = H.moe_linear(x, w, n, g, H.GateAct(0, 0.0, 0.0) if gated else None, gather=True, experts=experts, in_scale=g.weights, quarters=quarters)
        outs.append(y[g.place[g.place >= 0].long()])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    with pytest.raises(H.MvHipError):
        H.moe_linear(x, w, n, H.moe_group(ids, experts, 256), H.GateAct(0, 0.0, 0.0) if gated else None, gather=True, experts=experts, quarters=True)


@pytest.mark.parametrize("tokens, top", [(129, 4), (160, 8), (231, 4), (320, 4)])
@pytest.mark.parametrize("experts", [8, 32])
def test_a_few_dozen_pairs_an_expert_sum_as_tiles_of_32(monkeypatch, tokens, top, experts):
    """Up to 40 pairs an expert, whatever the tiles that they are worked on in."""
    from minivllm_amd.layers import ExpertMLP

    tokens = tokens * experts // 32
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    with torch.device(DEV):
        layer = ExpertMLP(512, experts, 0, top, 1, 1, 1.0, 384).to(torch.bfloat16)
    for p in layer.parameters():
        p.requires_grad_(False).copy_(torch.randn(p.shape, generator=gen, device=DEV) * 0.05)
    layer.finish_weights()
    h = torch.randn(tokens, 512, generator=gen, device=DEV).bfloat16()
    assert tokens * top <= 40 * experts
    out = lambda: (lambda y, place: y[place.long()])(*layer(h)[1][:2])
    got = out()
    monkeypatch.setattr(ExpertMLP, "tile_rows", lambda self, tokens: 32)
    assert torch.equal(got, out())
