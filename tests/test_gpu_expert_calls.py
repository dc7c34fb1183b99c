"""Router, grouping and both products of the experts as one call (mv_moe_mlp), against the four calls: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (up to 16 rows the router groups, a quarter of the pairs to a lane)
@pytest.mark.parametrize("rows, top, tile", [(1, 3, 16), (16, 3, 16), (16, 4, 16), (8, 8, 16), (13, 5, 16), (16, 8, 16), (5, 1, 16), (17, 3, 16), (24, 3, 32), (32, 3, 16), (33, 3, 16), (77, 3, 64),
                                             (700, 3, 256)])
@pytest.mark.parametrize("weigh", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_one_call_is_four(rows, top, tile, weigh, dtype):
    from minivllm_amd import hip_ops as H

    experts, extra, k, ff = 8, 0 if weigh else 2, 256, 128
    g = torch.Generator(device=DEV).manual_seed(rows)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    form = (lambda w: w) if dtype == torch.float32 else (lambda w: H.pack_weight(w.view(-1, w.shape[-1])))
    if dtype == torch.float32:
        tile = 16
    x = torch.nn.functional.pad(rand(rows, k), (0, 64))[:, :k]      # rows that are apart
    router, correction = rand(experts + extra, k), rand(experts + extra)
    gate_up, down = form(rand(experts, 2, ff, k) * k ** -0.5), form(rand(experts, k, ff) * ff ** -0.5)
    act, quarters = H.GateAct(0, 0.0, 0.0), tile == 64
    ids, weights = H.moe_route(x, router, correction, top, 2, 2, 1.5, weigh, weigh)
    groups = H.moe_group(ids, experts, tile, weights if weigh else None)
    z = H.moe_linear(x, gate_up, ff, groups, act, gather=True, experts=experts, in_scale=groups.weights, quarters=quarters)
    y = H.moe_linear(z, down, k, groups, experts=experts, quarters=quarters)
    got, place, got_weights = H.moe_mlp(x, router, correction, gate_up, down, experts, ff, k, top, tile, act, 2, 2, 1.5, weigh, weigh, weigh, quarters)
    assert torch.equal(place, groups.place) and torch.equal(got_weights, weights)
    used = place[place >= 0].long()
    assert torch.equal(got[used], y[used])
    with pytest.raises(H.MvHipError):
        H.moe_mlp(x, router, correction, gate_up, down[:-1], experts, ff, k, top, tile, act)
    with pytest.raises(H.MvHipError):
        H.moe_mlp(x[:, :k - 64], router, correction, gate_up, down, experts, ff, k, top, tile, act)
