"""Norms, rotation and cache rows of a token by one, two or four waves: the same bits, nothing but the tokens' slots written."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows of a token: fewer than a wave takes at a time, one more than a batch of them, many; tokens: by one, two and four waves
@pytest.mark.parametrize("heads, kv, dim", [(1, 1, 64), (9, 1, 128), (28, 4, 128), (8, 4, 256)])
@pytest.mark.parametrize("tokens", [513, 941, 1025, 1729])
@pytest.mark.parametrize("form", ["norm", "plain", "unit", "pairs"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_waves_of_a_token(heads, kv, dim, tokens, form, dtype):
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(tokens + heads)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    q, k, v = (t.view(tokens, -1, dim) for t in rand(tokens, (heads + 2 * kv) * dim).split([heads * dim, kv * dim, kv * dim], 1))
    pairs = 24 if form == "pairs" else None
    cos, sin = (torch.randn(tokens, pairs or dim // 2, generator=g, device=DEV) for _ in range(2))
    norms = (rand(dim), rand(dim)) if form in ("norm", "pairs") else (None, None)
    pages = tokens // 64 + 2
    slots = torch.randperm(pages * 64, generator=g, device=DEV)[:tokens].to(torch.int32)
    slots[::7] = -1      # rows that fill a batch up
    pos = torch.randint(-1, tokens + 1, (tokens,), generator=g, device=DEV)      # some outside the tables

    def run(at):
        caches = [torch.full((pages, 64, kv, dim), 7.0, dtype=dtype, device=DEV) for _ in range(2)]
        out = H.rope_qk_store(q[at], k[at], v[at], pos[at], cos, sin, *norms, 1e-6, *caches, slots[at], want_k_out=True, interleaved_pairs=pairs,
                              unit_norm=form == "unit")
        return (*out, *caches)

    got, few = run(slice(None)), [run(slice(i, min(i + 200, tokens))) for i in range(0, tokens, 200)]
    for i in range(2):
        assert torch.equal(got[i], torch.cat([t[i] for t in few]))
    for i in (2, 3):
        want = torch.full_like(got[i], 7.0)
        for t in few:
            want = torch.where(t[i] != 7.0, t[i], want)
        assert torch.equal(got[i], want)
