"""Contexts read in several parts: every number of parts at which the merge takes another number of rows a thread (csrc/paged_decode_body.h)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("parts", [2, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65])
def test_parts_meet(parts, dtype, d):
    from minivllm_amd import hip_ops as H

    heads, kv, page = 8, 8, 32                     # one sequence, pages of 32 keys: as many parts as pages, up to 64
    gen = torch.Generator(device=DEV).manual_seed(parts * d)
    lens = [parts * page, parts * page - 5, 1]
    for n in lens:
        q = torch.empty(1, heads, d, device=DEV).normal_(generator=gen).to(dtype)
        k, v = (torch.empty(parts, page, kv, d, device=DEV).normal_(generator=gen).to(dtype) for _ in range(2))
        table = torch.randperm(parts, generator=torch.Generator().manual_seed(n)).int().to(DEV)[None].contiguous()
        got = H.paged_decode(q, k, v, table, torch.tensor([n], dtype=torch.int32, device=DEV), d ** -0.5)
        ks, vs = (t[table[0].long()].flatten(0, 1)[:n].double() for t in (k, v))
        p = (torch.einsum("hd,nhd->hn", q[0].double(), ks) * d ** -0.5).softmax(-1)
        want = torch.einsum("hn,nhd->hd", p, vs)
        # one rounding of the result to the dtype (half a unit of 8 or 24 bits); sums in fp32 over at most 2080 keys behind it
        tol = dict(rtol=2 ** -8, atol=2e-4) if dtype == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(got[0].double(), want, **tol)
