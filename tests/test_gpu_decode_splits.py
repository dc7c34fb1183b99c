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


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("parts", [2, 3, 7, 13, 26, 32, 50, 64])
def test_order_of_the_merge(parts, dtype, d):
    """The parts' masses meet 32, 16, 8, 4, 2 and 1 parts apart, their rows by threads: the same bits in every build.  (The first key of each part outweighs the
    others by the same score, so that the factors are exactly 1.)"""
    from minivllm_amd import hip_ops as H

    heads, page = 8, 32
    if dtype == torch.float32 and d == 256:
        parts = min(parts, 32)                     # more workgroups a part: no more parts than that
    gen = torch.Generator(device=DEV).manual_seed(parts * d)
    q = torch.empty(1, heads, d, device=DEV).normal_(generator=gen).to(dtype)
    k, v = (torch.empty(parts, page, heads, d, device=DEV).normal_(generator=gen).to(dtype) for _ in range(2))
    k[:, 0] = q
    table = torch.arange(parts, dtype=torch.int32, device=DEV)[None]
    got = H.paged_decode(q, k, v, table, torch.tensor([parts * page], dtype=torch.int32, device=DEV), d ** -0.5)[0].cpu()
    left = H.workspace(256, DEV)[:heads * parts * (d + 2) * 4 + 256].cpu()
    at = -(-heads * parts * d * 4 // 256) * 256
    rows = left[:heads * parts * d * 4].view(torch.float32).view(heads, parts, d)
    m, mass = left[at:at + heads * parts * 8].view(torch.float32).view(heads, parts, 2).unbind(2)
    assert (m == m[:, :1]).all()
    lanes = torch.nn.functional.pad(mass, (0, 64 - parts))
    other = lanes.clone()
    for a, b in zip((32, 16, 8, 4, 2, 1), (8, 4, 2, 1, 16, 32)):
        lanes, other = (t + t[:, torch.arange(64) ^ off] for t, off in ((lanes, a), (other, b)))
    assert parts <= 16 or not torch.equal(lanes, other)      # (inputs that tell the orders apart)
    groups = 512 // d
    sums = torch.zeros(heads, groups, d)
    for i in range(parts):
        sums[:, i % groups] += rows[:, i]
    total = sums[:, 0]
    for i in range(1, groups):
        total = total + sums[:, i]
    assert torch.equal(got, (total / lanes[:, :1]).to(dtype))
