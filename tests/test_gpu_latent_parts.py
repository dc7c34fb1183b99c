"""A step's parts of a context added up (csrc/latent_decode.hip), around the numbers of parts that its forms take, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# keys that the table has room for: 2, 4, 5, 16, 17, 63 and 64 parts; contexts that leave some of them empty
@pytest.mark.parametrize("keys", [128, 256, 320, 1024, 1088, 4032, 4096])
@pytest.mark.parametrize("kv", [64, 192, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_parts(keys, kv, dtype):
    from minivllm_amd import hip_ops as H

    heads, rot, bs = 3, 64, 64
    g = torch.Generator(device=DEV).manual_seed(keys + kv)
    pages = keys // bs
    plane = torch.randn(2 * pages, bs, kv + rot, generator=g, device=DEV).to(dtype)
    for lens in ([keys], [keys // 2 + 1], [0, 33]):
        q = (torch.randn(len(lens), heads, kv + rot, generator=g, device=DEV) * 0.6).to(dtype)
        tables = torch.randperm(2 * pages, generator=g, device=DEV).to(torch.int32)[:pages * len(lens)].view(len(lens), pages)
        got = H.latent_decode(q, plane, tables, torch.tensor(lens, dtype=torch.int32, device=DEV), kv, (kv + rot) ** -0.5, 0)
        for i, n in enumerate(lens):
            rows = plane[tables[i].long()].flatten(0, 1)[:n].double()
            want = (q[i].double() @ rows.T * (kv + rot) ** -0.5).softmax(-1) @ rows[:, :kv] if n else torch.zeros(heads, kv, device=DEV, dtype=torch.float64)
            # probabilities enter their product with the rows in 16 bits, as does the result
            eps = torch.finfo(dtype).eps
            assert ((got[i].double() - want).norm() <= 2 * eps * want.norm() + 1e-30)
