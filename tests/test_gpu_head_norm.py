"""Norm and gate of heads (csrc/delta.hip): one item a thread, or four one behind the other where there are many; the bits of the sums and of the root."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lanes(p, dtype):
    vectors = p // (4 if dtype == torch.float32 else 8)
    return max(4, 1 << (vectors - 1).bit_length())


# heads: one, a number that does not divide the items of a pass, as many as those, more; whole and padded channels
@pytest.mark.parametrize("heads", [1, 3, 16, 70])
@pytest.mark.parametrize("p, p_true", [(16, 16), (64, 60), (128, 128), (200, 199), (512, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_four_items_a_thread_are_one_at_a_time(heads, p, p_true, dtype):
    from minivllm_amd import hip_ops as H

    if dtype == torch.float32:
        p, p_true = min(p, 256), min(p_true, 256)       # (up to 64 vectors a head)
    lanes = _lanes(p, dtype)
    need = 4096 * 256 // lanes                          # items from which a thread has four
    rows, skew = -(-need // heads) + 1, 8               # (and a last workgroup that is not full)
    gen = torch.Generator(device=DEV).manual_seed(heads * p)
    rand = lambda *s: torch.empty(s, device=DEV).normal_(generator=gen).to(dtype)
    y, z, w = rand(rows, heads * p + skew)[:, skew:], rand(rows, heads * p + 2 * skew)[:, skew:-skew], rand(p)
    out = torch.full((rows, heads * p + skew), 7.0, dtype=dtype, device=DEV)
    call = lambda a, b, to: H.head_norm_gate(a, b, w, heads, p, p_true, 1e-6, "silu", 0.5, out=to)
    call(y, z, out[:, skew:])
    assert (out[:, :skew] == 7).all()
    part = rows // 3 + 1
    assert rows * heads >= need > part * heads
    for r in range(0, rows, part):
        assert torch.equal(call(y[r:r + part], z[r:r + part], torch.empty_like(out[r:r + part])[:, skew:]), out[r:r + part, skew:])
    f, g = y[-part:].double().unflatten(1, (heads, p)), z[-part:].double().unflatten(1, (heads, p))
    f = torch.where(torch.arange(p, device=DEV) < p_true, f, 0.0)
    want = 0.5 * f * (f.square().sum(-1, keepdim=True) / p_true + 1e-6).rsqrt() * w.double() * torch.nn.functional.silu(g)
    # fp32 throughout (sums of up to 512 squares, a handful of roundings of 2^-24 each), rounded once to 8, 11 or 24 bits
    unit = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 2 ** -24}[dtype]
    got = out[-part:, skew:].double().unflatten(1, (heads, p))
    assert ((got - want).abs() <= (unit * 1.0001 + 2 ** -20) * want.abs() + 2 ** -25).all()
    call(y, z, y)                                       # in place
    assert torch.equal(y, out[:, skew:])


@pytest.mark.parametrize("p", [16, 64, 128, 256, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [300, 40000])
def test_bits_of_the_sum_and_of_the_root(p, dtype, rows):
    """Squares meet 1, 2, 4 .. vectors of a head apart, root and division are exact: the rounded results of just those sums."""
    from minivllm_amd import hip_ops as H

    heads, eps, lanes = 2, np.float32(1e-6), _lanes(p, dtype)
    gen = torch.Generator().manual_seed(p + rows)
    y, w = torch.randn(rows, heads * p, generator=gen).to(dtype), torch.randn(p, generator=gen).to(dtype)
    z = torch.zeros_like(y)                             # the gate: 1 / (1 + 1)
    got = H.head_norm_gate(y.to(DEV), z.to(DEV), w.to(DEV), heads, p, p, float(eps), "sigmoid", 0.7).cpu()
    f = np.zeros((rows * heads, lanes * 8), np.float32)
    f[:, :p] = y.float().numpy().reshape(rows * heads, p)
    f = f.reshape(rows * heads, lanes, 8)
    ss = np.zeros(f.shape[:2], np.float32)
    for j in range(8):
        ss = (f[:, :, j].astype(np.float64) ** 2 + ss).astype(np.float32)      # (a fused product and sum)
    off = 1
    while off < lanes:
        ss = ss + ss[:, np.arange(lanes) ^ off]
        off *= 2
    rs = np.float32(0.7) / np.sqrt(ss[:, :1] / np.float32(p) + eps)
    scaled = f.reshape(rows * heads, -1)[:, :p] * rs * w.float().numpy() * np.float32(0.5)
    assert torch.equal(got, torch.from_numpy(scaled).to(dtype).view(rows, heads * p))
