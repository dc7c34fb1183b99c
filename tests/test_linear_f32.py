"""Who goes by parts of bf16 in fp32 (csrc/linear_f32.hip), and what its entry points refuse before they launch anything."""
import pytest
import torch

from minivllm_amd import hip_ops as H


def test_split_refuses():
    """The library is handed addresses: whatever they would be read wrongly from is refused on the host."""
    m, norm = torch.zeros(16, 64), torch.nn.LayerNorm(64)
    for bad in (m.bfloat16(), m.double(), m[:, ::2], m.T, m[0], m[None]):
        with pytest.raises(H.MvHipError, match="side by side"):
            H.split_f32(m, bad)
    for n in (0, H.MV_SPLIT_F32_MAX + 1):
        with pytest.raises(H.MvHipError, match="matrices"):
            H.split_f32(*[m] * n)
    for bad in (torch.nn.LayerNorm(32), torch.nn.LayerNorm(64).bfloat16(), torch.nn.LayerNorm((64, 64)), torch.nn.LayerNorm(64, elementwise_affine=False)):
        with pytest.raises(H.MvHipError, match="norm: 64"):
            H.split_f32(m, norm=bad)
    norm.bias = torch.nn.Parameter(torch.zeros(63))
    with pytest.raises(H.MvHipError, match="norm: 64"):
        H.split_f32(m, norm=norm)
    for call in (lambda: H.split_f32(m), lambda: H.split_f32(m, norm=torch.nn.LayerNorm(64))):
        with pytest.raises(H.MvHipError, match="device tensors"):
            call()


def test_linear_refuses():
    part = lambda rows, k, n=None: H.F32Parts(torch.zeros(n or -(-rows // 16) * k * 96, dtype=torch.uint8), rows, k)
    x, w = part(20, 64), part(48, 64)
    for a, b in ((part(20, 32), w), (part(20, 64, 100), w), (x, part(48, 64, 100)), (x._replace(data=x.data.view(torch.int16)), w), (x, w._replace(rows=49))):
        with pytest.raises(H.MvHipError, match="inputs of|parts of a matrix"):
            H.linear_f32(a, b)
    with pytest.raises(H.MvHipError, match="bias"):
        H.linear_f32(x, w, torch.zeros(47))
    with pytest.raises(H.MvHipError, match="residual"):
        H.linear_f32(x, w, residual=torch.zeros(20, 96)[:, ::2])
    with pytest.raises(H.MvHipError, match="device tensors"):
        H.linear_f32(x, w)


@pytest.mark.gpu
def test_linear_refuses_vectors_elsewhere():
    x, w = H.split_f32(torch.zeros(20, 64, device="cuda:0"), torch.zeros(48, 64, device="cuda:0"))
    for kw in (dict(bias=torch.zeros(48)), dict(residual=torch.zeros(20, 48))):
        with pytest.raises(H.MvHipError, match="device tensors"):
            H.linear_f32(x, w, **kw)
