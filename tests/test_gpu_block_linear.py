"""Projections of a low rank over the same rows (csrc/block_linear.hip), against their products in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows", [1, 127, 128, 129, 700])
@pytest.mark.parametrize("rank, outputs", [(128, [256, 256]), (64, [192, 96]), (128, [8, 136, 1000]), (64, [128])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_blocks(rows, rank, outputs, dtype):
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(rows + rank)
    k, n = rank * len(outputs), sum(outputs)
    x = torch.randn(rows, k + 24, generator=g, device=DEV).to(dtype)[:, 8:8 + k]
    w = torch.full((n, k), float("nan"), dtype=dtype, device=DEV)       # what lies beside the blocks is not read
    blocks, want, to = [], [], 0
    for i, m in enumerate(outputs):
        w[to:to + m, i * rank:(i + 1) * rank] = (torch.randn(m, rank, generator=g, device=DEV) * rank ** -0.5).to(dtype)
        want.append(x[:, i * rank:(i + 1) * rank].float() @ w[to:to + m, i * rank:(i + 1) * rank].float().T)
        blocks.append((i * rank, rank, to, m))
        to += m
    got, want = H.block_linear(x, w, blocks), torch.cat(want, 1)
    # sums of up to 128 products in fp32, in another order (2^-24 sqrt(128) of sums of size 1), rounded once: a unit where they straddle an edge
    assert got.shape == (rows, n) and got.dtype == dtype
    assert ((got.float() - want).abs() <= want.abs() * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11) + 1e-5).all()


def test_the_layer_takes_either_path():
    """Rows of a decode step by the whole weight, more of them by the blocks: the same numbers; shapes that the kernel does not take too."""
    from minivllm_amd import hip_ops as H
    from minivllm_amd.layers.linear import MID_M_MAX, BlockLinear, Segment

    g = torch.Generator(device=DEV).manual_seed(3)
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            layers = [BlockLinear([(a, Segment("a2", 3, 40, 64)), (b, Segment("g2", 3, 20, 32))]) for a, b in ((128, 128), (24, 40), (128, 64))]
    finally:
        torch.set_default_dtype(before)
    for lin in layers:
        lin.requires_grad_(False)
        for name, (inputs, _, s) in lin.blocks.items():
            lin.weight_loader(lin.weight, torch.randn(s.units * s.unit, inputs, generator=g, device=DEV).bfloat16() * 0.1, name)
        many = 2 ** 20 // lin.weight.shape[0] + 1       # (two blocks of 128 inputs go by blocks from so many rows on)
        x = torch.randn(many, lin.input_size, generator=g, device=DEV).bfloat16()
        want = x.float() @ lin.weight.float().T
        assert lin._by_blocks(many)
        for rows in (MID_M_MAX, MID_M_MAX + 1, MID_M_MAX + 40, many):
            torch.testing.assert_close(lin(x[:rows]).float(), want[:rows], rtol=2 ** -8, atol=1e-5)
        assert (H.block_linear(x, lin.weight, lin._places) is None) == (lin.input_size == 192)
