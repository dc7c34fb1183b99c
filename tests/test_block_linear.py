"""Projections of a low rank over the same rows (layers/linear.py: BlockLinear): by their blocks, or over the whole weight."""
import pytest


@pytest.mark.parametrize("inputs, outputs, rows, blocks", [
    ((128, 128), 1024, 512, False), ((128, 128), 1024, 513, True), ((128, 128), 256, 2047, False), ((128, 128), 256, 2048, True), ((128, 128), 4096, 15000, True), ((128, 128), 4096, 16000, False),
    ((64, 64), 128, 513, True), ((64, 64), 4096, 16000, True), ((128,), 1024, 9939, False), ((64,), 1024, 9939, True), ((128, 128, 128), 1024, 513, True)])
def test_which_way(inputs, outputs, rows, blocks):
    import torch

    from minivllm_amd.layers.linear import BlockLinear, Segment

    with torch.device("meta"):
        layer = BlockLinear([(n, Segment(f"s{i}", outputs // 64, 64, 64)) for i, n in enumerate(inputs)])
    assert layer._by_blocks(rows) == blocks
