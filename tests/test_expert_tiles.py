"""Rows of the tiles that an expert launch works on (layers/moe.py): both sides of each line."""
import pytest
import torch


@pytest.mark.parametrize("experts, width, ff, pairs, rows", [
    (32, 2048, 768, 8, 16), (32, 2048, 768, 9, 32), (32, 2048, 768, 16, 32), (32, 2048, 768, 17, 64), (8, 2048, 768, 28, 32), (8, 2048, 768, 29, 64),
    (2, 4096, 1024, 40, 32), (2, 4096, 1024, 41, 64), (32, 4096, 1536, 24, 32), (32, 4096, 1536, 25, 64), (64, 2048, 768, 24, 32), (64, 1024, 384, 17, 64),
    (128, 768, 3072, 17, 64), (32, 2048, 768, 40, 64), (32, 2048, 768, 41, 256), (32, 1024, 384, 128, 64), (32, 1024, 384, 129, 256), (4, 2048, 768, 640, 64), (4, 2048, 768, 768, 256),
    (8, 768, 3072, 64, 64), (8, 768, 3072, 384, 64), (8, 768, 3072, 500, 256), (16, 1024, 2816, 128, 64), (16, 1024, 2816, 129, 256), (1, 1024, 2816, 2500, 256)])
def test_rows_of_a_tile(experts, width, ff, pairs, rows):
    from minivllm_amd.layers import ExpertMLP

    layer = ExpertMLP(64, 1, 0, 1, 1, 1, 1.0, 64).to(torch.bfloat16)
    layer.experts, layer.w, layer.f = experts, width, ff
    assert layer.tile_rows(pairs * experts) == rows
