"""Results in f16 of a product are rounded once (csrc/common.h: pack8), not to fp32 first."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("cols", [1024, 4096])
def test_rms_norm_rounds_its_products_once(cols):
    from minivllm_amd import hip_ops as H

    rng = np.random.default_rng(cols)
    x = rng.integers(-20, 21, (64, cols)).astype(np.float16)            # (the sum of squares is exact)
    w = rng.normal(1.0, 0.3, cols).astype(np.float16)
    mean = (x.astype(np.float64) ** 2).sum(1, keepdims=True).astype(np.float32) / np.float32(cols)
    t = x.astype(np.float32) * (np.float32(1) / np.sqrt(mean + np.float32(1e-6)))
    product = t.astype(np.float64) * w.astype(np.float64)               # (exact: 24 + 11 bits)
    once, twice = product.astype(np.float16), product.astype(np.float32).astype(np.float16)
    assert (once != twice).any()
    got = H.rmsnorm(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), 1e-6).cpu().numpy()
    assert np.array_equal(got, once)
