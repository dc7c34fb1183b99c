"""Nuclei without top-k of rows that stay on their CU (csrc/sampler.hip): mass and counts in one pass where the window of 2048 values ends above zero, kept
elements by their bits where the smallest is positive; against the form that reads memory in every pass.  Same order, so the same tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# few and many kept, with a floor and without
PARAMS = [(0.8, 0.9, 0.0), (2.0, 0.9, 0.0), (0.8, 0.9, 0.02), (2.0, 0.9, 1e-4), (1.0, 0.3, 0.0), (0.5, 0.999, 0.0)]


def _check(logits):
    from minivllm_amd import hip_ops as H

    t, p, m = (torch.tensor(v, device=DEV) for v in zip(*(PARAMS[i % len(PARAMS)] for i in range(logits.shape[0]))))
    k = torch.full((logits.shape[0],), -1, device=DEV)
    for offset in range(3):
        got = H.sample(logits, t, k, p, m, seed=11, offset=offset)
        want, _ = H.sample(logits, t, k, p, m, seed=11, offset=offset, return_mask=True)
        assert torch.equal(got, want), (got != want).nonzero().flatten().tolist()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vocab", [520, 50272, 18992 * 8])
@pytest.mark.parametrize("std, shift", [(2.5, 0.0), (6.0, 0.0), (1.0, 20.0), (1.0, -20.0)])
def test_nuclei(vocab, dtype, std, shift):
    g = torch.Generator(device=DEV).manual_seed(vocab)
    _check((torch.empty(2 * len(PARAMS), vocab, device=DEV).normal_(0, std, generator=g) + shift).to(dtype).contiguous())


# the largest value's bits: the window ends below, at and above zero
@pytest.mark.parametrize("top", [2046, 2047, 2048, 2049])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_windows_that_end_at_zero(dtype, top):
    g = torch.Generator().manual_seed(top)
    bits = torch.randint(0, top + 1, (2 * len(PARAMS), 4096), generator=g)
    bits[:, 17] = top
    bits[:, ::5] |= 0x8000                                   # negative ones (and -0) among them
    bits = torch.where(bits >= 0x8000, bits - 0x10000, bits)
    _check(bits.to(torch.int16).view(dtype).to(DEV))
