"""The kernels' tile edges, remainders and dispatch rules against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from wisp import quant

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bits", [8, 4, 3, 2])
@pytest.mark.parametrize("n", [128, 17 * 128, 16 * 128])  # 3, 51 and 48 groups: part of a workgroup, a remainder, whole ones
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])  # 1: values that are not 16-byte aligned take the general kernel
def test_quantize_group_128_edges(bits, n, dtype, shift):
    rng = np.random.default_rng(bits + n)
    w = (rng.standard_normal(3 * n) * 0.05).astype(np.float32)
    w[:128] = rng.integers(0, 2 * 2**bits - 1, 128) * np.float32(0.5)  # quotients at and next to ties
    w[128:256] *= np.float32(1e-4)  # scale clamped to 1e-5, an fp16 subnormal
    w[256:384] *= np.float32(3e6)  # minimum beyond fp16: -inf, and infinite quotients
    w = O.bf16_bits_to_f32(O.f32_to_bf16_bits(w)) if dtype == torch.bfloat16 else w
    buf = torch.zeros(3 * n + shift, dtype=dtype, device=DEV)
    buf[shift:] = torch.from_numpy(w).to(DEV)
    got = quant.quantize(buf[shift:].view(3, n), bits, 128).cpu().numpy()
    assert np.array_equal(got, O.quantize(w, bits, 128))
