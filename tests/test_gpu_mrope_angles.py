"""Cosine and sine of an mRoPE rotation in fp32, read off the rotation of (1, 0) pairs, against long double: small angles,
the longest real positions, and positions past 2^50, where a quotient by pi / 2 no longer fits a double to the unit."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from async_llm_amd.shared_cache import SharedCacheAttention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("log2_pos", [4, 14, 20, 31, 50, 51, 53, 57, 62])
def test_angles_of_any_position(log2_pos):
    rotary, n = 128, 4096
    op = SharedCacheAttention(SimpleNamespace(), torch.zeros(1, rotary, device=DEV), 8, 2, rotary, 16, torch.float32, DEV,
                              rotary_dim=rotary, mrope_section=(24, 20, 20), rope_base=1e7)
    gen = torch.Generator().manual_seed(log2_pos)
    position = (2.0 ** (log2_pos + torch.rand(n, generator=gen, dtype=torch.float64))).to(torch.int64)
    position[::2] *= -1
    x = torch.zeros(n, 1, rotary, device=DEV)
    x[..., :rotary // 2] = 1
    y = op._rope(x, position.expand(3, -1).contiguous().to(DEV))[:, 0].cpu().numpy().astype(np.longdouble)
    angle = (position.float()[:, None] * op._mrope_inv_freq.cpu()).double().numpy().astype(np.longdouble)
    for got, exact in ((y[:, :rotary // 2], np.cos(angle)), (y[:, rotary // 2:], np.sin(angle))):
        # half an ulp each for the remainder, its square or its product with the angle, the polynomial and the result
        ulp = np.spacing(np.abs(exact.astype(np.float32))).astype(np.longdouble)
        assert float((np.abs(got - exact) / ulp).max()) <= 2.0
