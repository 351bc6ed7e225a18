"""Query rotation of the wide prefill kernel, which takes another path per rotary width: widths whose half
spans whole operands (16 dims) of a head dim's half, quarter or eighth are rotated in registers, others piece
by piece; under mRoPE the rows' cosines and sines are shared through LDS.  Row counts leave a tile, a wave
and a 32-row block partly filled; positions reach far along the mRoPE axes."""

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, PrefillSpec
from tests.util import make_op_and_pool, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def widths(d):
    return [w for w in (0, 16, 32, 48, 64, 96, 128, 192, 256) if w <= d]


@pytest.mark.parametrize("mrope", [False, True])
@pytest.mark.parametrize("dtype,heads", [
    (torch.bfloat16, (4, 4, 64)), (torch.float16, (16, 2, 64)), (torch.bfloat16, (16, 1, 128)),
    (torch.float16, (8, 2, 128)), (torch.bfloat16, (8, 2, 128)), (torch.float16, (4, 4, 256)),
    (torch.bfloat16, (16, 4, 256)), (torch.float16, (16, 1, 256)),
])
def test_wide_tiles_rotate_every_width(dtype, heads, mrope):
    d, page = heads[2], 16
    for rotary in widths(d):
        if mrope and rotary == 0:
            continue
        print(f"rotary {rotary} heads {heads} mrope {mrope} {dtype}", flush=True)
        section = (rotary // 2 - 2 * (rotary // 6), rotary // 6, rotary // 6) if mrope else None
        op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, 40, 1e6, rotary_dim=rotary, mrope_section=section,
                                                       seed=rotary, scale=0.5, kernel="mfma", max_pos=1024)
        context = []
        for first, length in ((0, 75), (5, 32)):
            b = CacheBlock(DEV, page)
            b.grow_pages(torch.arange(first, first + -(-length // page)) * page, length)
            if mrope:
                b.mrope_span_override = 60000 if length == 75 else 9
            context.append(b)
        specs = []
        for w, (new, prefix) in enumerate(((133, 40), (65, 0), (18, 7))):
            pages = torch.arange(8 + 11 * w, 8 + 11 * w + -(-(new + prefix) // page), dtype=torch.int32) * page
            p = torch.arange(new)
            rel = torch.stack([p // 9, p // 3, p % 5]) if mrope and w != 1 else None
            specs.append(PrefillSpec(context[:2 - w % 2], pages, new, prefix, 50000 + prefix if mrope else prefix, rel))
        *_, meta = run_prefill_parity(op, cpu_pool, dev_pool, specs, 1e6, gen, scale=0.5)
        assert meta.launch.counts.n_wide_items > 0
