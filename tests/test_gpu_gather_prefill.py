"""Wide prefill over scattered rows (pages of 1, 2 or 8 tokens): a ring of index entries, four tiles to a load,
runs ahead of the ring of tiles.  Walk lengths lie around its periods (32-token tiles, groups of four, two groups
in flight), where the first, the last and the partly filled ones go wrong first."""

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, PrefillSpec
from tests.util import make_op_and_pool, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (8, 2, 64)), (torch.bfloat16, (8, 2, 128)),
                                         (torch.float16, (8, 2, 128)), (torch.bfloat16, (16, 4, 256))])
@pytest.mark.parametrize("page", [1, 2, 8])
def test_walks_around_the_index_ring_periods(page, dtype, heads):
    for n, lengths in enumerate(((1, 31), (32, 33), (64, 97), (127, 129), (160, 255), (256, 257), (289, 640))):
        print(f"page {page} heads {heads} blocks {lengths}", flush=True)
        new, prefix = ((70, 0), (33, 31), (150, 3))[n % 3]
        total = sum(-(-k // page) for k in lengths) + -(-(new + prefix) // page)
        op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total + 1, 1e6, seed=n, scale=0.5,
                                                       kernel="mfma", max_pos=2048)
        order = torch.randperm(total, generator=gen).to(torch.int32) * page
        blocks, at = [], 0
        for k in lengths:
            b = CacheBlock(DEV, page)
            b.grow_pages(order[at: at + -(-k // page)], k)
            at += -(-k // page)
            blocks.append(b)
        *_, meta = run_prefill_parity(op, cpu_pool, dev_pool, [PrefillSpec(blocks, order[at:], new, prefix)], 1e6, gen,
                                      scale=0.5)
        assert meta.launch.counts.n_wide_items > 0
