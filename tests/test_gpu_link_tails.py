"""Wide prefill whose blocks end inside a 32-token tile: a half tile of 16 tokens lies in one page, so the tail takes
one page lookup and repeats its last visible row.  Lengths lie around the edges of half tiles, tiles and pages; the
causal end of a chunk moves through them as well."""

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, PrefillSpec
from tests.util import make_op_and_pool, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.float16, (8, 2, 64)), (torch.bfloat16, (8, 2, 128)),
                                         (torch.bfloat16, (16, 4, 256))])
@pytest.mark.parametrize("page", [16, 32, 64])
def test_tails_repeat_the_last_visible_row(page, dtype, heads):
    for n, lengths in enumerate(((1, 15), (16, 17), (31, 32, 33), (47, 48, 49), (95, 97, 128), (129, 159, 161), (200, 641))):
        print(f"page {page} heads {heads} blocks {lengths}", flush=True)
        new, prefix = ((70, 0), (33, 31), (150, 3), (129, 16))[n % 4]
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
