"""Decode over scattered rows (pages of 1, 2 or 8 tokens, slot lists; 24: per-lane lookups): a ring of index entries,
four 16-token tiles to a load, runs ahead of the ring of tiles.  Walk lengths lie around its periods (tiles, the ring's
three or four buffers, groups of four tiles, two groups in flight), where the first, the last and the partly
filled ones go wrong first."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, WorkerGroup
from tests.util import make_op_and_pool, run_decode_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (16, 4, 64)), (torch.bfloat16, (8, 2, 128)),
                                         (torch.bfloat16, (16, 4, 256)), (torch.float16, (16, 4, 256))])
@pytest.mark.parametrize("page", [1, 2, 8, 24])
def test_walks_around_the_index_ring_periods(page, dtype, heads):
    lengths = (1, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65, 79, 81, 112, 127, 128, 129, 144, 191, 193, 255, 257, 1000)
    print(f"page {page} heads {heads}", flush=True)
    total = sum(-(-k // page) for k in lengths)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total + 2 * len(lengths), 1e6, seed=page,
                                                   scale=0.5, kernel="mfma", max_pos=4096)
    order = torch.randperm(total + 2 * len(lengths), generator=gen).to(torch.int32) * page
    blocks, at = [], 0
    for k in lengths:
        b = CacheBlock(DEV, page)
        b.grow_pages(order[at: at + -(-k // page)], k)
        at += -(-k // page)
        blocks.append(b)
    # every worker reads two blocks of its own and one that three share; every fifth writes outside its view
    views = [[blocks[i], blocks[(7 * i + 3) % len(blocks)], blocks[-1 - i % 3]] for i in range(0, len(blocks), 2)]
    targets = []
    for i, v in enumerate(views):
        outside = CacheBlock(DEV, page)
        targets.append(outside if i % 5 == 0 else v[0])
    spare = iter(order[at:].split(1))
    allocator = SimpleNamespace(alloc_pages=lambda n: torch.cat([next(spare) for _ in range(n)]))
    group = WorkerGroup(cache_structure=views, write_to=targets)
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, allocator, 1e6, gen)
    assert meta.launch.counts.n_wide_items == 0 < meta.launch.counts.n_items  # the streaming kernel's
