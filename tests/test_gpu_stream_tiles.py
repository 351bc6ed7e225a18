"""Decode tiles that one workgroup serves together (pairs, and fours on runs of 4096 tokens and more, in launches that give
every CU a workgroup): numbers of readers around whole and partly filled tiles, items around the tiles four waves take in
turn (64 tokens), the ends of their rings (two tiles a wave, four at 64 dims) and of the index entries' (eight)."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, WorkerGroup
from tests.util import make_op_and_pool, narrow_items, run_decode_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (16, 4, 64)), (torch.float16, (16, 4, 128)),
                                         (torch.bfloat16, (16, 4, 256)), (torch.bfloat16, (16, 8, 128)),
                                         (torch.float16, (32, 4, 256))])
@pytest.mark.parametrize("readers", [3, 5, 9, 18])
@pytest.mark.parametrize("page,length", [(16, 1), (16, 65), (16, 129), (16, 257), (16, 700), (16, 4095), (16, 4097),
                                         (1, 1), (1, 129), (1, 513), (1, 1000), (8, 257), (8, 961)])
def test_tiles_that_walk_together(dtype, heads, readers, page, length):
    print(f"heads {heads} readers {readers} length {length} page {page}", flush=True)
    # a run of 2100 tokens, cut in two and more: the launch's items are not short; more where fours are due, which the
    # launch has to outlast (at 57 ns a token of 256 dims); many of a token or two fill the CUs
    together = 4 if length >= 4096 and page == 16 else 2
    lengths = [2100] * (112 if together == 4 else 1) + [1 + i % 2 for i in range(560 // heads[1])]
    total = -(-length // page) + readers * -(-24 // page) + sum(-(-(n + 1) // page) for n in lengths)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total, 1e6, seed=length + readers, scale=0.5,
                                                   kernel="mfma", max_pos=8192)
    op.plan_params.kv_chunk = 2048  # (items keep their runs' lengths)
    order = torch.randperm(total, generator=gen).to(torch.int32) * page
    at = 0

    def block(n):
        nonlocal at
        b = CacheBlock(DEV, page)
        b.grow_pages(order[at: at + -(-n // page)], n)
        at += -(-n // page)
        return b

    shared = block(length)
    views = [[shared, block(1 + i % 20)] for i in range(readers)] + [[block(n)] for n in lengths]
    spare = iter(order[at:].split(1))
    allocator = SimpleNamespace(alloc_pages=lambda n: torch.cat([next(spare) for _ in range(n)]))
    group = WorkerGroup(cache_structure=views, write_to=[v[-1] for v in views])
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, allocator, 1e6, gen)
    counts = meta.launch.counts
    assert counts.n_wide_items == 0 < counts.n_items and not meta.launch.header[3] & 1  # not the kernel for short items
    items = narrow_items(meta)
    partners = [int(it[6]) for it in items]
    tiles = -(-readers // (16 // (heads[0] // heads[1])))
    assert max(partners) == min(together, tiles) - 1
    assert sum(1 + p for p in partners if p >= 0) == len(partners)  # every tile is served once
    if tiles > 1:  # the longest of them walks the run, or a third of the long one
        longest = max(int(it[4]) for it in items if it[6] > 0)
        assert longest == length if length < 2048 else longest >= 1344
        rings = 4 if heads[2] == 64 else 2
        assert length < 700 or longest > 64 * rings  # its waves refill their rings
        assert length not in (513, 1000, 961) or page == 16 or longest > 64 * 8  # and come round in their index entries
