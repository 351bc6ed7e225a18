"""Decode tiles that one workgroup serves together (pairs, and fours on runs of 4096 tokens and more): numbers of readers
around whole and partly filled tiles, run lengths around the tiles four waves take in turn and the ends of their rings."""

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, WorkerGroup
from tests.util import make_op_and_pool, run_decode_parity
from types import SimpleNamespace

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (16, 4, 64)), (torch.float16, (8, 2, 128)),
                                         (torch.bfloat16, (16, 4, 256)), (torch.bfloat16, (16, 2, 128)),
                                         (torch.float16, (16, 1, 256))])
@pytest.mark.parametrize("readers", [3, 5, 9, 18])
@pytest.mark.parametrize("length", [1, 65, 129, 4095, 4097])
@pytest.mark.parametrize("page", [16, 1])
def test_tiles_that_walk_together(dtype, heads, readers, length, page):
    if page == 1 and length > 300:
        pytest.skip("scattered rows go in pairs whatever the length")
    print(f"heads {heads} readers {readers} length {length} page {page}", flush=True)
    total = -(-length // page) + 2 * readers * -(-24 // page)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total, 1e6, seed=length + readers, scale=0.5,
                                                   kernel="mfma", max_pos=8192)
    order = torch.randperm(total, generator=gen).to(torch.int32) * page
    at = 0

    def block(n):
        nonlocal at
        b = CacheBlock(DEV, page)
        b.grow_pages(order[at: at + -(-n // page)], n)
        at += -(-n // page)
        return b

    shared = block(length)
    views = [[shared, block(1 + i % 20)] for i in range(readers)]
    spare = iter(order[at:].split(1))
    allocator = SimpleNamespace(alloc_pages=lambda n: torch.cat([next(spare) for _ in range(n)]))
    group = WorkerGroup(cache_structure=views, write_to=[v[1] for v in views])
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, allocator, 1e6, gen)
    assert meta.launch.counts.n_wide_items == 0 < meta.launch.counts.n_items
    partners = _partners(meta)
    tiles = -(-readers // max(1, 16 // (heads[0] // heads[1])))
    together = 4 if length >= 4096 and page == 16 else 2
    if 16 // (heads[0] // heads[1]) > 1:
        assert max(partners) == min(together, tiles) - 1
        assert sum(1 + p for p in partners if p >= 0) == len(partners)  # every tile is served once


def _partners(meta):
    header = meta.launch.header
    words = meta.launch.blob.cpu().numpy()
    items = words[header[10]: header[10] + 16 * meta.launch.counts.n_items].reshape(-1, 16)
    return [int(it[6]) for it in items if it[2] > 0]
