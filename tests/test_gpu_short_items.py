"""Launches of many short items, whose workgroups share a CU: item lengths around the tiles that four waves take in turn,
rings of one tile, the shared run's tiles apart; uniform pages and scattered rows."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, WorkerGroup
from tests.util import make_op_and_pool, run_decode_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
LENGTHS = [1, 15, 16, 17, 63, 64, 65, 127, 129, 191, 193, 257]


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (16, 4, 64)), (torch.float16, (8, 2, 128)),
                                         (torch.bfloat16, (16, 4, 256)), (torch.float16, (16, 2, 256)),
                                         (torch.bfloat16, (16, 16, 128))])
@pytest.mark.parametrize("page", [16, 24, 4, 1])
@pytest.mark.parametrize("shared_length", [3, 80])
def test_many_short_items(dtype, heads, page, shared_length):
    print(f"heads {heads} page {page} shared {shared_length}", flush=True)
    workers = 300 // heads[1]
    lengths = [LENGTHS[i % len(LENGTHS)] for i in range(workers)]
    total = -(-shared_length // page) + sum(-(-(n + 1) // page) for n in lengths) + workers
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total, 1e6, seed=page + shared_length,
                                                   scale=0.5, kernel="mfma", max_pos=1024)
    order = torch.randperm(total, generator=gen).to(torch.int32) * page
    at = 0

    def block(n):
        nonlocal at
        b = CacheBlock(DEV, page)
        b.grow_pages(order[at: at + -(-n // page)], n)
        at += -(-n // page)
        return b

    shared = block(shared_length)
    views = [[shared, block(n)] for n in lengths]
    spare = iter(order[at:].split(1))
    allocator = SimpleNamespace(alloc_pages=lambda n: torch.cat([next(spare) for _ in range(n)]))
    group = WorkerGroup(cache_structure=views, write_to=[v[1] for v in views])
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, allocator, 1e6, gen)
    assert meta.launch.counts.n_wide_items == 0
    assert meta.launch.header[3] & 1  # VA_CHUNK_SHORT_ITEMS beside the chunk
