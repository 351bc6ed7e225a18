"""Decode over scattered rows (pages of 1, 2 or 8 tokens, slot lists; 24: per-lane lookups): in each of a workgroup's four
waves a ring of index entries, a load for each 16-token tile, runs ahead of the ring of tiles.  Walk lengths lie around their
periods (tiles of a wave, 64 tokens apart; rings of one to four tiles; index entries of eight, 512 tokens), where the first,
the last and the partly filled ones go wrong first, in the ordinary kernel and in the one for short items."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, WorkerGroup
from tests.util import make_op_and_pool, narrow_items, run_decode_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads", [(torch.bfloat16, (16, 4, 64)), (torch.bfloat16, (8, 2, 128)),
                                         (torch.bfloat16, (16, 4, 256)), (torch.float16, (16, 4, 256))])
@pytest.mark.parametrize("page", [1, 2, 8, 24])
@pytest.mark.parametrize("short", [False, True])
def test_walks_around_the_index_ring_periods(short, page, dtype, heads):
    lengths = (1, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65, 79, 81, 112, 127, 128, 129, 144, 191, 193, 255, 257, 319, 321, 511,
               512, 513, 577, 641, 767, 769, 897, 1000)
    print(f"page {page} heads {heads} short {short}", flush=True)
    # many of a token or two, for more workgroups than start at once, and a run that is cut in items of 1050 tokens: not short
    others = [1 + i % 2 for i in range(560 // heads[1])] + ([] if short else [2100])
    total = sum(-(-(k + 1) // page) for k in lengths) + sum(-(-(k + 1) // page) for k in others)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total + 2 * len(lengths), 1e6, seed=page,
                                                   scale=0.5, kernel="mfma", max_pos=4096)
    op.plan_params.kv_chunk = 1024 if short else 2048  # (items keep their runs' lengths)
    order = torch.randperm(total + 2 * len(lengths), generator=gen).to(torch.int32) * page
    blocks, at = [], 0
    for k in (*lengths, *others):
        b = CacheBlock(DEV, page)
        b.grow_pages(order[at: at + -(-k // page)], k)
        at += -(-k // page)
        blocks.append(b)
    # every worker reads two blocks of its own and one that three share; every fifth writes outside its view
    views = [[blocks[i], blocks[(7 * i + 3) % len(lengths)], blocks[len(lengths) - 1 - i % 3]] for i in range(0, len(lengths), 2)]
    targets = []
    for i, v in enumerate(views):
        outside = CacheBlock(DEV, page)
        targets.append(outside if i % 5 == 0 else v[0])
    views += [[b] for b in blocks[len(lengths):]]
    targets += blocks[len(lengths):]
    spare = iter(order[at:].split(1))
    allocator = SimpleNamespace(alloc_pages=lambda n: torch.cat([next(spare) for _ in range(n)]))
    group = WorkerGroup(cache_structure=views, write_to=targets)
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, allocator, 1e6, gen)
    assert meta.launch.counts.n_wide_items == 0 < meta.launch.counts.n_items  # the streaming kernel's
    assert meta.launch.header[3] % 64 == short
    walked = {int(it[4]) for it in narrow_items(meta) if it[1] == 1}
    assert all(k in walked or k + 1 in walked for k in lengths if k > 64)  # (one more where a worker writes)
    assert short or max(walked) > 1024
