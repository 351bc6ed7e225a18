"""Merge of many rows (8192 (row, head) pairs and more): one workgroup per row, four floats a thread of every 1024 of
a row's [heads * dims] states, one, two or four runs of 1024 a pass.  Row widths at and past each of these, and no
multiple of 1024; rows of several states, rows of so many that they are found and merged head by head, rows an item
writes itself and (a fixed plan) rows nobody serves."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, PrefillSpec, WorkerGroup
from async_llm_amd.shared_cache.attention_graph import SharedPrefillAttentionBuffers
from tests.test_native_abi_cpu import H
from tests.util import assert_close, make_op_and_pool, oracle_prefill, prefill_inputs, run_decode_parity, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
OFF_ROW_INDPTR, MERGE_WORD = H["OFF_ROW_INDPTR"], H["MERGE_WAVES"]


def setup(dtype, heads, new, lengths, seed=3):
    page = 16
    total = sum(-(-k // page) for k in lengths) + sum(-(-n // page) for n in new)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total, 1e6, seed=seed, scale=0.5,
                                                   max_pos=4096)
    blocks, specs, at = [], [], 0
    for k in lengths:
        b = CacheBlock(DEV, page)
        b.grow_pages(torch.arange(at, at + -(-k // page)) * page, k)
        at += -(-k // page)
        blocks.append(b)
    for i, n in enumerate(new):
        pages = torch.arange(at, at + -(-n // page), dtype=torch.int32) * page
        at += -(-n // page)
        specs.append(PrefillSpec(blocks[:len(blocks) - i], pages, n))
    return op, cpu_pool, dev_pool, gen, specs


@pytest.mark.parametrize("dtype,heads,new", [
    (torch.bfloat16, (16, 4, 64), (513, 3)),     # 1024 floats a row
    (torch.float16, (16, 4, 128), (500, 40)),    # 2048
    (torch.float16, (32, 8, 128), (200, 60)),    # 4096
    (torch.bfloat16, (24, 6, 256), (345,)),      # 6144: a second, half-filled pass
])
def test_many_rows_of_several_states(dtype, heads, new):
    op, cpu_pool, dev_pool, gen, specs = setup(dtype, heads, new, (1700, 333))
    *_, meta = run_prefill_parity(op, cpu_pool, dev_pool, specs, 1e6, gen, scale=0.5)
    assert sum(new) * heads[0] >= 8192 and meta.launch.counts.n_partials > 0


@pytest.mark.parametrize("dtype,heads,workers", [
    (torch.float32, (5, 5, 64), 1650),   # 320 floats a row
    (torch.float32, (9, 3, 128), 920),   # 1152: one run and an eighth
    (torch.bfloat16, (10, 2, 64), 830),  # 640
])
def test_many_decode_rows(dtype, heads, workers):
    page = 16
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, 8 + 2 * workers, 1e6, seed=5, max_pos=512)
    shared = CacheBlock(DEV, page)
    shared.grow_pages(torch.arange(8) * page, 117)
    views = []
    for w in range(workers):
        own = CacheBlock(DEV, page)
        own.grow_pages(torch.tensor([(8 + w) * page]), 1 + w % 15)
        views.append([shared, own] if w % 3 else [own])
    group = WorkerGroup(cache_structure=views, write_to=[v[-1] for v in views])
    fresh = SimpleNamespace(alloc_pages=lambda n: torch.arange(8 + workers, 8 + workers + n, dtype=torch.int32) * page)
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, fresh, 1e6, gen)
    assert workers * heads[0] >= 8192 and meta.launch.counts.n_partials > 0


@pytest.mark.parametrize("dtype,heads,workers,blocks_of", [
    (torch.bfloat16, (16, 4, 64), 530, lambda w: 1 + w % 13),              # long rows (over eight states) all along
    (torch.float32, (32, 8, 128), 260, lambda w: 30 if w in (0, 259) else 1),  # first and last row, several rounds
    (torch.bfloat16, (64, 16, 64), 4200, lambda w: 9 if w > 4180 else 1),  # past the first 256 rows of a finder
])
def test_few_long_rows_among_many(dtype, heads, workers, blocks_of):
    page = 16
    total = sum(blocks_of(w) for w in range(workers))
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, total + workers, 1e6, seed=7, max_pos=512)
    at, views = 0, []
    for w in range(workers):
        view = []
        for i in range(blocks_of(w)):
            b = CacheBlock(DEV, page)
            b.grow_pages(torch.tensor([at * page]), 1 + (w + i) % 15)
            at += 1
            view.append(b)
        views.append(view)
    group = WorkerGroup(cache_structure=views, write_to=[v[-1] for v in views])
    fresh = SimpleNamespace(alloc_pages=lambda n: torch.arange(total, total + n, dtype=torch.int32) * page)
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, fresh, 1e6, gen)
    header = meta.launch.header
    assert header[MERGE_WORD] == 1  # the kernel under test
    indptr = meta.launch.blob[header[OFF_ROW_INDPTR]:][:workers + 1].cpu()
    assert torch.equal((indptr[1:] - indptr[:-1]) > 8, torch.tensor([blocks_of(w) > 8 for w in range(workers)]))


@pytest.mark.parametrize("out_offset,workspace_offset", [(1, 0), (0, 1), (3, 2)])
def test_buffers_aligned_to_an_element(out_offset, workspace_offset):
    heads, workers, page, dtype = (8, 2, 64), 1030, 16, torch.float32
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, 2 * workers, 1e6, seed=9, max_pos=512)
    blocks = []
    for w in range(workers):
        blocks.append(CacheBlock(DEV, page))
        blocks[-1].grow_pages(torch.tensor([w * page]), 1 + w % 15)
    views = [[blocks[0], b] if w % 2 else [b] for w, b in enumerate(blocks)]
    group = WorkerGroup(cache_structure=views, write_to=[v[-1] for v in views])
    fresh = SimpleNamespace(alloc_pages=lambda n: torch.arange(workers, workers + n, dtype=torch.int32) * page)
    *_, meta = run_decode_parity(op, cpu_pool, dev_pool, group, fresh, 1e6, gen)
    assert meta.launch.header[MERGE_WORD] == 1
    width = heads[0] * heads[2]
    q = torch.randn(workers, width, generator=gen).to(DEV)
    expected = op.attend(q, 0, meta).cpu()
    out = torch.full((workers * width + 8,), 7.0, device=DEV)
    used = meta.launch.counts.workspace_bytes
    room = torch.zeros(used + 64, dtype=torch.uint8, device=DEV)
    meta.launch.workspace = room[4 * workspace_offset:][:used]
    op.attend(q, 0, meta, out=out[out_offset:][:workers * width].view(workers, width))
    assert_close(out[out_offset:][:workers * width].view(workers, width), expected, dtype, "out")
    assert (out[:out_offset] == 7).all() and (out[out_offset + workers * width:] == 7).all()


def test_rows_nobody_serves_come_back_empty():
    heads, new = (32, 8, 128), (130, 20)
    op, cpu_pool, dev_pool, gen, specs = setup(torch.bfloat16, heads, new, (900, 333))
    buffers = SharedPrefillAttentionBuffers(op, 3, 2, 300, 400)
    meta = op.prepare_prefill_batch(specs, graph_buffers=buffers)
    positions, mrope, out_loc, q, k, v = prefill_inputs(op, specs, gen, 0.5)
    rows = torch.zeros(300, q.shape[1], dtype=q.dtype, device=DEV)
    rows[:150] = q.to(DEV)
    batch = SimpleNamespace(attn_metadata=meta, positions=positions.to(DEV), out_loc=out_loc.to(DEV), mrope_positions=None)
    op.store_new_kv(k.to(DEV), v.to(DEV), 0, batch)
    out, lse = op.attend(rows, 0, meta, return_lse=True)
    exp_out, exp_lse = oracle_prefill(op, cpu_pool, specs, 1e6, positions, mrope, out_loc, q, k, v)
    assert_close(out[:150], exp_out, op.dtype, "out")
    assert_close(lse[:150], exp_lse, op.dtype, "lse")
    assert not out[150:].any() and torch.isneginf(lse[150:]).all()
