"""``va_attention_static`` (the entry point that allocates nothing) against ``va_attention``:
the same plan, the same kernels, the partial states in the library's own per-GPU array instead
of a caller's workspace.  Results must be identical bit for bit, on two calls in a row of which
the second is smaller (the array keeps the first call's contents), and a plan whose partial
states exceed the array must be refused with a clear error -- but for one that exceeds it by its
fine cuts only, which the call plans anew with coarse ones."""

import pytest
import torch

from async_llm_amd import native, workloads
from async_llm_amd.shared_cache import CacheBlock, PrefillSpec
from tests.util import assert_close, make_op_and_pool, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _both_ways(wl):
    op, meta = wl.op, wl.meta
    counts = meta.launch.counts
    assert counts.n_partials > 0, "the workload must split rows over work items, or no scratch is used"
    assert counts.workspace_bytes <= native.STATIC_SCRATCH_BYTES
    op.store_new_kv(wl.k, wl.v, 0, wl.batch)
    want, want_lse = op.attend(wl.q, 0, meta, return_lse=True)
    W, Hq, D = meta.num_workers, op.num_qo_heads, op.head_dim
    out = torch.full((W, Hq * D), float("nan"), dtype=op.dtype, device=DEV)
    lse = torch.full((W, Hq), float("nan"), dtype=torch.float32, device=DEV)
    # one call first: the once-per-device lookup of the array's address (and whatever the runtime
    # sets up lazily for a kernel's first launch) is kept apart from the steady-state call measured below
    op.attend(wl.q, 0, meta, return_lse=True, out=out, lse=lse, static_scratch=True)
    out.fill_(float("nan"))
    lse.fill_(float("nan"))
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats(DEV)["allocation.all.allocated"]
    free_before, _ = torch.cuda.mem_get_info(DEV)
    got, got_lse = op.attend(wl.q, 0, meta, return_lse=True, out=out, lse=lse, static_scratch=True)
    assert torch.cuda.memory_stats(DEV)["allocation.all.allocated"] == before  # torch allocated nothing either
    torch.cuda.synchronize()
    # ... and neither did the library behind torch's back: the device's free memory is what it was
    free_after, _ = torch.cuda.mem_get_info(DEV)
    assert free_after == free_before, f"device memory in use changed by {free_before - free_after} bytes"
    assert got.data_ptr() == out.data_ptr()
    assert torch.equal(got, want) and torch.equal(got_lse, want_lse)
    return counts.workspace_bytes


def test_static_scratch_matches_the_workspace_path_twice_in_a_row():
    # 24 requests over a shared block: a few hundred partial states of 16 heads x (256 + 2) floats
    big = _both_ways(workloads.batched_decode(DEV, workers=24, shared_len=4096, private_lo=200, private_hi=3000))
    # then a smaller launch (other head layout, other plan) over the same array
    small = _both_ways(workloads.batched_decode(DEV, workers=3, shared_len=900, private_lo=40, private_hi=700,
                                                heads=(8, 2, 128), seed=7))
    assert small < big
    # and a prefill whose tiles are split by tokens (partial states written by the wide kernel)
    _both_ways(workloads.view_prefill(DEV, requests=1, new_tokens=64, own_prefix=32, prompt_len=6000))


def test_static_scratch_refuses_a_plan_that_does_not_fit():
    wl = workloads.mixed_batch(DEV, decode_rows=8, chunks=2, chunk_len=512, ctx_lo=20000, ctx_hi=30000)
    op, meta = wl.op, wl.meta
    assert meta.launch.counts.workspace_bytes > native.STATIC_SCRATCH_BYTES
    out = torch.empty((meta.num_workers, op.num_qo_heads * op.head_dim), dtype=op.dtype, device=DEV)
    with pytest.raises(native.ViewAttnError, match="va_attention_static.*scratch"):
        op.attend(wl.q, 0, meta, out=out, static_scratch=True)
    op.attend(wl.q, 0, meta, out=out)  # the workspace path takes it
    torch.cuda.synchronize()


def _cut_finely(heads, new, context):
    """A prefill whose fine cuts leave too many partial states for the array, and its coarse ones not."""
    page, total = 16, -(-new // 16) + -(-context // 16)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, torch.bfloat16, heads, page, total, 1e6, seed=new, scale=0.5)
    blocks = []
    if context:
        blocks.append(CacheBlock(DEV, page))
        blocks[0].grow_pages(torch.arange(-(-context // page)) * page, context)
    specs = [PrefillSpec(blocks, torch.arange(-(-context // page), total, dtype=torch.int32) * page, new)]
    *_, meta = run_prefill_parity(op, cpu_pool, dev_pool, specs, 1e6, gen, scale=0.5)
    assert meta.launch.counts.workspace_bytes > native.STATIC_SCRATCH_BYTES
    q = torch.randn(new, heads[0] * heads[2], generator=gen).to(op.dtype).to(DEV)
    return op, meta, q, op.attend(q, 0, meta, return_lse=True)


@pytest.mark.parametrize("heads,new,context", [((32, 8, 128), 1500, 0), ((16, 4, 256), 800, 1000)])
def test_static_scratch_takes_what_coarser_cuts_fit(heads, new, context):
    op, meta, q, (want, want_lse) = _cut_finely(heads, new, context)
    out, lse = torch.full_like(want, float("nan")), torch.full_like(want_lse, float("nan"))
    for _ in range(2):
        op.attend(q, 0, meta, return_lse=True, out=out, lse=lse, static_scratch=True)
        assert_close(out, want.float(), op.dtype, "out")
        assert_close(lse, want_lse, op.dtype, "lse")
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
    again = op.attend(q, 0, meta)  # the first plan is untouched
    assert torch.equal(again, want)


def test_static_scratch_takes_them_under_capture():
    op, meta, q, (want, want_lse) = _cut_finely((32, 8, 128), 1000, 500)
    out, lse = torch.empty_like(want), torch.empty_like(want_lse)
    other = op.attend(q, 0, meta)  # (loads the kernels)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        op.attend(q, 0, meta, return_lse=True, out=out, lse=lse, static_scratch=True)
    for _ in range(3):
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert_close(out, want.float(), op.dtype, "out")
        assert_close(lse, want_lse, op.dtype, "lse")
        assert torch.equal(op.attend(q, 0, meta), other)
