"""Decode rows and prefill chunks in one launch, with the CUs shared out between the wide tiles and the streaming ones:
the result is that of the same plan on the vector-ALU kernel, whose items all take the same path."""

import pytest
import torch

from async_llm_amd import native, workloads
from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,heads,page", [(torch.bfloat16, (16, 4, 256), 16), (torch.float16, (8, 2, 128), 16),
                                              (torch.bfloat16, (32, 8, 128), 1), (torch.bfloat16, (64, 16, 64), 32),
                                              (torch.float16, (16, 4, 256), 8)])
@pytest.mark.parametrize("rows,chunks,chunk", [(40, 2, 129), (9, 1, 33), (33, 3, 77), (1, 1, 300)])
def test_wide_and_streaming_items_share_a_launch(dtype, heads, page, rows, chunks, chunk):
    print(f"heads {heads} page {page} rows {rows} chunks {chunks} x {chunk}", flush=True)
    wl = workloads.mixed_batch(DEV, decode_rows=rows, chunks=chunks, chunk_len=chunk, ctx_lo=300, ctx_hi=6000,
                               shared_len=200, heads=heads, dtype=dtype, page_size=page, kernel="mfma")
    counts = wl.meta.launch.counts
    assert 0 < counts.n_wide_items < counts.n_items
    out, lse = wl.op.forward_with_lse(wl.q, wl.k, wl.v, 0, wl.batch)
    wl.op.plan_params.kernel = native.VA_KERNEL_GENERIC
    other = wl.op.prepare_mixed(wl.group, wl.pending, wl.new_token_slots, wl.specs)
    assert other.launch.counts.kernel == native.VA_KERNEL_GENERIC
    expected, expected_lse = wl.op.attend(wl.q, 0, other, return_lse=True)
    assert_close(out.cpu(), expected.cpu().view_as(out.cpu()), dtype, "out")
    assert_close(lse.cpu(), expected_lse.cpu(), dtype, "lse")
    # planned again, the same bits: nothing hangs on which workgroup a CU gets first
    wl.op.plan_params.kernel = native.VA_KERNEL_MFMA
    fresh = wl.op.prepare_mixed(wl.group, wl.pending, wl.new_token_slots, wl.specs)
    assert fresh.launch.counts.kernel == native.VA_KERNEL_MFMA
    for meta in (wl.meta, fresh):
        again, again_lse = wl.op.attend(wl.q, 0, meta, return_lse=True)
        assert torch.equal(out, again) and torch.equal(lse, again_lse)


@pytest.mark.parametrize("dtype,heads,page,apart", [(torch.bfloat16, (64, 16, 64), 16, 3), (torch.float16, (32, 8, 128), 16, 3),
                                                    (torch.bfloat16, (32, 16, 128), 1, 3), (torch.float16, (64, 16, 64), 24, 3),
                                                    (torch.bfloat16, (16, 4, 256), 16, 0)])
def test_short_rows_beside_a_chunk_get_a_launch_of_their_own(dtype, heads, page, apart):
    print(f"heads {heads} page {page}", flush=True)
    wl = workloads.mixed_batch(DEV, decode_rows=128, chunks=1, chunk_len=100, ctx_lo=200, ctx_hi=500, shared_len=64,
                               heads=heads, dtype=dtype, page_size=page, kernel="mfma")
    assert wl.meta.launch.counts.n_wide_items > 0 and wl.meta.launch.header[3] % 64 == apart
    out, lse = wl.op.forward_with_lse(wl.q, wl.k, wl.v, 0, wl.batch)
    wl.op.plan_params.kernel = native.VA_KERNEL_GENERIC
    expected, expected_lse = wl.op.attend(wl.q, 0, wl.op.prepare_mixed(wl.group, wl.pending, wl.new_token_slots, wl.specs),
                                          return_lse=True)
    assert_close(out.cpu(), expected.cpu().view_as(out.cpu()), dtype, "out")
    assert_close(lse.cpu(), expected_lse.cpu(), dtype, "lse")
