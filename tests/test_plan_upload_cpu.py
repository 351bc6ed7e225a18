"""A step's plan and tables go to the device as one staging tensor: what arrives is what was planned."""

import copy
import pickle
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from async_llm_amd import native
from async_llm_amd.shared_cache import SharedCacheAttention

from .test_chain_cuts_cpu import _tables

CPU = torch.device("cpu")


def _op(page=16):
    return SharedCacheAttention(SimpleNamespace(), torch.zeros(4, 256), 16, 4, 256, page, torch.bfloat16, CPU)


def _plan_args(requests, page):
    qo, kvp, kvi, lens, flags, chain, sw, n_rows = _tables(requests, page)
    return dict(qo_indptr=qo, kv_indptr=kvp, kv_indices_host=np.asarray(kvi, dtype=np.int32), seq_lens=lens, flags=flags,
                chain=chain, sub_worker_host=np.asarray(sw, dtype=np.int64), n_rows=n_rows)


def _launch(op, requests, refs):
    """Plan chained requests on ``op``; the launch, and the same of an op of its own."""
    args = _plan_args(requests, op.page_size)
    return op._build_launch(tables=(), refs=refs, **args)[0], _op(op.page_size)._build_launch(tables=(), refs=[], **args)[0]


@pytest.mark.parametrize("roomy", [False, True])
@pytest.mark.parametrize("page", [1, 16])
def test_every_table_arrives_on_a_boundary_of_its_own(roomy, page, monkeypatch):
    if roomy:  # a plan whose states exceed the library's own array keeps a blob apart, with room for a second plan
        monkeypatch.setattr(native, "STATIC_SCRATCH_BYTES", 0)
    op, args = _op(page), _plan_args([(58, 40, [700, 300]), (3, 1, [])], page)
    rng = np.random.default_rng(page)
    three_axes = rng.integers(-9, 1 << 40, (3, 77))
    tables = [rng.integers(0, 1 << 40, 61), three_axes, three_axes[:, 3:9], np.zeros(0, dtype=np.int64),
              rng.integers(0, 1 << 30, 65).astype(np.int32), rng.integers(0, 9, 1), np.zeros((3, 0), dtype=np.int64),
              np.zeros(0, dtype=np.int32)]
    refs = []
    launch, sent = op._build_launch(tables=tables, refs=refs, **args)
    assert (launch.subs is not None) == roomy and launch.counts.workspace_bytes > 0
    words = launch.counts.plan_words
    plan = np.empty(words, dtype=np.int32)
    subs, counts = launch.subs, native.VaPlanCounts()
    if subs is None:
        monkeypatch.setattr(native, "STATIC_SCRATCH_BYTES", 0)
        subs = _op(page)._build_launch(tables=(), refs=[], **args)[0].subs
    assert native.lib.va_plan_build_within(subs, op._shape, op.plan_params, -1, plan.ctypes.data, words, counts) == 0
    assert np.array_equal(launch.blob.numpy()[:words], plan) and launch.blob.numel() == (2 if roomy else 1) * words
    assert np.array_equal(launch.header, plan[: native.PLAN_HEADER_WORDS])
    assert len(sent) == len(tables)
    for want, got in zip([args["kv_indices_host"], *tables], [launch.kv_indices, *sent]):
        assert np.array_equal(got.numpy(), want) and got.numpy().dtype == want.dtype and got.is_contiguous()
        assert got.numel() == 0 or got.storage_offset() * got.element_size() % 256 == 0
    shared = {t.untyped_storage().data_ptr() for t in [launch.kv_indices, *sent] if t.numel()}
    assert len(shared) == 1 and (launch.blob.untyped_storage().data_ptr() in shared) == (not roomy)
    assert {t.untyped_storage().data_ptr() for t in refs} >= shared  # what the transfer reads and writes is kept alive


def test_plans_of_one_op_may_overlap():
    # Another thread may plan on the same op wherever this one's planner or transfers let go of the interpreter: the
    # header that shapes the launch has to be that of the tables beside it.
    op = _op()

    class Interrupted(list):
        def extend(self, items):
            super().extend(items)
            if len(self) == len(items):
                _launch(op, [(700, 5, [3000, 40])], [])

    launch, alone = _launch(op, [(58, 40, [700, 300]), (3, 1, [])], Interrupted())
    assert np.array_equal(launch.header, alone.header)
    assert np.array_equal(launch.blob.numpy()[: native.PLAN_HEADER_WORDS], launch.header)
    assert torch.equal(launch.blob, alone.blob)


def test_the_header_handed_to_a_launch_is_the_plans_own():
    op = _op()
    launch = op._build_launch(tables=(), refs=[], **_plan_args([(58, 40, [700, 300])], 16))[0]
    kept = launch.header.ctypes.data
    copies = [copy.deepcopy(launch), pickle.loads(pickle.dumps(launch))]
    launch.header = launch.header.copy()
    for plan in [launch, *copies]:
        assert plan.header_ptr == plan.header.ctypes.data != kept
        plan.header.flags.writeable = False
        assert plan.header_ptr == plan.header.ctypes.data
