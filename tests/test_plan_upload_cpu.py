"""A step's plan and tables go to the device as one staging tensor: what arrives is what was planned."""

from types import SimpleNamespace

import numpy as np
import torch

from async_llm_amd import native
from async_llm_amd.shared_cache import SharedCacheAttention

from .test_chain_cuts_cpu import _tables

CPU = torch.device("cpu")


def _op(page=16):
    return SharedCacheAttention(SimpleNamespace(), torch.zeros(4, 256), 16, 4, 256, page, torch.bfloat16, CPU)


def _launch(op, requests, refs):
    """Plan chained requests on ``op``; the launch, and the plan's words as an op of its own makes them."""
    qo, kvp, kvi, lens, flags, chain, sw, n_rows = _tables(requests, op.page_size)
    args = dict(qo_indptr=qo, kv_indptr=kvp, kv_indices_host=np.asarray(kvi, dtype=np.int32), seq_lens=lens, flags=flags,
                chain=chain, sub_worker_host=np.asarray(sw, dtype=np.int64), n_rows=n_rows)
    return op._build_launch(tables=(), refs=refs, **args)[0], _op(op.page_size)._build_launch(tables=(), refs=[], **args)[0]


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
