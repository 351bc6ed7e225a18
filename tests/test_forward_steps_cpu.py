"""``forward`` and ``forward_with_lse`` are the store and the attention of a layer: steps that a subclass, a class-wide or an
instance-wide wrapper puts in their place are the ones that run."""

from types import SimpleNamespace

import pytest
import torch

from async_llm_amd import native
from async_llm_amd.shared_cache import SharedCacheAttention
from async_llm_amd.shared_cache.attention import SharedCacheAttnMetadata


@pytest.mark.parametrize("place", ["subclass", "class", "instance"])
@pytest.mark.parametrize("replaced", [("store_new_kv", "attend"), ("store_new_kv",), ("attend",), ()])
def test_replaced_steps_run(place, replaced, monkeypatch):
    seen = []

    class Quiet(SharedCacheAttention):  # what the steps that are not replaced launch, without a GPU
        def _store(self, k, v, layer_id, batch, *rest):
            seen.append(("store", k, v, layer_id))

        def _attend(self, q, meta, pools, stream, return_lse=False, lse_base2=False, *rest):
            seen.append(("attend", q, pools[0], return_lse, lse_base2))

    def store_new_kv(k, v, layer_id, batch):
        seen.append(("replaced store", k, v, layer_id))

    def attend(q, layer_id, meta, return_lse=False, lse_base2=False):
        seen.append(("replaced attend", q, layer_id, return_lse, lse_base2))

    steps = {"store_new_kv": store_new_kv, "attend": attend}
    methods = {name: lambda self, *args, _f=steps[name], **kwargs: _f(*args, **kwargs) for name in replaced}
    own = type("Own", (Quiet,), methods if place == "subclass" else {})
    if place == "class":
        for name, method in methods.items():
            monkeypatch.setattr(SharedCacheAttention, name, method)
    monkeypatch.setattr(native, "current_stream_ptr", lambda device: 0)
    pool = SimpleNamespace(k_cache=lambda layer: None if layer == 0 else layer, v_cache=lambda layer: None)
    op = own(pool, torch.zeros(4, 64), 8, 2, 64, 16, torch.bfloat16, torch.device("cpu"))
    if place == "instance":
        for name in replaced:
            setattr(op, name, steps[name])
    nothing = torch.zeros(0)
    batch = SimpleNamespace(attn_metadata=SharedCacheAttnMetadata(op, nothing, nothing, nothing, 1, 1))
    op.forward("q", "k", "v", 2, batch)
    op.forward_with_lse("q", "k", "v", 3, batch, True)
    store, attend = (("replaced " if name in replaced else "") for name in steps)
    assert seen == [(store + "store", "k", "v", 2), (attend + "attend", "q", 2, False, False),
                    (store + "store", "k", "v", 3), (attend + "attend", "q", 3, True, True)]
