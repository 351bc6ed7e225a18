"""The work a serving program has this framework do, as measurable cases.

A pass is one step of such a program as it calls the framework: plan the step
(``prepare`` / ``prepare_prefill_batch`` / ``prepare_mixed`` / ``prepare_metadata``)
from blocks, views and slots that the program holds, then run ``forward`` once per
attention layer; or, for a block merge, one ``merge_blocks`` over all layers.  Planning
belongs to the pass because every step has other lengths and positions.  The pool, the
blocks with their scattered pages, this step's slots and each layer's unrotated q/k/v
are what the program has in hand before it.  A pass writes the same new rows into the
same slots every time, so it can be repeated.

Results are the attention output of every layer and the pool with the new rows in it.

Ragged lengths come from a case's ``shape`` number, so that ``work`` knows them; values,
page order and token slots come from the seed.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

from async_llm_amd.attention_backend import ViewAttnBackend
from async_llm_amd.kvcache import MHAKVCache, PageAllocator
from async_llm_amd.shared_cache import BlockKVOps, CacheBlock, PrefillSpec, SharedCacheAttention, WorkerGroup
from async_llm_amd.shared_cache.attention_graph import SharedDecodeAttentionBuffers
from async_llm_amd.shared_cache.session_planning import plan_decode_writes

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
MROPE_SECTIONS = {64: (12, 10, 10), 128: (24, 20, 20)}  # by rotary width: pair dims of time, height and width


def _model(hq, hkv, d, dtype="bf16", layers=4, rope="table", page=16):
    return dict(hq=hq, hkv=hkv, d=d, dtype=dtype, layers=layers, rope=rope, page=page)


def listed():
    wide = (16, 4, 256)  # the attention shape of the benchmark's configurations
    usual = (32, 8, 128)  # the same query width in the more common head size
    return [
        # one agent with a short view, float32: the smallest step there is (benchmark configuration 1)
        dict(name="plumbing_decode", kind="decode", workers=1, shared=256, views=2, private_lo=512, private_hi=1024,
             shape=1, **_model(8, 2, 128, "f32", layers=1)),
        # a few cooperating agents over one prompt and each other's notes, launched layer by layer
        dict(name="agents_decode", kind="decode", workers=4, shared=1500, views=3, private_lo=64, private_hi=2048,
             shape=2, **_model(*wide)),
        # the same kind of step replayed from one recorded graph, as a serving loop does it
        dict(name="agents_replay", kind="replay", workers=8, shared=700, views=3, private_lo=64, private_hi=1500,
             shape=3, **_model(*usual)),
        # a full decode batch over a long shared prompt (benchmark configuration 2)
        dict(name="batched_decode", kind="decode", workers=64, shared=8192, views=3, private_lo=256, private_hi=8192,
             shape=4, **_model(*wide)),
        # eight long-context requests with images in their blocks (benchmark configuration 5)
        dict(name="mrope_decode", kind="decode", workers=8, shared=0, views=8, private_lo=16384, private_hi=16384,
             shape=5, **_model(*wide, layers=2, rope="mrope")),
        # one request takes in a tool result with an image between two decode steps
        dict(name="image_chunk_prefill", kind="prefill", requests=1, new_lo=333, new_hi=333, prefix_lo=100,
             prefix_hi=400, prompt=2048, views=2, private_lo=200, private_hi=1500, peers=False, shape=6,
             **_model(*wide, rope="mrope")),
        # eight long writes at once over a long prompt and each other's blocks (benchmark configuration 3)
        dict(name="view_prefill", kind="prefill", requests=8, new_lo=2048, new_hi=2048, prefix_lo=1024, prefix_hi=1024,
             prompt=32768, views=0, private_lo=0, private_hi=0, peers=True, shape=7, **_model(*wide, layers=1)),
        # ragged writes of ordinary length in float16
        dict(name="ragged_prefill_f16", kind="prefill", requests=4, new_lo=300, new_hi=1500, prefix_lo=0,
             prefix_hi=1000, prompt=8000, views=1, private_lo=50, private_hi=3000, peers=True, shape=8,
             **_model(*usual, "f16", layers=2)),
        # a continuous batch: decode rows and prefill chunks planned as one step (benchmark configuration 4)
        dict(name="mixed_batch", kind="mixed", workers=48, chunks=4, chunk=512, shared=512, views=4, ctx_lo=1024,
             ctx_hi=32768, shape=9, **_model(*wide, layers=2)),
        # requests without a view: ragged prompts, some extending a cached prefix, over token slots
        dict(name="plain_prefill", kind="plain", requests=6, new_lo=60, new_hi=4096, cached_lo=0, cached_hi=2000,
             shape=10, **_model(*usual, page=1)),
        # requests without a view: their decode step
        dict(name="plain_decode", kind="plain", requests=32, new_lo=1, new_hi=1, cached_lo=100, cached_hi=8000,
             shape=11, **_model(*usual, page=1)),
        # two blocks of odd lengths become one
        dict(name="block_merge", kind="merge", left=7001, right=5555, shape=12, **_model(*wide)),
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _span(rng, lo, hi):
    a, b = _log(rng, lo, hi), _log(rng, lo, hi)
    return min(a, b), max(a, b)


def _draw_model(rng, page=None, rope=None):
    hq, hkv, d = rng.choice([(16, 4, 256), (16, 4, 256), (32, 8, 128), (32, 8, 128), (8, 2, 128), (64, 16, 64)])
    return _model(hq, hkv, d, rng.choice(["bf16", "bf16", "bf16", "f16"]), rng.choice([1, 2, 4]),
                  rope or rng.choice(["table", "table", "mrope"]), page or rng.choice([16, 16, 32]))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "decode", "replay", "prefill", "prefill", "prefill", "mixed", "plain",
                       "plain", "merge", "f32"])
    shape = rng.randrange(1 << 20)
    if kind in ("decode", "f32"):
        lo, hi = _span(rng, 64, 16384 if kind == "decode" else 1024)
        model = _draw_model(rng) if kind == "decode" else _model(8, 2, 128, "f32", 1)
        return dict(kind="decode", workers=_log(rng, 1, 64 if kind == "decode" else 8),
                    shared=_log(rng, 64, 8192 if kind == "decode" else 1024), views=rng.randint(1, 4), private_lo=lo,
                    private_hi=hi, shape=shape, **model)
    if kind == "replay":
        lo, hi = _span(rng, 64, 4096)
        return dict(kind="replay", workers=_log(rng, 1, 16), shared=_log(rng, 64, 4096), views=rng.randint(1, 3),
                    private_lo=lo, private_hi=hi, shape=shape, **_draw_model(rng, rope="table"))
    if kind == "prefill":
        n, c, p = _span(rng, 16, 2048), _span(rng, 16, 2048), _span(rng, 1, 1024)
        return dict(kind="prefill", requests=_log(rng, 1, 8), new_lo=n[0], new_hi=n[1], prefix_lo=p[0], prefix_hi=p[1],
                    prompt=_log(rng, 64, 32768), views=rng.randint(0, 2), private_lo=c[0], private_hi=c[1],
                    peers=rng.random() < 0.5, shape=shape, **_draw_model(rng))
    if kind == "mixed":
        lo, hi = _span(rng, 1024, 32768)
        return dict(kind="mixed", workers=_log(rng, 2, 48), chunks=rng.randint(1, 4), chunk=_log(rng, 64, 512),
                    shared=_log(rng, 64, 512), views=rng.randint(1, 4), ctx_lo=lo, ctx_hi=hi, shape=shape,
                    **_draw_model(rng, rope="table"))
    if kind == "plain":
        decode = rng.random() < 0.5
        n = (1, 1) if decode else _span(rng, 16, 4096)
        c = _span(rng, 16, 8000 if decode else 2000)
        return dict(kind="plain", requests=_log(rng, 1, 32 if decode else 8), new_lo=n[0], new_hi=n[1], cached_lo=c[0],
                    cached_hi=c[1], shape=shape, **_draw_model(rng, page=1, rope="table"))
    return dict(kind="merge", left=_log(rng, 64, 16384), right=_log(rng, 64, 16384), shape=shape, **_draw_model(rng))


def draw(rng):
    # no drawn pass is dearer than the dearest listed one: at most half its products (other head sizes
    # reach lower rates), no more memory traffic than the full decode batch
    while True:
        case = _draw_once(rng)
        w = work(case)
        if w["flops"] <= 5.5e12 and w["bytes"] <= 9.2e9:
            return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _sizes(case):
    """The ragged lengths of a case, the same for every seed."""
    r = random.Random(case["shape"])
    k = case["kind"]
    if k in ("decode", "replay"):
        # long-context requests have full views; otherwise the number of blocks differs from agent to agent
        full = case["workers"] == 1 or case["views"] > 4
        return [[r.randint(case["private_lo"], case["private_hi"])
                 for _ in range(case["views"] if full else r.randint(1, case["views"]))] for _ in range(case["workers"])]
    if k == "prefill":
        return [dict(new=r.randint(case["new_lo"], case["new_hi"]), prefix=r.randint(case["prefix_lo"], case["prefix_hi"]),
                     private=[r.randint(case["private_lo"], case["private_hi"]) for _ in range(case["views"])])
                for _ in range(case["requests"])]
    if k == "mixed":
        rows = []
        for _ in range(case["workers"] + case["chunks"]):
            total, parts = r.randint(case["ctx_lo"], case["ctx_hi"]), r.randint(1, case["views"])
            rest = max(total - case["shared"], 16 * parts)
            cuts = sorted(r.randint(0, rest - 16 * parts) for _ in range(parts - 1))
            ends = cuts + [rest - 16 * parts]
            rows.append([16 + b - a for a, b in zip([0] + cuts, ends)])
        return rows
    if k == "plain":
        return [(r.randint(case["cached_lo"], case["cached_hi"]), r.randint(case["new_lo"], case["new_hi"]))
                for _ in range(case["requests"])]
    return case["left"], case["right"]


def work(case):
    """K and V of every distinct token read once, q, out and the new rows once, per layer; 4*D*Hq operations
    per visible (query row, key) pair."""
    size = {"f32": 4, "f16": 2, "bf16": 2}[case["dtype"]]
    row = 2 * case["hkv"] * case["d"] * size  # K and V of one token
    sizes, k = _sizes(case), case["kind"]
    if k == "merge":
        return {"bytes": 2 * case["layers"] * row * sum(sizes), "flops": 0}
    if k in ("decode", "replay"):
        rows = len(sizes)
        tokens = case["shared"] + sum(map(sum, sizes)) + rows
        pairs = sum(case["shared"] + sum(s) + 1 for s in sizes)
    elif k == "prefill":
        rows = sum(s["new"] for s in sizes)
        held = sum(s["prefix"] for s in sizes)
        tokens = case["prompt"] + held + rows + sum(sum(s["private"]) for s in sizes)
        pairs = sum(s["new"] * (case["prompt"] + sum(s["private"]) + (held if case["peers"] else s["prefix"]))
                    + s["new"] * (s["new"] + 1) // 2 for s in sizes)
    elif k == "mixed":
        w, c = case["workers"], case["chunk"]
        rows = w + case["chunks"] * c
        tokens = case["shared"] + sum(map(sum, sizes)) + rows
        pairs = sum(case["shared"] + sum(s) + 1 for s in sizes[:w])
        pairs += sum(c * (case["shared"] + sum(s)) + c * (c + 1) // 2 for s in sizes[w:])
    else:
        rows = sum(n for _, n in sizes)
        tokens = sum(c + n for c, n in sizes)
        pairs = sum(n * c + n * (n + 1) // 2 for c, n in sizes)
    width = case["hq"] * case["d"]
    return {"bytes": case["layers"] * (row * tokens + 2 * rows * width * size + rows * row),
            "flops": case["layers"] * 4 * width * pairs}


def tolerance(case):
    # four times the 2-norm difference measured between the matrix-core kernels and the vector-ALU one, and
    # between plans that sum in another order: 1.7e-7 in float32, 3.8e-4 in float16, 3.0e-3 in bfloat16
    return {"rel": {"f32": 8e-7, "f16": 1.5e-3, "bf16": 1.2e-2}[case["dtype"]]}


# ---------------------------------------------------------------------------
# what a program holds before the step
# ---------------------------------------------------------------------------
class _Setup:
    """Pool with content, the op over it, and blocks on scattered pages."""

    def __init__(self, case, seed, tokens, spare_pages, max_pos):
        self.dev = torch.device("cuda")
        self.case, self.page, self.dtype = case, case["page"], DTYPES[case["dtype"]]
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        pages = sum(-(-n // self.page) for n in tokens) + spare_pages
        self.pool = MHAKVCache(hkv, case["layers"], d, pages, self.page, self.dtype, self.dev)
        for layer in range(case["layers"]):
            self.pool.k_cache(layer).normal_(generator=self.gen)
            self.pool.v_cache(layer).normal_(generator=self.gen)
        self.allocator = PageAllocator(pages, self.page, self.dev)
        every = self.allocator.alloc_pages(pages)
        self.allocator.free_pages(every[torch.randperm(pages, device=self.dev, generator=self.gen)])
        if case["rope"] == "mrope":
            rotary = min(d, 128)
            self.op = SharedCacheAttention(self.pool, torch.zeros(1, rotary, device=self.dev), hq, hkv, d, self.page,
                                           self.dtype, self.dev, rotary_dim=rotary,
                                           mrope_section=MROPE_SECTIONS[rotary], rope_base=1e7)
        else:
            inv = 1.0 / (1e7 ** (torch.arange(0, d, 2, dtype=torch.float32, device=self.dev) / d))
            angle = torch.arange(max_pos, dtype=torch.float32, device=self.dev)[:, None] * inv[None, :]
            self.op = SharedCacheAttention(self.pool, torch.cat([angle.cos(), angle.sin()], dim=1), hq, hkv, d,
                                           self.page, self.dtype, self.dev)

    def block(self, length):
        b = CacheBlock(self.dev, self.page)
        if length:
            b.grow_pages(self.allocator.alloc_pages(b.pages_needed(length)), length)
            if self.case["rope"] == "mrope":  # an image of a quarter of the block moves positions by its side only
                side = math.isqrt(length // 4)
                b.mrope_span_override = length - side * side + side
        return b

    def rows(self, n):
        """This step's q, k and v of every layer."""
        c = self.case
        scale = c["d"] ** -0.5 if c["dtype"] == "f32" else 1.0

        def one(heads):
            x = torch.randn(n, heads * c["d"], device=self.dev, generator=self.gen) * scale
            return x.to(self.dtype)

        return [(one(c["hq"]), one(c["hkv"]), one(c["hkv"])) for _ in range(c["layers"])]

    def pools(self):
        return [f(layer) for layer in range(self.case["layers"]) for f in (self.pool.k_cache, self.pool.v_cache)]


def _chunk(setup, own, new):
    """Pages and slots of `new` tokens written behind block `own`."""
    P = setup.page
    fresh = setup.allocator.alloc_pages(own.pages_needed(new)).cpu()
    starts = torch.cat([torch.tensor(own.page_starts, dtype=torch.int32), fresh])
    slots = (starts[:, None] + torch.arange(P, dtype=torch.int32)[None, :]).reshape(-1)
    return starts, slots[own.num_tokens: own.num_tokens + new]


def _image_positions(new):
    """Positions of text, one image of a quarter of the tokens, text, in three axes."""
    side = math.isqrt(new // 4)
    lead = (new - side * side) // 2
    tail = new - lead - side * side
    text = torch.arange(lead).expand(3, -1)
    grid = torch.stack([torch.zeros(side * side, dtype=torch.int64), torch.arange(side * side) // max(1, side),
                        torch.arange(side * side) % max(1, side)]) + lead
    return torch.cat([text, grid, (torch.arange(tail) + lead + side).expand(3, -1)], dim=1)


def _decode_group(setup, shared, lengths):
    views = [([shared] if shared is not None else []) + [setup.block(n) for n in ls] for ls in lengths]
    group = WorkerGroup(cache_structure=views, write_to=[v[-1] for v in views])
    pending, slots, positions = plan_decode_writes(group, setup.page, setup.allocator, setup.dev)
    return group, pending, slots, positions


def _batch(positions, out_loc, mrope_positions=None):
    return SimpleNamespace(attn_metadata=None, positions=positions, out_loc=out_loc, mrope_positions=mrope_positions)


def prepare(case, seed):
    return {"decode": _prepare_decode, "replay": _prepare_replay, "prefill": _prepare_prefill,
            "mixed": _prepare_mixed, "plain": _prepare_plain, "merge": _prepare_merge}[case["kind"]](case, seed)


def _prepare_decode(case, seed):
    lengths = _sizes(case)
    tokens = [case["shared"]] + [n for ls in lengths for n in ls]
    max_pos = case["shared"] + max(map(sum, lengths)) + 64
    setup = _Setup(case, seed, tokens, len(lengths), max_pos)
    shared = setup.block(case["shared"]) if case["shared"] else None
    group, pending, slots, positions = _decode_group(setup, shared, lengths)
    batch = _batch(torch.tensor(positions, dtype=torch.int64, device=setup.dev), slots)
    return dict(run=_run_decode, setup=setup, group=group, pending=pending, slots=slots, batch=batch,
                rows=setup.rows(len(lengths)))


def _prepare_replay(case, seed):
    state = _prepare_decode(case, seed)
    setup, workers, depth = state["setup"], case["workers"], case["views"] + 1
    op, batch = setup.op, state["batch"]
    entries = -(-(case["shared"] + 1) // setup.page) + depth * (-(-(case["private_hi"] + 1) // setup.page) + 1)
    buffers = SharedDecodeAttentionBuffers(op, workers, depth, workers * entries)
    op.prepare_workspace([buffers])
    batch.attn_metadata = op.prepare(state["group"], state["pending"], state["slots"], graph_buffers=buffers)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        op.forward(*state["rows"][0], 0, batch)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [op.forward(q, k, v, layer, batch) for layer, (q, k, v) in enumerate(state["rows"])]
    state.update(run=_run_replay, buffers=buffers, graph=graph, outs=outs)
    return state


def _prepare_prefill(case, seed):
    sizes = _sizes(case)
    tokens = [case["prompt"]] + [n for s in sizes for n in s["private"] + [s["prefix"], s["new"]]]
    max_pos = case["prompt"] + sum(s["prefix"] for s in sizes) + max(s["new"] + sum(s["private"]) for s in sizes) + 64
    setup = _Setup(case, seed, tokens, len(sizes), max_pos)
    prompt = setup.block(case["prompt"])
    own = [setup.block(s["prefix"]) for s in sizes]
    specs, positions, out_loc = [], [], []
    for r, s in enumerate(sizes):
        context = [prompt] + [setup.block(n) for n in s["private"]]
        if case["peers"]:
            context += [b for i, b in enumerate(own) if i != r and b.num_tokens]
        starts, slots = _chunk(setup, own[r], s["new"])
        image = _image_positions(s["new"]) if case["rope"] == "mrope" else None
        specs.append(PrefillSpec(context, starts, s["new"], own[r].num_tokens, own[r].mrope_span, image))
        positions.append((torch.arange(s["new"]) if image is None else image) + own[r].mrope_span)
        out_loc.append(slots)
    pos = torch.cat(positions, dim=-1).to(setup.dev)
    mrope = pos.contiguous() if case["rope"] == "mrope" else None
    batch = _batch(pos if mrope is None else pos[0].contiguous(), torch.cat(out_loc).to(setup.dev), mrope)
    return dict(run=_run_prefill, setup=setup, specs=specs, batch=batch, rows=setup.rows(sum(s["new"] for s in sizes)))


def _prepare_mixed(case, seed):
    sizes, w, c = _sizes(case), case["workers"], case["chunk"]
    tokens = [case["shared"]] + [n for ls in sizes for n in ls]
    setup = _Setup(case, seed, tokens, w + case["chunks"] * (-(-c // case["page"]) + 1),
                   case["shared"] + max(map(sum, sizes)) + c + 64)
    shared = setup.block(case["shared"])
    group, pending, slots, written = _decode_group(setup, shared, sizes[:w])
    specs, positions, out_loc = [], [torch.tensor(written, dtype=torch.int64)], [slots.cpu()]
    for ls in sizes[w:]:
        blocks = [setup.block(n) for n in ls]
        own, context = blocks[-1], [shared] + blocks[:-1]
        starts, new_slots = _chunk(setup, own, c)
        specs.append(PrefillSpec(context, starts, c, own.num_tokens))
        positions.append(torch.arange(own.num_tokens, own.num_tokens + c))
        out_loc.append(new_slots)
    batch = _batch(torch.cat(positions).to(setup.dev), torch.cat(out_loc).to(setup.dev))
    return dict(run=_run_mixed, setup=setup, group=group, pending=pending, slots=slots, specs=specs, batch=batch,
                rows=setup.rows(w + case["chunks"] * c))


def _prepare_plain(case, seed):
    sizes = _sizes(case)
    setup = _Setup(case, seed, [c + n for c, n in sizes], 0, 64)
    longest = max(c + n for c, n in sizes)
    table = torch.zeros(len(sizes), longest, dtype=torch.int32, device=setup.dev)
    reqs, out_loc = [], []
    for i, (cached, new) in enumerate(sizes):
        table[i, : cached + new] = setup.allocator.alloc_pages(cached + new)  # pages of one token: token slots
        reqs.append(SimpleNamespace(table_idx=i, cached_len=cached, extend_len=new, device_len=cached + new))
        out_loc.append(table[i, cached: cached + new])
    config = SimpleNamespace(num_qo_heads=case["hq"], num_kv_heads=case["hkv"], head_dim=case["d"])
    decode = case["new_hi"] == 1
    batch = SimpleNamespace(reqs=reqs, padded_reqs=reqs, size=len(reqs), padded_size=len(reqs), is_decode=decode,
                            is_prefill=not decode, out_loc=torch.cat(out_loc), attn_metadata=None)
    return dict(run=_run_plain, setup=setup, backend=ViewAttnBackend(config, setup.pool, table), batch=batch,
                rows=setup.rows(sum(n for _, n in sizes)))


def _prepare_merge(case, seed):
    left, right = _sizes(case)
    spare = 2 * -(-(left + right) // case["page"]) + 2  # room for two merged blocks
    setup = _Setup(case, seed, [left, right], spare, left + right + 64)
    ops = BlockKVOps(setup.pool, setup.op, setup.allocator)
    ids = random.Random(seed)
    blocks = [setup.block(left), setup.block(right)]
    for b in blocks:
        b.token_ids = [ids.randrange(150000) for _ in range(b.num_tokens)]
    return dict(run=_run_merge, setup=setup, ops=ops, blocks=blocks)


# ---------------------------------------------------------------------------
# the step
# ---------------------------------------------------------------------------
def run(state):
    return state["run"](state)


def _layers(op, state):
    batch = state["batch"]
    outs = [op.forward(q, k, v, layer, batch) for layer, (q, k, v) in enumerate(state["rows"])]
    return outs, state["setup"].pools()


def _run_decode(state):
    op = state["setup"].op
    state["batch"].attn_metadata = op.prepare(state["group"], state["pending"], state["slots"])
    return _layers(op, state)


def _run_replay(state):
    state["setup"].op.prepare(state["group"], state["pending"], state["slots"], graph_buffers=state["buffers"])
    state["graph"].replay()
    return state["outs"], state["setup"].pools()


def _run_prefill(state):
    op = state["setup"].op
    state["batch"].attn_metadata = op.prepare_prefill_batch(state["specs"])
    return _layers(op, state)


def _run_mixed(state):
    op = state["setup"].op
    state["batch"].attn_metadata = op.prepare_mixed(state["group"], state["pending"], state["slots"], state["specs"])
    return _layers(op, state)


def _run_plain(state):
    state["backend"].prepare_metadata(state["batch"])
    return _layers(state["backend"], state)


def _run_merge(state):
    merged = state["ops"].merge_blocks(*state["blocks"])
    # the program is done with it at once here: the pages go back to the end of the free list
    setup = state["setup"]
    setup.allocator.free_pages(torch.tensor(merged.clear(), dtype=torch.int32))
    return setup.pools()
