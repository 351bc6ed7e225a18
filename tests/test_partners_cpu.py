"""Narrow tiles that one workgroup serves: its item and the ones behind it at the next turns of its die walk the same
tokens, lie inside the plan, and every tile is served once, in packed and in fixed plans."""

import random

import numpy as np
import pytest

from async_llm_amd import native
from tests.test_fixed_plan_cpu import fixed_plan
from tests.test_native_abi_cpu import H, build_plan, check_coverage, decode_plan

KIND, PARTNERS, LINK0 = 5, 6, 8


def _tables(rng, page):
    kvi, kvp, lens, sw = [], [0], [], []
    fresh = n_rows = 0
    for _ in range(rng.randint(1, 4)):
        length, readers = rng.choice([1, 40, 700, 4095, 4096, 9000]), rng.randint(1, 40)
        pages = list(range(fresh, fresh + -(-length // page)))
        fresh += len(pages)
        for _ in range(readers):
            kvi += pages
            kvp.append(len(kvi)), lens.append(length), sw.append(n_rows)
            own = rng.randint(1, 60)
            kvi += list(range(fresh, fresh + -(-own // page)))
            fresh += -(-own // page)
            kvp.append(len(kvi)), lens.append(own), sw.append(n_rows)
            n_rows += 1
    return list(range(len(lens) + 1)), kvp, kvi, lens, [0] * len(lens), [-1] * len(lens), sw, n_rows


@pytest.mark.parametrize("heads", [(16, 4, 256), (32, 8, 128), (16, 16, 64), (16, 1, 128), (64, 16, 64)])
@pytest.mark.parametrize("page", [1, 8, 16, 24, 64])
@pytest.mark.parametrize("fixed", [False, True])
def test_partners_walk_the_tokens_of_the_item_before_them(heads, page, fixed):
    rng = random.Random(f"{heads}{page}")
    most = 0
    for _ in range(3):
        tables = _tables(rng, page)
        qo, kvp, kvi, lens, flags, chain, sw, n_rows = tables
        if fixed:
            limits = native.VaPlanLimits(len(lens), len(sw), 0, 0, 0, n_rows)
            rc, blob, *_ = fixed_plan(tables, limits, heads=heads, page=page, kernel=native.VA_KERNEL_MFMA)
        else:
            rc, blob, _ = build_plan(*tables, heads=heads, page=page, dtype=native.VA_BF16, kernel=native.VA_KERNEL_MFMA,
                                     wide_tile=-1)
        assert rc == 0, native.lib.va_last_error()
        check_coverage(blob, qo, kvp, lens, flags, sw, n_rows, fixed=fixed)
        header, items, *_ = decode_plan(blob)
        narrow = items[header[H["N_WIDE"]]:]
        served = np.zeros(len(narrow), dtype=int)
        for p, item in enumerate(narrow):
            if item[2] == 0 or item[PARTNERS] < 0:
                continue
            assert item[KIND] == 0 and item[PARTNERS] <= (3 if page >= 16 else 1)
            most = max(most, int(item[PARTNERS]))
            for k in range(1 + item[PARTNERS]):
                other = narrow[p + 8 * k]
                served[p + 8 * k] += 1
                assert other[2] > 0 and (k == 0 or other[PARTNERS] == -1)
                if k:  # one link each, over the same tokens and found the same way; none is causal
                    assert item[1] == other[1] == 1
                    same = [0, 1, 2, 4, 5]  # list, first and last token, causal base, flags: all but the query rows
                    assert [other[LINK0 + w] for w in same] == [item[LINK0 + w] for w in same]
        assert np.array_equal(served, (narrow[:, 2] > 0).astype(int))
    if fixed:  # (packed plans of short items keep their tiles apart; 16 rows of one request fill a tile)
        assert (most > 0) == (heads[0] // heads[1] < 16)


def _readers(readers, shared, own, page=16):
    kvi, kvp, lens, sw = [], [0], [], []
    fresh = -(-shared // page)
    for r in range(readers):
        for pages, length in ((list(range(-(-shared // page))), shared), (list(range(fresh, fresh - (-own // page))), own)):
            kvi += pages
            kvp.append(len(kvi)), lens.append(length), sw.append(r)
        fresh += -(-own // page)
    return list(range(len(lens) + 1)), kvp, kvi, lens, [0] * len(lens), [-1] * len(lens), sw, readers


@pytest.mark.parametrize("heads,readers,shared,own,short,packed,recorded", [
    # all start at once apart (pairs 12.7 us, apart 10.1)
    ((16, 4, 256), 8, 64, 130, False, 0, 0), ((16, 4, 256), 16, 64, 40, True, 0, 0), ((32, 8, 128), 8, 64, 130, False, 0, 0),
    # pairs or fours would leave CUs without a workgroup (fours 29.5 us, apart 16.9; recorded fours 41, pairs 23)
    ((16, 4, 256), 16, 4096, 130, True, 0, 0), ((32, 8, 128), 16, 4096, 130, True, 0, 0),
    ((16, 4, 256), 30, 4096, 130, True, 0, 1),
    # short items with few tokens read again; many read again; long items
    ((32, 8, 128), 64, 2048, 250, True, 0, 1),
    # fours would take most of a recorded launch, whose chunks are longer (235 us, in pairs 198)
    ((16, 4, 256), 256, 4096, 430, False, 3, 1),
    ((32, 8, 128), 128, 4096, 250, False, 3, 3), ((16, 4, 256), 64, 8192, 5000, False, 3, 3),
])
def test_tiles_walk_together_where_the_launch_is_long(heads, readers, shared, own, short, packed, recorded):
    tables = _readers(readers, shared, own)
    rc, blob, _ = build_plan(*tables, heads=heads, page=16, dtype=native.VA_BF16, kernel=native.VA_KERNEL_MFMA, wide_tile=-1)
    assert rc == 0
    header, items, *_ = decode_plan(blob)
    assert (header[H["KV_CHUNK"]] & 1 == 1) == short and max(items[:, PARTNERS]) == packed
    limits = native.VaPlanLimits(2 * readers, 2 * readers, 0, 0, 0, readers)
    rc, blob, *_ = fixed_plan(tables, limits, heads=heads, page=16, kernel=native.VA_KERNEL_MFMA)
    assert rc == 0 and max(decode_plan(blob)[1][:, PARTNERS]) == recorded


@pytest.mark.parametrize("heads,readers,shared,own,wide", [
    ((64, 16, 64), 256, 4096, 250, True), ((64, 16, 64), 128, 8192, 200, True), ((64, 16, 64), 64, 8192, 200, False),
    ((64, 16, 64), 64, 16384, 800, False), ((32, 8, 128), 256, 4096, 64, True), ((32, 8, 128), 256, 4096, 250, False),
    ((32, 8, 128), 512, 4096, 250, True), ((16, 4, 256), 64, 16384, 250, True), ((16, 4, 256), 64, 4096, 250, False)])
def test_many_readers_get_wide_tiles_where_the_rest_is_short(heads, readers, shared, own, wide):
    # us, narrow / wide: 199 / 134, 120 / 114, 70 / 61 (but 106 / 140 beside longer blocks), 129 / 151, 157 / 105, 144 / 154,
    # 315 / 228, 112 / 75, 59 / 64
    rc, _, counts = build_plan(*_readers(readers, shared, own), heads=heads, page=16, dtype=native.VA_BF16,
                               kernel=native.VA_KERNEL_MFMA)
    assert rc == 0 and (counts.n_wide_items > 0) == wide
