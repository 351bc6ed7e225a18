"""Wide tiles whose first exponentials are taken before the tile's maxima are tested (head dims under 256): where the
test then raises the reference they are dropped and the scores computed anew.  Keys whose scores tower over everything
before them are planted in elements that are taken early and late, in tiles around the ends of the part of the walk that
works ahead, one of them right behind another."""

import pytest
import torch

from async_llm_amd.shared_cache import CacheBlock, PrefillSpec
from tests.util import make_op_and_pool, run_prefill_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 128)])
@pytest.mark.parametrize("page", [16, 1])
@pytest.mark.parametrize("planted", [(32,), (64, 97), (65, 79, 126), (128, 160, 192, 224), (90, 351), (383,), (415, 416)])
@pytest.mark.parametrize("step", [15.0, 45.0])
def test_scores_that_rise_within_the_part_that_works_ahead(dtype, D, page, planted, step):
    heads, rotary, length = (8, 2, D), D // 2, 450
    print(f"{dtype} D {D} page {page} planted {planted} step {step}", flush=True)
    op, cpu_pool, dev_pool, gen = make_op_and_pool(DEV, dtype, heads, page, 800 // page, 1e4, rotary_dim=rotary, seed=5,
                                                   scale=1.0, kernel="mfma", max_pos=2048)
    context = CacheBlock(DEV, page)
    pages = -(-length // page)
    context.grow_pages(torch.arange(0, pages) * page, length)
    for n, token in enumerate(planted):  # pages are in order here; the dims past the rotation carry the score
        a = (n + 1) * step * 2.0 / (D ** 0.5 * 1.4426950408889634)
        for pool in (cpu_pool[0], dev_pool[0]):
            pool.view(-1, heads[1], D)[token, :, :rotary] = 0
            pool.view(-1, heads[1], D)[token, :, rotary:] = a
    new = 130
    own = torch.arange(pages, pages + -(-new // page), dtype=torch.int32) * page

    def mutate(q, k, v):
        q.view(-1, heads[0], D)[:, :, rotary:] = 1.0

    *_, meta = run_prefill_parity(op, cpu_pool, dev_pool, [PrefillSpec([context], own, new, 0)], 1e4, gen, scale=0.5,
                                  mutate=mutate)
    assert meta.launch.counts.n_wide_items > 0
