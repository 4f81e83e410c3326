"""The decode plan's item length where whole pages alone would give more items than workgroups (each
row's last item is partly filled): the launch and its merge against the oracle for batches whose first
choice overshoots the grid by a little and by much, and for one where even one item per row and head
is too many (the length then stays); and the lengths themselves: longer ones only where that fits the grid
and they are not too long for it to pay."""
import numpy as np
import pytest
import torch

import q38a
from gpu_util import HD, LD, NKV, NQ, Batch, Pool, attention_params, host, stream
from test_gpu_decode import decode_step

pytestmark = pytest.mark.gpu


def first_plan(ctxs, target):
    pages = [(c + 64) // 64 for c in ctxs]
    cp = max(1, -(-sum(pages) * NKV // target))
    return cp, sum(-(-p // cp) for p in pages) * NKV


@pytest.mark.parametrize("kv_dtype", [q38a.KV_INT8, q38a.KV_BF16])
@pytest.mark.parametrize("rows,tokens", [(49, 385), (100, 257), (140, 64)])
def test_decode_fitted_plan(orc, kv_dtype, rows, tokens):
    target = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    ctxs = [tokens + (7 * i) % 62 for i in range(rows)]
    cp, items = first_plan(ctxs, target)
    assert items > target and (rows == 140) == (rows * NKV > target)
    print(f"fitted plan: rows={rows} cp={cp} items={items}", flush=True)
    decode_step(orc, ctxs, kv_dtype, seed=rows)


def fitted_plan(pages, target, max_splits):
    """csrc/plan.hpp wave_decode_plan<true>: (first choice, pages per item)."""
    rows, total, longest = len(pages), sum(pages), max(pages)
    first = max(1, -(-longest // max_splits), -(-total * NKV // target))
    over = lambda c: sum(-(-p // c) for p in pages) * NKV - target  # noqa: E731
    left = o = over(first)
    if first == 1 or o <= 0 or rows * NKV > target:
        return first, first
    c = first
    for i in range(2):
        if i == 0 and 10 * total >= 9 * rows * longest:
            c = -(-longest // (target // (rows * NKV)))
        else:
            c += -(-c * left // (target - rows * NKV // 2))
        if (min(c, longest) - first - 1) * 2 * target > first * (target + o):
            return first, first
        left = over(c)
        if left <= 0:
            return first, c
    return first, first


# rows of equal length: two items each would become one, past the bound (66, 70, 75) and within it (80, 90,
# 110), three become two (43, 45) and four three (33), one item per row already (126), 128 rows and more; ragged
# rows, where one step fits and where two do
@pytest.mark.parametrize("rows,tokens,spread,longer", [
    (66, 1000, 0, False), (66, 3000, 0, False), (70, 2000, 0, False), (75, 2000, 0, False), (43, 4700, 0, True),
    (45, 3000, 0, True), (43, 1900, 0, True), (33, 6000, 0, True), (80, 1000, 0, True), (90, 2000, 0, True),
    (110, 1800, 0, True), (65, 400, 0, True), (126, 1500, 0, False), (128, 129, 0, False),
    (140, 500, 0, False), (8, 15000, 12000, None), (21, 4000, 700, None), (53, 2200, 1800, None),
    (100, 900, 800, None), (1, 130000, 0, False), (4, 16000, 12000, True), (20, 9000, 6000, True),
    (65, 700, 600, True), (86, 1500, 1200, True), (107, 1500, 1200, None)])
def test_item_lengths(rows, tokens, spread, longer):
    """Keys of zeros give every position the weight 1, so an item's sum of weights is its tokens."""
    target, splits = 2 * torch.cuda.get_device_properties(0).multi_processor_count, 64
    rng = np.random.default_rng(rows)
    lens = [tokens + (int(rng.integers(-spread, spread + 1)) if spread else 0) for _ in range(rows)]
    pages = [-(-n // 64) for n in lens]
    first, cp = fitted_plan(pages, target, splits)
    if target == 512 and longer is not None:
        assert (cp > first) == longer
    print(f"item lengths: rows={rows} tokens={tokens} cp={first}->{cp}", flush=True)
    pool = Pool(q38a.KV_INT8, 1, np.zeros((rows, max(pages)), np.int32))  # one page for all
    b = Batch([(i, n - 1, 1) for i, n in enumerate(lens)])
    q = torch.zeros(rows * NQ * HD, dtype=torch.int16, device="cuda")
    proj = torch.zeros(rows * LD, dtype=torch.int16, device="cuda")
    out = torch.zeros(rows * NQ * HD, dtype=torch.int16, device="cuda")
    scratch = torch.full((q38a.split_scratch_floats(rows, NQ, splits),), float("nan"), device="cuda")
    q38a.attention_decode_partials(attention_params(q, proj, out, scratch, splits), b.desc, pool.desc, stream())
    torch.cuda.synchronize()
    got = host(scratch)[:rows * NQ * splits * (HD + 2)].reshape(rows, NQ, splits, HD + 2)[..., HD + 1]
    for r, n in enumerate(lens):
        want = np.full(splits, np.nan)
        items = -(-pages[r] // cp)
        want[:items] = [min(64 * cp, n - 64 * cp * i) for i in range(items)]
        assert np.array_equal(got[r], np.broadcast_to(want, (NQ, splits)), equal_nan=True), (r, n, got[r, 0])
