"""The decode plan's item length where whole pages alone would give more items than workgroups (each
row's last item is partly filled): the launch and its merge against the oracle for batches whose first
choice overshoots the grid by a little and by much, and for one where even one item per row and head
is too many (the length then stays)."""
import pytest
import torch

import q38a
from gpu_util import NKV
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
