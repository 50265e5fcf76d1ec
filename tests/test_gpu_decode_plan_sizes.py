"""GPU: the item size of decode plans around 1024 requests, where the plan searches it another way."""

import numpy as np
import pytest
import torch

from gpu_helpers import P, custom_batch, log, workspace
from mstar_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1023, 1024, 1025, 2049])
@pytest.mark.parametrize("served", [0, 1, 37, 100, None])  # requests with pages; None: all
def test_item_size_matches_the_rule(gpu, batch, served):
    """Requests without pages make a large batch a small job: searched among those
    that have some, and not at all where they outnumber the slots."""
    hq, hkv, d, ps = 8, 1, 256, 16  # one slot per CU; no kv-head pairs
    r = np.random.default_rng(batch)
    lens = np.zeros(batch, np.int64)
    at = r.permutation(batch)[: batch if served is None else served]
    lens[at] = r.integers(1, 40 if served is None else 2000, len(at))
    pool = int((-(-lens // ps)).sum()) + 1
    _, indptr, indices, last = custom_batch(lens, ps, pool, 3)
    ws = workspace(gpu, 512 << 20)
    dev = [torch.as_tensor(x).to(gpu) for x in (indptr, np.append(indices, 0).astype(np.int32), last)]
    _lib.check(_lib.lib().mi_decode_plan(None, *(t.data_ptr() for t in dev), batch, ps, hq, hkv, d, None,
                                         ws.data_ptr(), ws.numel(), _lib.stream_ptr(gpu)), "mi_decode_plan")
    h = ws[:20].cpu().view(torch.int32).tolist()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    pages, items = P.split_chunks(indptr, ps, 1024, hkv, slots=cus)
    log(f"decode plan of {batch} requests, {len(at)} with pages: item pages {h[3]}, rule {pages}")
    assert h[1] == batch and h[3] == pages and h[2] == int(items.sum())
