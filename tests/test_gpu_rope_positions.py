"""GPU: RoPE positions where lengths and starts just fit the launch argument, and where the upload takes over."""

import numpy as np
import pytest
import torch

from gpu_helpers import R, log
from mstar_amd import _lib
from mstar_amd.cache_manager import BatchedCacheManager, WorkspaceBufferManager
from mstar_amd.kv_store import KVCacheConfig, PagedAllocationManager

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 399, 400])  # 3, 799 and 801 values; the argument holds 800
def test_positions_at_the_arguments_limit(gpu, batch):
    log(f"positions of {batch} requests")
    cfg = KVCacheConfig(num_layers=1, num_kv_heads=2, head_dim=64, max_seq_len=4096, max_num_pages=16, page_size=16,
                        num_qo_heads=4)
    kv = torch.zeros(1, 16, 2, 16, 2, 64, dtype=torch.bfloat16, device=gpu)
    mgr = PagedAllocationManager(cfg, kv, device=gpu)
    r = np.random.default_rng(batch)
    rids, starts = [f"r{i}" for i in range(batch)], r.integers(0, 3000, batch).tolist()
    for rid, s in zip(rids, starts):
        mgr.add_request(rid, ["main"])
        mgr.get_state(rid, "main").position_id_start = s
    cm = BatchedCacheManager(rids, {rid: "main" for rid in rids}, kv, mgr, WorkspaceBufferManager(64 << 20, gpu), cfg,
                             gpu)
    lens = r.integers(0, 6, batch).tolist()
    lens[-1] = 3
    cm.plan_rope(lens)
    assert cm._plan_states["main"].pos_ids.tolist() == R.positions(lens, starts).tolist()


def test_the_call_refuses_more_than_the_argument_holds(gpu):
    log("positions: 801 values refused")
    meta, out = np.zeros(801, np.int32), torch.full((4,), -1, dtype=torch.long, device=gpu)
    meta[1:401] = 4
    base = meta.ctypes.data
    call = lambda b: _lib.lib().mi_rope_positions_host(base, base + 4 * (b + 1), b, out.data_ptr(), 4, _lib.stream_ptr(gpu))
    assert call(400) == -2 and out.tolist() == [-1] * 4
