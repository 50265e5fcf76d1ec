"""GPU: arguments that the plan calls over host and pinned index arrays refuse before they launch."""

import ctypes

import pytest
import torch

from gpu_helpers import log, workspace
from mstar_amd import _lib

pytestmark = pytest.mark.gpu

INVALID = -1


@pytest.mark.parametrize("num_indices,kv_indices,status", [(5, False, INVALID), (-1, True, INVALID), (5, True, 0), (0, False, 0)])
def test_pinned_plans_without_requests(gpu, num_indices, kv_indices, status):
    """No request needs a page list, but the launch copies num_indices values: they need a destination."""
    log(f"pinned plans, no requests: num_indices={num_indices} kv_indices given={kv_indices}")
    L, ws = _lib.lib(), workspace(gpu, 64 << 20)
    src = torch.zeros(64, dtype=torch.int32, pin_memory=True)
    src[2:7] = torch.arange(7, 12, dtype=torch.int32)  # behind qo_indptr [0] and kv_indptr [0]
    dst = torch.full((4, 16), -1, dtype=torch.int32, device=gpu)
    qo, ip, last, idx = (ctypes.c_void_p(t.data_ptr()) for t in dst)
    idx = idx if kv_indices else None
    tail = (ctypes.c_void_p(ws.data_ptr()), ws.numel(), _lib.stream_ptr(gpu))
    assert L.mi_prefill_plan_pinned(src.data_ptr(), num_indices, qo, ip, idx, last, 0, 0, 16, 8, 2, 128, None, None, 0,
                                    *tail) == status
    torch.cuda.synchronize()
    if status == 0 and num_indices:
        assert dst[3, :5].tolist() == src[2:7].tolist()
    assert L.mi_decode_plan_pinned(src[1:].data_ptr(), num_indices, ip, idx, last, 0, 16, 8, 2, 128, None,
                                   *tail) == status
    torch.cuda.synchronize()
    if status == 0 and num_indices:
        assert dst[3, :5].tolist() == src[2:7].tolist()
