"""GPU: arguments that the plan calls over host and pinned index arrays refuse before they launch."""

import ctypes

import pytest
import torch

from gpu_helpers import custom_batch, log, workspace
from mstar_amd import _lib
from mstar_amd.paged_attention import FlashInferDecodeWrapper, FlashInferPrefillWrapper

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


@pytest.mark.parametrize("kind", ["decode", "prefill"])
@pytest.mark.parametrize("pages", [40, 2000])  # in the launch argument; in pinned memory
def test_page_lists_longer_than_the_indices(gpu, kind, pages):
    """A graph-mode plan whose kv_indptr ends past the given indices takes the rest
    from the static buffer, whichever way the arrays come in."""
    log(f"{kind} plan: page lists end 5 past {pages} indices")
    qo, indptr, indices, last = custom_batch([16 * (pages // 2), 16 * (pages - pages // 2) + 75], 16, pages + 10, 3,
                                             new_lens=[1, 1] if kind == "decode" else [20, 90])
    assert indptr[-1] == pages + 5
    meta = [torch.as_tensor(x) for x in (qo, indptr, indices[:pages], last)]
    got = []
    for dev in ("cpu", gpu):
        fixed = {"batch_size": 2, "max_num_pages": pages + 10, "use_cuda_graph": True, "device": gpu}
        if kind == "decode":
            w = FlashInferDecodeWrapper(workspace(gpu), 8, 2, 128, 16, **fixed)
        else:
            w = FlashInferPrefillWrapper(workspace(gpu), 8, 2, 128, 16, max_total_tokens=110, **fixed)
        w._paged_kv_indices_buf.copy_(torch.arange(pages + 10))
        w.plan(*(t.to(dev) for t in meta[kind == "decode":]))
        got.append([w._indices, w.kv_cache_locations] if kind == "decode" else
                   [w._indices, w.token_to_page, w.token_to_cache])
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_host_plans_refuse_page_lists_past_the_argument(gpu):
    log("host plans: kv_indptr ends past num_indices")
    L, ws = _lib.lib(), workspace(gpu, 64 << 20)
    i32 = ctypes.c_int32 * 2
    indptr, qo, idx, last = i32(0, 3), i32(0, 1), i32(4, 5), i32(1, 0)
    dst = [ctypes.c_void_p(t.data_ptr()) for t in torch.zeros(4, 16, dtype=torch.int32, device=gpu)]
    tail = (ctypes.c_void_p(ws.data_ptr()), ws.numel(), _lib.stream_ptr(gpu))
    assert L.mi_decode_plan_host(indptr, idx, last, 2, *dst[1:], 1, 16, 8, 2, 128, None, *tail) == INVALID
    assert L.mi_prefill_plan_host(qo, indptr, idx, last, 2, *dst, 1, 1, 16, 8, 2, 128, None, None, 0, *tail) == INVALID
