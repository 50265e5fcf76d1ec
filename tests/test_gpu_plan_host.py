"""GPU: plans whose CPU index tensors travel in the launch argument or pinned memory.

At the argument's limit of 800 values and one beyond it (the staged copy),
plan() must leave the same arrays on the device, the same token map and write
locations, and run() the same bits, as plan() over device tensors, which takes
neither path; also in graph mode, where the arrays are static buffers.
"""

import pytest
import torch

from gpu_helpers import custom_batch, log, random_cache, workspace
from mstar_amd import _lib
from mstar_amd.paged_attention import FlashInferDecodeWrapper, FlashInferPrefillWrapper

pytestmark = pytest.mark.gpu


def _lens(batch, values, fixed, ps):
    """Context lengths whose index arrays hold ``values`` values in all (``fixed`` beside the pages)."""
    pages = values - fixed
    per = pages // batch
    return [ps * per - (7 * i) % ps for i in range(batch - 1)] + [ps * (pages - per * (batch - 1)) - 3]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("batch", [1, 5, 200])
def test_decode_plan_host(gpu, batch, extra, graph):
    hq, hkv, d, ps = 8, 2, 128, 16
    log(f"decode plan host batch={batch} extra={extra} graph={graph}")
    lens = _lens(batch, _lib.PLAN_HOST_ARGS + extra, 2 * batch + 1, ps)
    qo, indptr, indices, last = custom_batch(lens, ps, 1000, 3)
    assert len(indptr) + len(indices) + len(last) == _lib.PLAN_HOST_ARGS + extra
    cache = random_cache(1000, ps, hkv, d, 5).to(gpu)
    q = torch.randn(batch, hq, d, device=gpu).to(torch.bfloat16)
    got = []
    for dev in ("cpu", gpu):
        fixed = {"batch_size": batch, "max_num_pages": 1000, "use_cuda_graph": True} if graph else {}
        w = FlashInferDecodeWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu, **fixed)
        w.plan(*(torch.as_tensor(x).to(dev) for x in (indptr, indices, last)))
        out = w.run(q, cache)
        got.append((out, w.kv_cache_locations, w._indptr, w._indices[: len(indices)], w._last))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert got[0][3].cpu().tolist() == indices.tolist()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("batch", [1, 40])
def test_prefill_plan_host(gpu, batch, extra, graph):
    hq, hkv, d, ps = 8, 2, 128, 16
    log(f"prefill plan host batch={batch} extra={extra} graph={graph}")
    lens = _lens(batch, _lib.PLAN_HOST_ARGS + extra, 3 * batch + 2, ps)
    new = [min(n, 1 + 37 * (i % 3)) for i, n in enumerate(lens)]  # short-query and tiled requests
    meta = custom_batch(lens, ps, 1000, 3, new_lens=new)
    assert sum(len(x) for x in meta) == _lib.PLAN_HOST_ARGS + extra
    cache = random_cache(1000, ps, hkv, d, 5).to(gpu)
    q = torch.randn(sum(new), hq, d, device=gpu).to(torch.bfloat16)
    got = []
    for dev in ("cpu", gpu):
        fixed = ({"batch_size": batch, "max_num_pages": 1000, "max_total_tokens": sum(new) + 5, "use_cuda_graph": True}
                 if graph else {})
        w = FlashInferPrefillWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu, **fixed)
        w.plan(*(torch.as_tensor(x).to(dev) for x in meta))
        out = w.run(q, cache)
        got.append((out, w.token_to_page, w.token_to_cache, w._qo, w._indptr, w._indices[: len(meta[2])], w._last))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_plan_host_leaves_the_caller_its_tensors(gpu):
    """The indices are read before plan() returns: a caller may overwrite them at once."""
    log("plan host: inputs overwritten after plan()")
    hq, hkv, d, ps = 8, 2, 128, 16
    qo, indptr, indices, last = custom_batch([100, 300], ps, 64, 3)
    parts = [torch.as_tensor(x).clone() for x in (indptr, indices, last)]
    w = FlashInferDecodeWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu)
    w.plan(*parts)
    for t in parts:
        t.fill_(-1)
    torch.cuda.synchronize()
    assert w._indices.cpu().tolist() == indices.tolist() and w._indptr.cpu().tolist() == indptr.tolist()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("batch,values", [(1, 801), (64, 5000), (1024, 16384), (1024, 16385), (1025, 16384)])
def test_decode_plan_pinned(gpu, batch, values, graph):
    """Index arrays in pinned memory up to its 16384 values and 1024 requests, the staged copy
    beyond, against device tensors; more plans in flight than the ring has rows."""
    hq, hkv, d, ps = 8, 2, 128, 16
    log(f"decode plan pinned batch={batch} values={values} graph={graph}")
    lens = _lens(batch, values, 2 * batch + 1, ps)
    qo, indptr, indices, last = custom_batch(lens, ps, 17000, 3)
    assert len(indptr) + len(indices) + len(last) == values
    cache = torch.randn(17000, 2, ps, hkv, d, device=gpu, dtype=torch.bfloat16)
    q = torch.randn(batch, hq, d, device=gpu).to(torch.bfloat16)
    got = []
    for dev, dtype in (("cpu", torch.int64), (gpu, torch.int32)):
        fixed = {"batch_size": batch, "max_num_pages": 17000, "use_cuda_graph": True} if graph else {}
        w = FlashInferDecodeWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu, **fixed)
        other = [torch.as_tensor(x).to(dev, dtype) for x in (indptr, indices[::-1].copy(), last)]
        parts = [torch.as_tensor(x).to(dev, dtype) for x in (indptr, indices, last)]
        for _ in range(2 * _lib.PinnedRing.SLOTS):
            w.plan(*other)
            w.plan(*parts)
        out = w.run(q, cache)
        got.append((out, w.kv_cache_locations, w._indptr, w._indices[: len(indices)], w._last))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert got[0][3].cpu().tolist() == indices.tolist()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("batch,values", [(1, 801), (40, 5000), (1024, 16384), (40, 16385), (1025, 16384)])
def test_prefill_plan_pinned(gpu, batch, values, graph):
    """The same for ragged plans, whose tiles, split-KV items and token map all come from the pinned rows."""
    hq, hkv, d, ps = 8, 2, 128, 16
    log(f"prefill plan pinned batch={batch} values={values} graph={graph}")
    lens = _lens(batch, values, 3 * batch + 2, ps)
    new = [min(n, 1 + 37 * (i % 3)) for i, n in enumerate(lens)]  # short-query and tiled requests
    qo, indptr, indices, last = custom_batch(lens, ps, 17000, 3, new_lens=new)
    assert len(qo) + len(indptr) + len(indices) + len(last) == values
    cache = torch.randn(17000, 2, ps, hkv, d, device=gpu, dtype=torch.bfloat16)
    q = torch.randn(sum(new), hq, d, device=gpu).to(torch.bfloat16)
    got = []
    for dev, dtype in (("cpu", torch.int64), (gpu, torch.int32)):
        fixed = ({"batch_size": batch, "max_num_pages": 17000, "max_total_tokens": sum(new) + 5, "use_cuda_graph": True}
                 if graph else {})
        w = FlashInferPrefillWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu, **fixed)
        other = [torch.as_tensor(x).to(dev, dtype) for x in (qo, indptr, indices[::-1].copy(), last)]
        parts = [torch.as_tensor(x).to(dev, dtype) for x in (qo, indptr, indices, last)]
        for _ in range(2 * _lib.PinnedRing.SLOTS):
            w.plan(*other)
            w.plan(*parts)
        out = w.run(q, cache)
        got.append((out, w.token_to_page, w.token_to_cache, w._qo, w._indptr, w._indices[: len(indices)], w._last))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert got[0][5].cpu().tolist() == indices.tolist()
