"""GPU: plans and runs of several streams beside each other."""

import time

import pytest
import torch

from gpu_helpers import custom_batch, log, random_cache, workspace
from mstar_amd import _lib
from mstar_amd.paged_attention import FlashInferDecodeWrapper, FlashInferPrefillWrapper

pytestmark = pytest.mark.gpu


def _busy(gpu, seconds):
    """Keeps the current stream busy for about so long; an event behind it."""
    per = 1 << 20
    torch.cuda.synchronize()
    t = time.perf_counter()
    torch.cuda._sleep(per)
    torch.cuda.synchronize()
    took = time.perf_counter() - t
    torch.cuda._sleep(int(per * seconds / took))
    ev = torch.cuda.Event()
    ev.record()
    return ev  # of the sleep: what is queued behind it has not begun before


def test_a_pinned_plan_waits_for_no_other_stream(gpu):
    """As many plans as a ring has rows are queued on a busy stream: the call on an idle one returns
    before they are done (its launch may still share a hardware queue with them)."""
    log("pinned plans of two streams")
    hq, hkv, d, ps = 8, 2, 128, 16
    meta = [torch.as_tensor(x) for x in custom_batch([16 * 1000], ps, 1001, 3)[1:]]  # beyond the launch argument
    ws = [FlashInferDecodeWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu) for _ in range(2)]
    a, b = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    for s, w in zip((a, b), ws):  # the rings exist
        with torch.cuda.stream(s):
            w.plan(*meta)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        done = _busy(gpu, 0.4)
        for _ in range(_lib.PinnedRing.SLOTS):
            ws[0].plan(*meta)
    with torch.cuda.stream(b):
        ws[1].plan(*meta)
    assert not done.query(), "the call on the idle stream waited for the busy one"
    torch.cuda.synchronize()
    assert ws[1]._indices.cpu().tolist() == meta[1].tolist()


def test_streams_beyond_the_last_ring_share_one(gpu, monkeypatch):
    log("pinned rings: bounded")
    monkeypatch.setattr(_lib, "_rings", {})
    monkeypatch.setattr(_lib, "MAX_PINNED_RINGS", 2)
    rings = [_lib.pinned_ring(gpu, s) for s in (11, 12, 13, 14, 11, 13)]
    assert rings[0] is rings[4] and rings[0] is not rings[1]
    assert rings[2] is rings[3] is rings[5] and rings[2] not in rings[:2]


@pytest.mark.parametrize("kind", ["decode", "prefill"])
@pytest.mark.parametrize("pages", [40, 2000])  # indices in the launch argument; in pinned memory
@pytest.mark.parametrize("part", ["run", "append"])
def test_plan_arrays_outlive_a_reader_on_another_stream(gpu, kind, pages, part):
    """Planned on one stream and read on another that is busy, then dropped: the plan's memory
    is not handed out again while the reader is queued."""
    log(f"{kind} plan of {pages} pages, {part} on another stream")
    hq, hkv, d, ps = 8, 2, 128, 16
    new = [1] if kind == "decode" else [60]
    meta = [torch.as_tensor(x) for x in custom_batch([16 * pages], ps, pages, 3, new_lens=new)]
    cache = torch.zeros(pages, 2, ps, hkv, d, dtype=torch.bfloat16, device=gpu)
    q, k = (torch.zeros(new[0], h, d, dtype=torch.bfloat16, device=gpu) for h in (hq, hkv))
    ws, out = workspace(gpu), torch.empty_like(q)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    cls = FlashInferDecodeWrapper if kind == "decode" else FlashInferPrefillWrapper
    w = cls(ws, hq, hkv, d, ps, device=gpu)
    w.plan(*meta[kind == "decode":])
    mine = [(w._indices.data_ptr(), 4 * pages)] if part == "run" else [
        (t.data_ptr(), t.numel() * 8) for t in ([w.kv_cache_locations] if kind == "decode" else [w.token_to_page])]
    other = torch.cuda.Stream(gpu)
    other.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(other):
        done = _busy(gpu, 0.3)
        w.run(q, cache, out=out) if part == "run" else w.set_kv_cache(cache, k, k)
    del w
    taken = [torch.empty(n // 4, dtype=torch.int32, device=gpu) for n in (mine[0][1], 4 * pages + 12, 16, 480)
             for _ in range(40)]
    overlap = [t for t in taken for a, n in mine if t.data_ptr() < a + n and a < t.data_ptr() + 4 * t.numel()]
    assert not done.query(), "the reader is no longer queued: nothing was tested"
    assert not overlap
    torch.cuda.synchronize()
