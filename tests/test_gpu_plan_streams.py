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
    return ev


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
