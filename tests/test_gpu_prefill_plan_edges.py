"""GPU: ragged plans at the edges of what the plan's tables hold."""

import pytest
import torch

from gpu_helpers import custom_batch, log
from mstar_amd import _lib
from mstar_amd.paged_attention import FlashInferPrefillWrapper

pytestmark = pytest.mark.gpu

PART_O = 4 * 256 * 128  # bytes of one partial's output at head_dim 128


def _hdr(ws):
    return ws[:32].cpu().view(torch.int32).tolist()


@pytest.mark.parametrize("stated", [16, 17, 32])
def test_tiles_past_the_stated_tokens_are_not_priced(gpu, stated):
    """Device index tensors with more query tokens than the caller states: the
    tiles beyond the list are left out of the costs as well, so the cut of the
    listed ones keeps to the workspace's room for partials (about 16 here; priced
    with the last listed tile carrying the others' 1600-1700 key steps, it had 90
    to 106)."""
    log(f"prefill plan: 320 query tokens, {stated} stated")
    hq, hkv, d, ps, room = 16, 1, 128, 16, 16
    meta = [torch.as_tensor(x).to(gpu) for x in custom_batch([3200], ps, 210, 3, new_lens=[320])]
    size = _lib.lib().mi_prefill_workspace_bytes(1, stated, hq, hkv, d) - (768 - room) * PART_O
    guard = torch.full((size + (4 << 20),), 0x5A, dtype=torch.uint8, device=gpu)
    w = FlashInferPrefillWrapper(guard[:size], hq, hkv, d, ps, device=gpu)
    w.plan_device(*meta, total_tokens=stated)
    tiles, _, pieces, split = _hdr(guard)[:4]
    log(f"  tiles={tiles} pieces={pieces} split tiles={split}")
    assert tiles == -(-stated * hq // 256) + 1
    assert tiles <= pieces <= tiles + 2 * room and split <= tiles
    assert bool((guard[size:] == 0x5A).all())
