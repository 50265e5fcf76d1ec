"""GPU: ragged plans at the edges of what the plan's tables hold."""

import pytest
import torch

import test_gpu_prefill_split as split
from gpu_helpers import custom_batch, log, random_cache
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
    listed ones keeps to the workspace's room for partials (24 here; priced
    with the last listed tile carrying the others' 1600-1700 key steps, it had 90
    to 106)."""
    log(f"prefill plan: 320 query tokens, {stated} stated")
    hq, hkv, d, ps, room = 16, 1, 128, 16, 24
    meta = [torch.as_tensor(x).to(gpu) for x in custom_batch([3200], ps, 210, 3, new_lens=[320])]
    size = _lib.lib().mi_prefill_workspace_bytes(1, stated, hq, hkv, d) - (768 - room) * PART_O
    guard = torch.full((size + (4 << 20),), 0x5A, dtype=torch.uint8, device=gpu)
    w = FlashInferPrefillWrapper(guard[:size], hq, hkv, d, ps, device=gpu)
    w.plan_device(*meta, total_tokens=stated)
    tiles, _, pieces, split = _hdr(guard)[:4]
    log(f"  tiles={tiles} pieces={pieces} split tiles={split}")
    assert tiles == -(-stated * hq // 256) + 1
    assert tiles <= pieces <= tiles + room and split <= tiles
    assert bool((guard[size:] == 0x5A).all())


@pytest.mark.parametrize("heads,fp8", [((8, 2, 128), False), ((8, 2, 128), True), ((16, 4, 64), False),
                                       ((8, 1, 256), False), ((8, 1, 256), True)])
def test_runs_that_state_another_workspace_size(gpu, heads, fp8):
    """A plan and its runs given different sizes of one workspace, each of which
    holds the plan: tiles are computed whole wherever the run's size has no room
    for the plan's partials, and the bits are those of equal sizes."""
    hq, hkv, d = heads
    log(f"workspace sizes of plan and run {heads} fp8={fp8}")
    ps, kv, new = 16, [3000, 700, 900], [90, 50, 1]  # cut tiles, and a short-query request
    meta = custom_batch(kv, ps, 300, 3, new_lens=new)
    cache = random_cache(300, ps, hkv, d, 5).to(gpu)
    scales = (None, None)
    if fp8:
        cache, scales = cache.to(torch.float8_e4m3fn), (torch.full((hkv,), 0.5, device=gpu),) * 2
    q = torch.randn(sum(new), hq, d, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).to(gpu)
    full = _lib.lib().mi_prefill_workspace_bytes(len(kv), sum(new), hq, hkv, d)
    part = 4 * d * (128 if d == 256 else 256)
    roomy, few, none = full, full - (768 - 2 * hkv) * part, full - 768 * part
    ws = torch.empty(full, dtype=torch.uint8, device=gpu)

    def go(planned, ran, serial):
        w = FlashInferPrefillWrapper(ws[:planned], hq, hkv, d, ps, device=gpu)
        w.plan(*(torch.as_tensor(x) for x in meta))
        cut = _hdr(ws)[3] > 0
        w._workspace, w._serial = ws[:ran], serial
        out = torch.full_like(q, float("nan"))
        w.run(q, cache, *scales, out=out)
        again = w.run(q, cache, *scales)
        assert torch.equal(out, again), "a plan's second run differs"
        return out, cut

    whole, cut = go(none, none, True)
    assert not cut
    cut_out, cut = go(roomy, roomy, True)
    assert cut and bool(cut_out.isfinite().all())
    for serial in (True, False):
        assert torch.equal(go(roomy, roomy, serial)[0], cut_out)
        for planned, ran in ((roomy, few), (roomy, none), (none, roomy), (none, few)):
            out, cut = go(planned, ran, serial)
            assert cut == (planned == roomy)
            assert torch.equal(out, whole), (planned, ran, serial)
        small, _ = go(few, few, serial)
        assert torch.equal(go(few, roomy, serial)[0], small)


@pytest.mark.parametrize("heads,ps,kv_lens,new", [
    ((6, 3, 128), 16, [2500, 300], [150, 20]),    # 3, 6, 10 kv-heads: (piece, head) pairs in turn
    ((24, 6, 64), 16, [2000], [90]),
    ((10, 10, 256), 16, [900], [70]),
    ((16, 16, 128), 32, [1700, 500], [60, 1]),    # 16 kv-heads: two a queue
])
def test_split_tiles_of_other_head_counts(gpu, heads, ps, kv_lens, new):
    split.test_split_tiles_match_unsplit_and_fp32(gpu, heads, ps, kv_lens, new, True, torch.bfloat16, False)


@pytest.mark.parametrize("heads", [(32, 4, 128), (32, 4, 64)])
def test_whole_tiles_are_dealt(gpu, heads):
    """With room for few partials, tiles of uneven requests are dealt uncut where that is
    the better schedule; each tile's arithmetic, so every bit, is that of the local queues."""
    hq, hkv, d = heads
    log(f"whole tiles dealt {heads}")
    ps, kv, new = 16, [2500, 9000, 1200, 5000], [500, 2000, 600, 1200]
    meta = custom_batch(kv, ps, 1110, 3, new_lens=new)
    cache = torch.randn(1110, 2, ps, hkv, d, device=gpu, dtype=torch.bfloat16)
    q = torch.randn(sum(new), hq, d, device=gpu, dtype=torch.bfloat16)
    full = _lib.lib().mi_prefill_workspace_bytes(len(kv), sum(new), hq, hkv, d)
    outs = []
    for room in (0, 2 * hkv):
        ws = torch.empty(full - (768 - room) * 4 * 256 * d, dtype=torch.uint8, device=gpu)
        w = FlashInferPrefillWrapper(ws, hq, hkv, d, ps, device=gpu)
        w.plan(*(torch.as_tensor(x) for x in meta))
        tiles, units, pieces, cut = _hdr(ws)[:4]
        log(f"  room for {room} partials: tiles={tiles} pieces={pieces} split tiles={cut}")
        assert cut == 0 and pieces == (tiles if room else 0) and units == tiles * hkv
        outs.append(w.run(q, cache))
        assert torch.equal(outs[-1], w.run(q, cache))
    assert torch.equal(*outs)


@pytest.mark.parametrize("at", [0, 700, 1090])
def test_cut_plans_of_more_than_a_thread_per_tile(gpu, at):
    """More than 1024 requests and tiles: two windows of each, and cut tiles on either side.

    The bound is that of the split tests: with probabilities and outputs rounded to bf16,
    |out - ref| <= 2^-8 (sum_i p_i |v_i| + 2 |ref|) + fp32 rounding."""
    hq, hkv, d, ps = 8, 1, 256, 16
    log(f"cut plan of 1102 requests, a long one at {at}")
    kv, new = [20] * 1102, [20] * 1102
    kv[at], new[at] = 24000, 320
    kv[1101], new[1101] = 20000, 40
    pool = int(sum(-(-n // ps) for n in kv))
    meta = custom_batch(kv, ps, pool, 3, new_lens=new)
    cache = torch.randn(pool, 2, ps, hkv, d, device=gpu, dtype=torch.bfloat16)
    q = torch.randn(sum(new), hq, d, device=gpu, dtype=torch.bfloat16)
    ws = torch.empty(512 << 20, dtype=torch.uint8, device=gpu)
    w = FlashInferPrefillWrapper(ws, hq, hkv, d, ps, device=gpu)
    w.plan_device(*(torch.as_tensor(x).to(gpu) for x in meta), total_tokens=sum(new))
    tiles, _, pieces, cut = _hdr(ws)[:4]
    log(f"  tiles={tiles} pieces={pieces} split tiles={cut}")
    assert tiles > 1024 and pieces > tiles and cut > 0
    out = w.run(q, cache)
    qo, indptr, indices, _ = meta
    worst = 0.0
    for r in sorted({0, 1, 699, 700, 701, 1022, 1023, 1024, 1025, 1089, 1090, 1100, 1101}):
        rows = cache[torch.as_tensor(indices[indptr[r]:indptr[r + 1]]).long().to(gpu)]
        k, v = rows.transpose(0, 1).reshape(2, -1, d)[:, :kv[r]].double()
        part = q[qo[r]:qo[r + 1]].double()
        s = part @ k.t().contiguous() * d ** -0.5
        seen = torch.arange(kv[r], device=gpu) <= torch.arange(kv[r] - new[r], kv[r], device=gpu)[:, None, None]
        p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
        ref, mag = p @ v, p @ v.abs()
        bound = 2.0 ** -8 * (mag + 2 * ref.abs()) + 1e-4
        worst = max(worst, float(((out[qo[r]:qo[r + 1]].double() - ref).abs() / bound).max()))
    log(f"  error/bound={worst:.2f}")
    assert worst <= 1.0
