"""GPU parity: prefill tiles cut into key pieces (few tiles on many CUs) and their merge.

Each problem runs with a workspace that has room for partials, where the plan
must cut, and with one that has none, where it must not; both are held to the
elementwise bound of the arithmetic.  With probabilities rounded to the
16-bit type (relative error u = half a unit in the last of its 8 or 11 bits:
2^-8 for bf16, 2^-11 for fp16) and the output rounded once more,
    |out - ref| <= u * (sum_i p_i |v_i| + 2 |ref|) + fp32 rounding,
the first term from attention over |V|; the row sum adds the same rounded
probabilities.
"""

import numpy as np
import pytest
import torch

from gpu_helpers import A, P, custom_batch, log, random_cache, workspace
from mstar_amd.paged_attention import FlashInferPrefillWrapper

pytestmark = pytest.mark.gpu

ROOMY, TIGHT = 256 << 20, 4 << 20


def _hdr(ws):
    return ws[:32].cpu().view(torch.int32).tolist()


def _run(gpu, ws_bytes, heads, ps, meta, causal, dtype, cache, q, scales):
    w = FlashInferPrefillWrapper(workspace(gpu, ws_bytes), *heads, ps, device=gpu)
    w.plan(*(torch.as_tensor(x) for x in meta), causal=causal, dtype=dtype)
    out = w.run(q.to(gpu), cache, *scales)
    again = w.run(q.to(gpu), cache, *scales)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), again.view(torch.int16)), "a plan's second run differs (queues not reset)"
    return out, _hdr(w._workspace)


CASES = [
    # heads, page size, kv lengths, new tokens, causal, dtype, fp8
    ((28, 4, 128), 16, [4608], [512], True, torch.bfloat16, False),          # 14 tiles x 4 heads
    ((32, 4, 128), 32, [1025, 3000, 64], [33, 100, 64], True, torch.bfloat16, False),
    ((8, 1, 256), 16, [850, 1001], [50, 50], False, torch.bfloat16, False),  # last tile: one row group in use
    ((8, 1, 256), 64, [2000, 40, 700], [130, 40, 3], True, torch.float16, False),
    ((16, 2, 256), 16, [1500], [77], True, torch.bfloat16, True),
    ((16, 4, 64), 16, [3000, 500], [90, 1], True, torch.bfloat16, False),    # a short-query request beside the pieces
    ((8, 2, 128), 128, [5000], [300], False, torch.float16, True),
    ((8, 8, 128), 48, [257, 2050], [257, 17], True, torch.bfloat16, False),  # piece ends inside the causal edge
    ((28, 4, 128), 16, [36000], [40], True, torch.bfloat16, False),          # unsplit: two chunks of staged tiles
]


@pytest.mark.parametrize("heads,ps,kv_lens,new,causal,dtype,fp8", CASES)
def test_split_tiles_match_unsplit_and_fp32(gpu, heads, ps, kv_lens, new, causal, dtype, fp8):
    hq, hkv, d = heads
    log(f"split prefill {heads} ps={ps} kv={kv_lens} new={new} causal={causal} {dtype} fp8={fp8}")
    meta = custom_batch(kv_lens, ps, int(sum(-(-np.array(kv_lens) // ps))) + 4, 3, new_lens=new)
    qo, indptr, indices, last = meta
    pool = int(indices.max()) + 1
    src = random_cache(pool, ps, hkv, d, 5, torch.float32)
    q = torch.randn(int(qo[-1]), hq, d, generator=torch.Generator().manual_seed(6)).to(dtype)
    ks = vs = None
    if fp8:
        ks, vs = (A.head_scales(src[:, j].reshape(-1, hkv, d)) for j in (0, 1))
        cache = torch.empty(src.shape, dtype=torch.float8_e4m3fn)
        for j, s in ((0, ks), (1, vs)):
            cache[:, j] = A.quantize_e4m3(src[:, j].reshape(-1, hkv, d), s).view(pool, ps, hkv, d)
    else:
        cache = src.to(dtype)
    absv = cache.clone()
    raw = absv.view(torch.uint8) if fp8 else absv
    raw[:, 1] = raw[:, 1] & 0x7F if fp8 else raw[:, 1].abs()
    ref, ref_abs = (A.paged_attention(q, c, qo, indptr, indices, last, causal=causal, k_scale=ks, v_scale=vs)
                    for c in (cache, absv))
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = u * (ref_abs + 2 * ref.abs()) + 1e-4
    scales = (None, None) if ks is None else (ks.to(gpu), vs.to(gpu))
    for ws_bytes in (ROOMY, TIGHT):
        out, hdr = _run(gpu, ws_bytes, heads, ps, meta, causal, dtype, cache.to(gpu), q, scales)
        over = ((out.float().cpu() - ref).abs() / bound).max().item()
        log(f"  tiles={hdr[0]} pieces={hdr[2]} split tiles={hdr[3]} error/bound={over:.2f}")
        assert (hdr[2] > hdr[0]) == (ws_bytes == ROOMY)
        assert over <= 1.0


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (8, 1, 256)])
def test_split_tiles_keep_non_finite_rows(gpu, hq, hkv, d):
    """A NaN key in one piece: the rows that see it are NaN, the others as without it."""
    log(f"split prefill with a NaN key d={d}")
    ps, kv, new, at = 16, 2000, 64, 1960  # seen by the queries of positions >= 1960 only
    meta = custom_batch([kv], ps, 130, 3, new_lens=[new])
    cache = random_cache(130, ps, hkv, d, 5).to(gpu)
    q = torch.randn(new, hq, d, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16)
    clean, hdr = _run(gpu, ROOMY, (hq, hkv, d), ps, meta, True, torch.bfloat16, cache, q, (None, None))
    assert hdr[2] > hdr[0]
    cache[int(meta[2][at // ps]), 0, at % ps] = float("nan")
    out, _ = _run(gpu, ROOMY, (hq, hkv, d), ps, meta, True, torch.bfloat16, cache, q, (None, None))
    first = at - (kv - new)
    assert torch.equal(out[:first], clean[:first]) and bool(out[first:].isnan().all())


@pytest.mark.parametrize("heads,dtype,fp8,short,long", [
    ((28, 4, 128), torch.bfloat16, False, [20000, 40, 9000], [(3000, 100)]),
    ((28, 4, 128), torch.float16, True, [20000], [(3000, 33), (40, 40)]),     # one tile cut, one whole
    ((8, 1, 256), torch.bfloat16, False, [9000, 1], [(850, 50), (1001, 3)]),  # 24 rows: the smallest tile
    ((16, 2, 256), torch.bfloat16, True, [5000], [(1500, 77)]),
    ((16, 4, 64), torch.float16, False, [9000, 300], [(3000, 90)]),
    ((16, 4, 64), torch.bfloat16, True, [16], [(16, 16)]),                    # nothing to merge on either side
])
def test_one_merge_launch_for_both_parts(gpu, heads, dtype, fp8, short, long):
    """Both parts in one call merge in one launch: the rows' arithmetic is that of
    a merge launch each (the two-stream route), so the results are equal bit for bit."""
    hq, hkv, d = heads
    log(f"one merge launch {heads} {dtype} fp8={fp8} short={short} long={long}")
    ps, kv_lens = 16, [n for n, _ in long] + short
    meta = custom_batch(kv_lens, ps, int(sum(-(-np.array(kv_lens) // ps))) + 4, 3,
                        new_lens=[n for _, n in long] + [1] * len(short))
    pool = int(meta[2].max()) + 1
    cache = random_cache(pool, ps, hkv, d, 5).to(gpu)
    scales = (None, None)
    if fp8:
        cache, scales = cache.to(torch.float8_e4m3fn), (torch.full((hkv,), 0.5, device=gpu),) * 2
    elif cache.dtype != dtype:
        cache = cache.to(dtype)
    q = torch.randn(int(meta[0][-1]), hq, d, generator=torch.Generator().manual_seed(6)).to(dtype).to(gpu)
    w = FlashInferPrefillWrapper(workspace(gpu, ROOMY), *heads, ps, device=gpu)
    w.plan(*(torch.as_tensor(x) for x in meta), causal=True, dtype=dtype)
    outs = []
    for serial in (True, False):
        w._serial = serial
        out = torch.full_like(q, float("nan"))
        outs.append(w.run(q, cache, *scales, out=out))
        torch.cuda.synchronize()
    assert bool(outs[0].isfinite().all())
    assert torch.equal(outs[0], outs[1])
    assert (_hdr(w._workspace)[2] > _hdr(w._workspace)[0]) == (max(n for n, _ in long) > 16)
