"""GPU: the fp32 prefill kernel that shares K and V, over values that show what its sums meet.

The sizes lie above the line from which it takes a batch (1.4-2.3 blocks of 64
rows per CU).
"""

import numpy as np
import pytest
import torch

from gpu_helpers import custom_batch, log, random_cache, workspace
from mstar_amd.paged_attention import FlashInferPrefillWrapper

pytestmark = pytest.mark.gpu

F32 = torch.float32
HEADS = [(16, 2, 256), (28, 4, 128), (32, 4, 64)]


def _wrapper(gpu, heads, ps, meta, causal):
    w = FlashInferPrefillWrapper(workspace(gpu), *heads, ps, device=gpu)
    w.plan(*(torch.as_tensor(x) for x in meta), causal=causal, dtype=F32)
    return w


@pytest.mark.parametrize("heads", HEADS)
@pytest.mark.parametrize("at", [205, 1403, 2012])  # among the new tokens' positions 101..2100
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_v_reaches_its_16_row_blocks_only(gpu, heads, at, value):
    """A masked key's V meets a probability of zero, which NaN and Inf survive: within
    the 16-key group of a 16-row block's last key, and no further."""
    hq, hkv, d = heads
    log(f"f32 shared prefill, V {value} at {at}, {heads}")
    ps, kv, new = 16, 2101, 2000
    meta = custom_batch([kv], ps, 140, 3, new_lens=[new])
    cache = random_cache(140, ps, hkv, d, 5, F32).to(gpu)
    q = torch.randn(new, hq, d, generator=torch.Generator().manual_seed(6)).to(gpu)
    w = _wrapper(gpu, heads, ps, meta, True)
    clean = w.run(q, cache)
    cache[int(meta[2][at // ps]), 1, at % ps] = value
    out = w.run(q, cache)
    g = hq // hkv
    row = np.arange(new * g)                                 # (token, head of the group), token-major
    last_tok = np.minimum(row // 16 * 16 + 15, new * g - 1) // g  # of the row's 16-row block
    met = at < -(-(kv - new + last_tok + 1) // 16) * 16
    met = torch.from_numpy(met.reshape(new, g)).to(gpu)
    for h in range(hkv):
        rows, ref = out[:, h * g:(h + 1) * g], clean[:, h * g:(h + 1) * g]
        assert torch.equal(rows[~met], ref[~met])
        first = at - (kv - new)
        assert not bool(rows[first:].isfinite().any())


def _attention64(q, k, v, first, scale):
    """[tokens, heads, dim] attention in 64 bits; query i sees the keys up to first + i (all: first None)."""
    g = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for h in range(q.shape[1]):
        s = (q[:, h].double() @ k[:, h // g].double().t().contiguous()) * scale
        if first is not None:
            at = torch.arange(q.shape[0], device=q.device)[:, None] + first
            s.masked_fill_(torch.arange(k.shape[0], device=q.device)[None] > at, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ v[:, h // g].double()
    return out


@pytest.mark.parametrize("heads", HEADS)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kv,new", [(2600, 2000), (2000, 2000)])
def test_no_further_from_64_bits_than_the_16_row_kernel(gpu, heads, causal, kv, new):
    """The same queries in batches too small for the kernel run through
    attend_f32_kernel, whose sums are quarters of the keys long; a row's error is
    random, so over a million outputs the two 2-norms compare to well under 5 %."""
    hq, hkv, d = heads
    ps = 16
    meta = custom_batch([kv], ps, 170, 3, new_lens=[new])
    cache = random_cache(170, ps, hkv, d, 5, F32).to(gpu)
    q = torch.randn(new, hq, d, generator=torch.Generator().manual_seed(6)).to(gpu)
    rows = cache[torch.as_tensor(meta[2]).long().to(gpu)].transpose(0, 1).reshape(2, -1, hkv, d)[:, :kv]
    ref = _attention64(q, rows[0], rows[1], kv - new if causal else None, d ** -0.5)
    shared = _wrapper(gpu, heads, ps, meta, causal).run(q, cache)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    part = int(0.7 * cus * 64 / hq)  # query tokens of a batch below the line
    split = torch.empty_like(shared)
    for a in range(0, new, part):
        b = min(new, a + part)
        seen = kv - new + b if causal else kv
        m = custom_batch([seen], ps, 170, 3, new_lens=[b - a])  # the same pages
        split[a:b] = _wrapper(gpu, heads, ps, m, causal).run(q[a:b], cache)
    err = [float((o.double() - ref).norm() / ref.norm()) for o in (shared, split)]
    log(f"f32 prefill {heads} causal={causal} kv={kv}: error shared {err[0]:.3e}, 16-row {err[1]:.3e}")
    assert err[0] <= 1.05 * err[1]


@pytest.mark.parametrize("heads", HEADS)
def test_large_v_overflows_no_sooner_than_its_mean(gpu, heads):
    """Probabilities relative to the row's max sum to at most the number of keys, so V
    of 2^127 / keys keeps every partial sum finite, also where later keys score higher."""
    hq, hkv, d = heads
    log(f"f32 prefill, large V {heads}")
    ps, kv, new = 16, 2048, 2000
    meta = custom_batch([kv], ps, 140, 3, new_lens=[new])
    cache = random_cache(140, ps, hkv, d, 5, F32).to(gpu)
    pages = torch.as_tensor(meta[2]).long().to(gpu)
    cache[pages, 1] = 2.0 ** 127 / kv
    unit = torch.nn.functional.normalize(torch.randn(hkv, d, generator=torch.Generator().manual_seed(8)), dim=-1).to(gpu)
    # scores rise with the key's position: by 5 (in exp2's terms 7.2) from first to last
    rise = torch.linspace(0, 5, kv, device=gpu).view(-1, ps, 1, 1)
    cache[pages, 0] = rise * unit * d ** 0.5
    q = unit.repeat_interleave(hq // hkv, 0).expand(new, -1, -1).contiguous()
    out = _wrapper(gpu, heads, ps, meta, False).run(q, cache)
    assert bool(out.isfinite().all())
    assert float((out / (2.0 ** 127 / kv) - 1).abs().max()) < 1e-5


@pytest.mark.parametrize("heads", [(8, 1, 256), (16, 4, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_captured_layer_takes_the_kernel_of_each_plan(gpu, heads, causal):
    """A graph of up to 8192 tokens replayed over plans on both sides of the line: the bits
    are those of a plain call, which knows its rows, away from the line (where the two lie
    apart for captured and plain calls), and every row is written at each size."""
    hq, hkv, d = heads
    log(f"captured f32 prefill {heads} causal={causal}")
    ps, most, pool = 16, 8192, 600
    cache = random_cache(pool, ps, hkv, d, 5, F32).to(gpu)
    q = torch.randn(most, hq, d, generator=torch.Generator().manual_seed(6)).to(gpu)
    g = FlashInferPrefillWrapper(workspace(gpu), *heads, ps, batch_size=4, max_total_tokens=most, max_num_pages=pool,
                                 device=gpu, use_cuda_graph=True)

    def meta(tokens):
        new = [min(2048, max(0, tokens - 2048 * i)) for i in range(4)]
        return [torch.as_tensor(x) for x in custom_batch(new, ps, pool, 3, new_lens=new)]

    out = torch.empty_like(q)
    g.plan(*meta(most), causal=causal, dtype=F32)
    g.run(q, cache, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.run(q, cache, out=out)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_cu = 64 * cus / hq  # tokens of one block a CU
    for tokens in (20, 700, int(1.2 * per_cu), int(3 * per_cu), most):
        tokens = min(tokens, most)
        g.plan(*meta(tokens), causal=causal, dtype=F32)
        out.fill_(float("nan"))
        graph.replay()
        plain = _wrapper(gpu, heads, ps, meta(tokens), causal).run(q[:tokens], cache)
        assert bool(out[:tokens].isfinite().all())
        if tokens in (20, 700, most) and not 2.2 <= tokens / per_cu <= 4.1:
            assert torch.equal(out[:tokens], plain), tokens
        else:
            assert float((out[:tokens] - plain).abs().max()) < 2e-5, tokens
