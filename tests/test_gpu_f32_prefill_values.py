"""GPU: the fp32 prefill kernel that shares K and V, over values that show what its sums meet.

The sizes lie above the line from which it takes a batch (0.8 blocks of 64 rows
per CU, 1.5 at head_dim 64).
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
@pytest.mark.parametrize("at", [205, 703, 912])  # among the new tokens' positions 101..1000
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_v_reaches_its_16_row_blocks_only(gpu, heads, at, value):
    """A masked key's V meets a probability of zero, which NaN and Inf survive: within
    the 16-key group of a 16-row block's last key, and no further."""
    hq, hkv, d = heads
    log(f"f32 shared prefill, V {value} at {at}, {heads}")
    ps, kv, new = 16, 1001, 900
    meta = custom_batch([kv], ps, 70, 3, new_lens=[new])
    cache = random_cache(70, ps, hkv, d, 5, F32).to(gpu)
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
