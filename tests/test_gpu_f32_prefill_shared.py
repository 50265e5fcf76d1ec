"""GPU parity of the fp32 prefill kernel that shares K and V within a workgroup.

It takes batches of at least LINE blocks of 64 rows per CU; the sizes here lie
just above that, with rows, keys and pages that end inside
a block, a key step and a page, requests the kernel does not serve, and more
keys than one request's rows can see.  The bar is the fp32 path's 2e-5
(``test_gpu_f32``): with |q|, |k| ~ sqrt(head_dim) a score of fp32 products
summed in any order is off by about sqrt(head_dim) 2^-24 |q||k| / sqrt(head_dim)
~ 1e-6, which a softmax over N(0, 1) values turns into as much in the output.
"""

import numpy as np
import pytest
import torch

from gpu_helpers import custom_batch, log, max_abs, random_cache, workspace
from mstar_amd.paged_attention import FlashInferPrefillWrapper
from test_gpu_f32 import F32, TOL_F32
from test_gpu_prefill import _run_prefill

pytestmark = pytest.mark.gpu

LINE = {256: 1.8, 128: 1.7, 64: 2.3}  # with and without a causal mask


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv,d,ps,kv,new", [
    (16, 2, 256, 16, [700, 33, 300, 1, 17, 800, 500], [600, 33, 199, 1, 0, 700, 450]),
    (28, 4, 128, 48, [500, 449, 31, 300, 400], [251, 240, 1, 300, 290]),
    (32, 4, 64, 128, [1100, 65, 129, 600], [640, 64, 129, 500]),
])
def test_f32_shared_prefill_shapes(gpu, causal, hq, hkv, d, ps, kv, new):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert sum(new) * hq / 64 >= LINE[d] * cus, "below the kernel's range"
    out, ref = _run_prefill(gpu, hq, hkv, d, ps, kv, new, causal, seed=d + ps, dtype=F32)
    err = max_abs(out, ref)
    log(f"f32 shared prefill causal={causal} {hq}/{hkv}/{d} ps={ps}: max_abs={err:.3e}")
    assert err < TOL_F32


@pytest.mark.parametrize("hq,hkv,d", [(16, 2, 256), (28, 4, 128), (32, 4, 64)])
def test_f32_shared_prefill_non_finite(gpu, hq, hkv, d):
    """Slots past kv_len may hold anything; a NaN key reaches the rows that see it and no others."""
    log(f"f32 shared prefill with NaN tail and key d={d}")
    ps, kv, new, at = 32, 2101, 2000, 2000
    qo, indptr, indices, last = custom_batch([kv], ps, 70, 3, new_lens=[new])
    cache = random_cache(70, ps, hkv, d, 5, F32).to(gpu)
    q = torch.randn(new, hq, d, generator=torch.Generator().manual_seed(6)).to(gpu)
    w = FlashInferPrefillWrapper(workspace(gpu), hq, hkv, d, ps, device=gpu)
    w.plan(*(torch.as_tensor(x) for x in (qo, indptr, indices, last)), causal=True, dtype=F32)
    clean = w.run(q, cache)
    cache[int(indices[-1]), :, int(last[0]):] = float("nan")
    assert torch.equal(w.run(q, cache), clean)
    cache[int(indices[at // ps]), 0, at % ps] = float("nan")
    out = w.run(q, cache)
    first = at - (kv - new)
    assert torch.equal(out[:first], clean[:first]) and bool(out[first:].isnan().all())
    assert np.isfinite(clean.cpu().numpy()).all()
