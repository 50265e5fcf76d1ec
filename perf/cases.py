"""Workloads of the paged-attention path, as a program that serves a model issues them.

A case is one pass: plan the step's ragged batch, then for each layer append
the new K/V to the paged cache and attend, through the wrappers or the cache
manager; or one KV page transfer.  Lengths follow from the case alone, every
value and every page id from the seed.

``api`` says how the pass is issued:

* ``graph``   -- plan() into a graph-mode wrapper's static buffers, then a
  replay of the layers' captured append + attention (decode loops and other
  fixed-shape steps run this way);
* ``eager``   -- plan(), then set_kv_cache() and run() per layer;
* ``manager`` -- BatchedCacheManager.plan_attention and plan_rope, then the
  fused rotation, append and attention per layer;
* ``wire``    -- pack_wire of a request's pages, unpack_wire into another pool.
"""

import math

import numpy as np
import torch

WORKSPACE_BYTES = 512 << 20  # per label, as M*'s engine allocates it
ROPE_THETA = 1e6
TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "fp32": torch.float32, "fp8": torch.float8_e4m3fn}
ELEM = {"bf16": 2, "f16": 2, "fp32": 4, "fp8": 1}


def _attn(name, api, heads, kv, *, layers=1, page=16, causal=True, chunks=0, new=(0, 0), prefix=(0, 0), decodes=0,
          ctx=(0, 0), lens=0):
    """``chunks`` requests of ``new`` tokens over ``prefix`` cached ones, then ``decodes`` one-token requests
    of ``ctx`` tokens; lengths are drawn log-uniformly (prefixes uniformly) by ``lens``."""
    case = {"api": api, "q_heads": heads[0], "kv_heads": heads[1], "head_dim": heads[2], "kv": kv, "layers": layers,
            "page": page, "causal": causal, "chunks": chunks, "new_lo": new[0], "new_hi": new[1],
            "prefix_lo": prefix[0], "prefix_hi": prefix[1], "decodes": decodes, "ctx_lo": ctx[0], "ctx_hi": ctx[1],
            "lens": lens}
    return {"name": name, **case} if name else case


def _wire(name, pages, layers, kv_heads, head_dim, page, lens):
    case = {"api": "wire", "pages": pages, "layers": layers, "kv_heads": kv_heads, "head_dim": head_dim, "page": page,
            "kv": "bf16", "lens": lens}
    return {"name": name, **case} if name else case


def listed():
    return [
        # a handful of short chats: launches and latency are all there is
        _attn("decode_b8_short", "graph", (8, 2, 128), "bf16", layers=8, decodes=8, ctx=(16, 512)),
        # one user in a long conversation, the interactive case of a speech model
        _attn("decode_b1_8k", "graph", (32, 4, 128), "bf16", layers=4, decodes=1, ctx=(8192, 8192)),
        # Orpheus (Llama-3.2-3B) shaped serving at a middling batch
        _attn("decode_orpheus_b64", "graph", (24, 8, 128), "bf16", layers=3, decodes=64, ctx=(128, 4096), lens=1),
        # Qwen3-Omni thinker shaped serving at full batch, the headline workload
        _attn("decode_thinker_b256", "manager", (32, 4, 128), "bf16", decodes=256, ctx=(512, 32768), lens=2),
        # the same over an fp8 cache
        _attn("decode_thinker_fp8_b256", "manager", (32, 4, 128), "fp8", decodes=256, ctx=(1024, 32768), lens=4),
        # BAGEL (Qwen2.5-7B) shaped continuous batching: prefill chunks among decode requests
        _attn("mixed_bagel", "eager", (28, 4, 128), "bf16", chunks=8, new=(512, 2048), prefix=(0, 8192), decodes=120,
              ctx=(1024, 16384), lens=3),
        # prefill chunks over an fp8 cache
        _attn("prefill_fp8_b4", "eager", (32, 4, 128), "fp8", chunks=4, new=(512, 2048), prefix=(0, 8192), lens=5),
        # the chunk of one arriving request: its time is the time to first token
        _attn("prefill_one_chunk", "eager", (32, 4, 128), "bf16", layers=4, chunks=1, new=(512, 512),
              prefix=(4096, 4096)),
        # Pi0.5 shaped action steps: a short bidirectional suffix over an encoded prefix, the same shape each step
        _attn("suffix_pi05_b2", "graph", (8, 1, 256), "bf16", layers=8, causal=False, chunks=2, new=(50, 50),
              prefix=(800, 1000)),
        # Pi0.5 shaped prefix encoding with its cache in fp32
        _attn("prefix_pi05_fp32_b4", "eager", (8, 1, 256), "fp32", causal=False, chunks=4, new=(800, 1000)),
        # long prompts at head_dim 256
        _attn("prefill_d256_b8", "eager", (16, 2, 256), "bf16", chunks=8, new=(2048, 2048), prefix=(2048, 5632),
              lens=6),
        # the pages of one 32k-token request handed to another engine
        _wire("kv_wire_2048_pages", 2048, 8, 4, 128, 16, 0),
    ]


HEADS = [(8, 2, 128), (24, 8, 128), (32, 4, 128), (28, 4, 128), (8, 1, 256), (16, 2, 256), (16, 4, 64)]
MOST_BYTES, MOST_FLOPS = 3.2e9, 7e11


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "decode", "full", "mixed", "chunk", "suffix", "fp32", "wire"])
    lens, page = rng.randrange(1 << 20), rng.choice([16, 16, 16, 32, 64, 128])
    if kind == "wire":
        return _wire(None, _log(rng, 32, 2048), rng.randint(1, 8), rng.choice([1, 2, 4, 8]), 128, page if page < 64 else 16,
                     lens)
    while True:
        if kind in ("small", "decode"):
            hi = _log(rng, 64, 32768)
            n = _log(rng, 1, 8) if kind == "small" else _log(rng, 4, 120)
            c = _attn(None, "graph", rng.choice(HEADS), rng.choice(["bf16", "bf16", "f16", "fp8", "fp32"]),
                      layers=rng.randint(1, 8), page=page, decodes=n, ctx=(max(16, hi // _log(rng, 1, 64)), hi),
                      lens=lens)
        elif kind == "full":
            hi = _log(rng, 2048, 32768)
            c = _attn(None, "manager", rng.choice([(32, 4, 128), (24, 8, 128), (28, 4, 128), (16, 2, 256)]),
                      rng.choice(["bf16", "fp8"]), page=page, decodes=_log(rng, 96, 320),
                      ctx=(hi // _log(rng, 2, 64), hi), lens=lens)
        elif kind == "mixed":
            hi = _log(rng, 1024, 16384)
            c = _attn(None, "eager", rng.choice(HEADS), rng.choice(["bf16", "bf16", "f16", "fp8"]), page=page,
                      chunks=_log(rng, 1, 8), new=(_log(rng, 24, 512), _log(rng, 512, 2048)),
                      prefix=(0, _log(rng, 64, 8192)), decodes=_log(rng, 1, 150), ctx=(hi // _log(rng, 2, 32), hi),
                      lens=lens)
        elif kind == "chunk":
            lo = _log(rng, 24, 2048)
            c = _attn(None, "eager", rng.choice(HEADS), rng.choice(["bf16", "bf16", "f16", "fp8"]),
                      layers=rng.randint(1, 4), page=page, causal=rng.random() < 0.75, chunks=_log(rng, 1, 8),
                      new=(lo, max(lo, _log(rng, 64, 2048))), prefix=(0, _log(rng, 16, 16384)), lens=lens)
        elif kind == "suffix":
            lo = _log(rng, 4, 128)
            c = _attn(None, "graph", rng.choice([(8, 1, 256), (8, 1, 256), (28, 4, 128), (32, 4, 128)]), "bf16",
                      layers=rng.randint(1, 8), page=page, causal=rng.random() < 0.25, chunks=_log(rng, 1, 16),
                      new=(lo, max(lo, _log(rng, 16, 256))), prefix=(_log(rng, 16, 256), _log(rng, 256, 4096)),
                      lens=lens)
        else:
            lo = _log(rng, 24, 1024)
            c = _attn(None, "eager", rng.choice([(8, 1, 256), (8, 2, 128), (16, 4, 64)]), "fp32", page=page,
                      causal=rng.random() < 0.5, chunks=_log(rng, 1, 4), new=(lo, max(lo, _log(rng, 64, 1024))),
                      prefix=(0, _log(rng, 16, 1024)), lens=lens)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= (MOST_FLOPS if c["kv"] != "fp32" else 4e10):
            return c


def _lengths(case):
    """(tokens after the append, new tokens) of each request."""
    r = np.random.default_rng(case["lens"])

    def between(lo, hi, n):
        return np.rint(np.exp(r.uniform(math.log(max(lo, 1)), math.log(max(hi, 1)), n))).astype(np.int64)

    new = between(case["new_lo"], case["new_hi"], case["chunks"])
    prefix = r.integers(case["prefix_lo"], case["prefix_hi"] + 1, case["chunks"])
    one = np.ones(case["decodes"], np.int64)
    return (np.concatenate([prefix + new, between(case["ctx_lo"], case["ctx_hi"], case["decodes"])]),
            np.concatenate([new, one]))


def _pages(case):
    """A wire case's record ranges: whole pages, the first and the last record in part."""
    r = np.random.default_rng(case["lens"])
    ts, te = np.zeros(case["pages"], np.int64), np.full(case["pages"], case["page"], np.int64)
    ts[0], te[-1] = r.integers(0, case["page"] // 2), r.integers(case["page"] // 2 + 1, case["page"] + 1)
    return ts, te


def work(case):
    if case["api"] == "wire":
        ts, te = _pages(case)
        return {"bytes": 4 * 2 * int((te - ts).sum()) * case["layers"] * case["kv_heads"] * case["head_dim"] * 2,
                "flops": 0}
    kv_len, new = _lengths(case)
    n, d, hq, hkv, e = int(new.sum()), case["head_dim"], case["q_heads"], case["kv_heads"], ELEM[case["kv"]]
    eq = max(e, 2)
    pairs = (new * (kv_len - new) + new * (new + 1) // 2) if case["causal"] else new * kv_len
    cache = int(kv_len.sum()) * hkv * d * 2 * e  # every cached row read once, the new ones among them
    rows = 2 * n * hq * d * eq + n * hkv * d * 2 * (eq + e)  # q in, out back, new K/V in and into the cache
    return {"bytes": case["layers"] * (cache + rows), "flops": case["layers"] * 4 * d * hq * int(pairs.sum())}


def tolerance(case):
    if case["api"] == "wire":
        return "exact"
    # About four times the error against 64 bits that the path shows: 6e-7 in fp32, 2.9e-4 with fp16 and
    # 2.8e-3 with bf16 probabilities and outputs (relative to the output, so no larger for long contexts).
    rel = {"fp32": 3e-6, "f16": 1.2e-3}.get(case["kv"], 1e-2)
    return {"rel": rel, "max": 10 * rel}


def _inputs(case, seed):
    """Pool, page lists and new rows of a case, without this repository's code."""
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(seed)
    hkv, d, ps, layers, kind = case["kv_heads"], case["head_dim"], case["page"], case["layers"], case["kv"]
    if case["api"] == "wire":
        pool = 2 * case["pages"]
        src, dst = (torch.empty(layers, pool, 2, ps, hkv, d, dtype=torch.bfloat16, device=dev).normal_(generator=g)
                    for _ in range(2))
        at = np.random.default_rng(seed)
        return {"src": src, "dst": dst, "src_pages": at.permutation(pool)[: case["pages"]],
                "dst_pages": at.permutation(pool)[: case["pages"]]}
    kv_len, new = _lengths(case)
    pages = -(-kv_len // ps)
    pool = int(pages.sum()) + max(8, int(pages.sum()) // 8)  # the rest of the pool is free or other requests'
    perm = np.random.default_rng(seed).permutation(pool).astype(np.int32)
    indptr = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    qo = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    x = {"kv_len": kv_len, "new": new, "pool": pool, "free": perm[indptr[-1]:], "qo": torch.from_numpy(qo),
         "indptr": torch.from_numpy(indptr), "indices": torch.from_numpy(perm[: indptr[-1]].copy()),
         "last": torch.from_numpy((kv_len - (pages - 1) * ps).astype(np.int32)), "scales": None}
    wide = torch.bfloat16 if kind == "fp8" else TORCH[kind]
    kv = torch.empty(layers, pool, 2, ps, hkv, d, dtype=TORCH[kind], device=dev)
    if kind == "fp8":  # N(0, 1) values stored against per-head scales near amax / 448
        x["scales"] = (4.5 + torch.rand(layers, 2, hkv, device=dev, generator=g)) / 448
        for i in range(layers):
            for p in range(0, pool, 1 << 14):
                part = torch.empty(kv[i, p:p + (1 << 14)].shape, device=dev).normal_(generator=g)
                kv[i, p:p + (1 << 14)] = _to_fp8(part, x["scales"][i].view(1, 2, 1, hkv, 1))
    else:
        for i in range(layers):
            kv[i].normal_(generator=g)
    n = int(qo[-1])
    x["kv"] = kv
    x["q"], x["k"], x["v"] = (torch.empty(layers, n, h, d, dtype=wide, device=dev).normal_(generator=g)
                              for h in (case["q_heads"], hkv, hkv))
    return x


def _to_fp8(x, scale):
    return (x.float() * (1.0 / scale)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def prepare(case, seed):
    x = _inputs(case, seed)
    s = {"case": case, "x": x}
    if case["api"] == "wire":
        from mstar_amd.kv_transfer import wire_nbytes

        s["ts"], s["te"] = _pages(case)
        s["wire"] = torch.empty(wire_nbytes(x["src"], int((s["te"] - s["ts"]).sum())), dtype=torch.uint8,
                                device=x["src"].device)
        return s
    from mstar_amd.paged_attention import PagedDecodeWrapper, PagedPrefillWrapper

    dev, dt = x["kv"].device, x["q"].dtype
    heads = (case["q_heads"], case["kv_heads"], case["head_dim"], case["page"])
    batch, tokens, decode = len(x["new"]), int(x["qo"][-1]), case["chunks"] == 0
    s["scales"] = [(None, None) if x["scales"] is None else (x["scales"][i, 0], x["scales"][i, 1])
                   for i in range(case["layers"])]
    if case["api"] == "manager":
        s["manager"] = _manager(case, x, dev)
        return s
    graph = case["api"] == "graph"
    fixed = {"batch_size": batch, "max_num_pages": x["pool"], "use_cuda_graph": True} if graph else {}
    ws = torch.empty(WORKSPACE_BYTES, dtype=torch.uint8, device=dev)
    if decode:
        s["w"] = PagedDecodeWrapper(ws, *heads, device=dev, **fixed)
        s["plan"] = lambda: s["w"].plan(x["indptr"], x["indices"], x["last"], dtype=dt)
    else:
        if graph:
            fixed["max_total_tokens"] = tokens
        s["w"] = PagedPrefillWrapper(ws, *heads, device=dev, **fixed)
        s["plan"] = lambda: s["w"].plan(x["qo"], x["indptr"], x["indices"], x["last"], causal=case["causal"], dtype=dt)
    if graph:
        s["plan"]()
        _layers(s)  # kernels are loaded before the capture
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _layers(s)
    return s


def _manager(case, x, dev):
    """A cache manager whose requests hold all but the newest token of their contexts."""
    from mstar_amd.cache_manager import BatchedCacheManager, WorkspaceBufferManager
    from mstar_amd.kv_store import KVCacheConfig, PagedAllocationManager

    cfg = KVCacheConfig(num_layers=case["layers"], num_kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                        max_seq_len=40960, max_num_pages=x["pool"], page_size=case["page"],
                        num_qo_heads=case["q_heads"])
    alloc = PagedAllocationManager(cfg, x["kv"], device=dev)
    alloc.page_allocator.free_pages.clear()
    alloc.page_allocator.free_pages.extend(x["free"].tolist())
    names = ["request%d" % i for i in range(len(x["new"]))]
    indptr, indices = x["indptr"].tolist(), x["indices"].tolist()
    for i, name in enumerate(names):
        alloc.add_request(name, ["main"])
        state = alloc.get_state(name, "main")
        state.page_indices = indices[indptr[i]:indptr[i + 1]]
        state.seq_len = state.position_id_start = int(x["kv_len"][i]) - 1
    return BatchedCacheManager(names, {name: "main" for name in names}, x["kv"], alloc,
                               WorkspaceBufferManager(WORKSPACE_BYTES, dev), cfg, dev, kv_scales=x["scales"])


def _layers(s):
    x, w, out = s["x"], s["w"], []
    for i, (ks, vs) in enumerate(s["scales"]):
        w.set_kv_cache(x["kv"][i], x["k"][i], x["v"][i], ks, vs)
        out.append(w.run(x["q"][i], x["kv"][i], ks, vs))
    return out


def run(s):
    x, case = s["x"], s["case"]
    if case["api"] == "wire":
        from mstar_amd.kv_transfer import pack_wire, unpack_wire

        wire = pack_wire(x["src"], x["src_pages"], s["ts"], s["te"], out=s["wire"])
        unpack_wire(wire, x["dst"], x["dst_pages"], s["ts"], s["te"])
        return {"wire": wire, "kv": x["dst"]}
    if case["api"] == "manager":
        m, ones = s["manager"], [1] * len(x["new"])
        m.plan_attention(ones)
        m.plan_rope(ones)
        out = []
        for i in range(case["layers"]):
            out.append(m.apply_rope_and_run_attention(x["q"][i], x["k"][i], x["v"][i], rope_theta=ROPE_THETA,
                                                      layer_idx=i, keep_k=False))
    elif case["api"] == "graph":
        s["plan"]()
        s["graph"].replay()
        out = s["out"]
    else:
        s["plan"]()
        out = _layers(s)
    kv = x["kv"]
    return {"out": out, "kv": kv.view(torch.uint8) if kv.dtype == torch.float8_e4m3fn else kv}


def _rotate(x, pos):
    """RoPE (half split) in 64 bits."""
    d = x.shape[-1]
    freq = ROPE_THETA ** (-torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)
    a = (pos.double()[:, None] * freq)[:, None]
    lo, hi = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def exact(case, seed):
    """Append and attention in 64 bits, the cache's own rounding included."""
    if case["api"] == "wire":
        return None  # nothing is computed
    x = _inputs(case, seed)
    ps, hkv, d, dev = case["page"], case["kv_heads"], case["head_dim"], x["kv"].device
    group, qo, indptr, fp8 = case["q_heads"] // hkv, x["qo"].tolist(), x["indptr"].tolist(), case["kv"] == "fp8"
    outs = []
    for i in range(case["layers"]):
        q, k, v = (x[name][i].double() for name in "qkv")
        if case["api"] == "manager":
            pos = torch.from_numpy(x["kv_len"] - 1).to(dev)
            q, k = _rotate(q, pos), _rotate(k, pos)
        out = torch.empty_like(q)
        for r, (kv_len, new) in enumerate(zip(x["kv_len"].tolist(), x["new"].tolist())):
            at = torch.arange(kv_len - new, kv_len, device=dev)
            pages = x["indices"][indptr[r]:indptr[r + 1]].to(dev).long()
            rows = slice(qo[r], qo[r + 1])
            for j, t in enumerate((k, v)):
                t = t[rows]
                t = _to_fp8(t.to(x["k"].dtype), x["scales"][i, j].view(1, hkv, 1)) if fp8 else t.to(x["kv"].dtype)
                raw = torch.uint8 if fp8 else t.dtype
                x["kv"][i].view(raw)[pages[at // ps], j, at % ps] = t.view(raw)
            cached = x["kv"][i][pages].transpose(0, 1).reshape(2, -1, hkv, d)[:, :kv_len].double()
            if fp8:
                cached = cached * x["scales"][i].double().view(2, 1, hkv, 1)
            keys = torch.arange(kv_len, device=dev)
            for h in range(hkv):
                for a in range(0, new, 512):
                    b = min(new, a + 512)
                    part = q[qo[r] + a:qo[r] + b, h * group:(h + 1) * group].reshape(-1, d)
                    score = (part @ cached[0, :, h].t().contiguous()) / math.sqrt(d)
                    if case["causal"]:
                        score.masked_fill_(keys > at[a:b].repeat_interleave(group)[:, None], -math.inf)
                    out[qo[r] + a:qo[r] + b, h * group:(h + 1) * group] = (
                        torch.softmax(score, -1) @ cached[1, :, h].contiguous()).view(b - a, group, d)
        outs.append(out)
    return {"out": outs, "kv": None if fp8 else x["kv"]}
