"""Performance cases of the Q8_0 paged-attention backend.

Each case is one attention layer's work as a serving program has it done
through the public entry points (``gfx906_fa``, ``gfx906_fa_paged``): the
decode, speculative-verify, prefill and mixed steps of the paged path (the
step's K/V written to the cache, then attention over it), the contiguous and
padded entries, the fused rotary cache write, and the gather.  Values are
N(0, 1), as in the repository's benchmark; lengths are ragged and drawn from
the case's own ``lens`` number, so that a case always has the same sizes;
block tables are random permutations of the pool.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gfx906-fa-vllm_amd"))

import gfx906_fa  # noqa: E402
import gfx906_fa_paged  # noqa: E402

D = 128
ROW = D // 32 * 34           # bytes of a Q8_0 row
SCALE = 1.0 / math.sqrt(D)
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}
HEADS = [(48, 8), (48, 8), (6, 1), (8, 1), (8, 4), (32, 8), (64, 8)]


def listed():
    return [
        # The next token of a few short conversations: launches and latency.
        dict(name="decode_small", kind="decode", seqs=3, ctx_lo=33, ctx_hi=900, nq=1, hq=48, hkv=8, bs=16,
             dtype="f16", fused=False, lens=1),
        # A full decode batch, the headline of the benchmark, K/V written inside the call.
        dict(name="decode_batch", kind="decode", seqs=32, ctx_lo=2048, ctx_hi=16384, nq=1, hq=48, hkv=8, bs=16,
             dtype="f16", fused=True, lens=2),
        # Speculative verify on long contexts, one shard of an 8-way tensor-parallel deployment.
        dict(name="verify_long", kind="decode", seqs=8, ctx_lo=131077, ctx_hi=131077, nq=5, hq=6, hkv=1, bs=16,
             dtype="f16", fused=False, lens=3),
        # Chunked prefill beside running conversations: the ordinary step of a busy server.
        dict(name="mixed", kind="prefill", prompts=4, len_lo=2048, len_hi=2048, prior_lo=0, prior_hi=65536,
             decodes=60, ctx_lo=1024, ctx_hi=131072, hq=48, hkv=8, bs=16, dtype="f16", lens=4),
        # One long prompt.
        dict(name="prefill_32k", kind="prefill", prompts=1, len_lo=32768, len_hi=32768, prior_lo=0, prior_hi=0,
             decodes=0, ctx_lo=0, ctx_hi=0, hq=48, hkv=8, bs=16, dtype="bf16", lens=5),
        # A few ordinary prompts of odd lengths.
        dict(name="prefill_short", kind="prefill", prompts=3, len_lo=77, len_hi=1283, prior_lo=0, prior_hi=0,
             decodes=0, ctx_lo=0, ctx_hi=0, hq=48, hkv=8, bs=16, dtype="f16", lens=6),
        # Short turns on long cached prefixes.
        dict(name="prefix_chunk", kind="prefill", prompts=8, len_lo=12, len_hi=12, prior_lo=32768, prior_hi=32768,
             decodes=0, ctx_lo=0, ctx_hi=0, hq=48, hkv=8, bs=16, dtype="f16", lens=7),
        # The contiguous entry: one new token against a long context, K kept quantized.
        dict(name="forward_decode", kind="forward", batch=1, sq=1, skv=65536, hq=8, hkv=4, how="full",
             quantize=False, lens=8),
        # The contiguous entry on a prompt: K quantized, then causal attention.
        dict(name="forward_prefill", kind="forward", batch=1, sq=2048, skv=2048, hq=8, hkv=4, how="causal",
             quantize=True, lens=9),
        # The padded batch entry over the paged cache.
        dict(name="padded", kind="padded", batch=4, sq=32, ctx_lo=1000, ctx_hi=4096, hq=48, hkv=8, bs=16,
             dtype="f32", how="causal", lens=10),
        # Rotary embedding and cache write of a prefill step.
        dict(name="rope_write", kind="rope", tokens=8192, hq=48, hkv=8, bs=16, dtype="bf16", neox=True, lens=11),
        # Paged rows gathered into contiguous ones (the reference's cache contract).
        dict(name="gather", kind="gather", seqs=16, ctx_lo=2048, ctx_hi=16384, hkv=8, bs=16, form="rows", lens=12),
    ]


def _between(rng, lo, hi):
    """A whole number, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "prefill", "forward", "forward",
                       "padded", "rope", "gather"])
    hq, hkv = rng.choice(HEADS)
    bs = rng.choice([16, 16, 32, 64])
    dtype = rng.choice(["f16", "bf16"])
    c = dict(kind=kind, lens=rng.randrange(1 << 20))
    if kind == "decode":
        seqs = _between(rng, 1, 64)
        hi = _between(rng, 40, min(131077, max(64, (1 << 22) // (seqs * hkv))))
        c.update(seqs=seqs, ctx_lo=max(16, hi // rng.choice([1, 2, 8])), ctx_hi=hi, nq=rng.choice([1, 1, 1, 2, 5, 6, 8]),
                 hq=hq, hkv=hkv, bs=bs, dtype=dtype, fused=rng.random() < 0.5)
    elif kind == "prefill":
        prompts = _between(rng, 1, 8)
        hi = _between(rng, 20, 16384 // prompts)
        prior = rng.choice([0, 0, _between(rng, 100, 65536 // prompts)])
        decodes = rng.choice([0, 0, _between(rng, 1, 32)])
        c.update(prompts=prompts, len_lo=max(1, hi // rng.choice([1, 3])), len_hi=hi, prior_lo=prior // 2, prior_hi=prior,
                 decodes=decodes, ctx_lo=64 if decodes else 0, ctx_hi=_between(rng, 100, 32768) if decodes else 0,
                 hq=hq, hkv=hkv, bs=bs, dtype=dtype)
    elif kind == "forward":
        batch = _between(rng, 1, 4)
        how = rng.choice(["full", "causal", "causal", "mask"])
        if rng.random() < 0.5:
            c.update(batch=batch, sq=rng.choice([1, 1, 2]), skv=_between(rng, 128, 131072 // batch), hq=hq, hkv=hkv,
                     how=how if how != "mask" else "full", quantize=False)
        else:
            skv = _between(rng, 64, 8192 // batch)
            c.update(batch=batch, sq=max(1, skv // rng.choice([1, 1, 2, 7])), skv=skv, hq=hq, hkv=hkv, how=how,
                     quantize=rng.random() < 0.5)
    elif kind == "padded":
        hi = _between(rng, 100, 16384)
        c.update(batch=_between(rng, 1, 8), sq=min(hi // 2, _between(rng, 1, 256)), ctx_lo=hi // 2, ctx_hi=hi, hq=hq,
                 hkv=hkv, bs=bs, dtype=rng.choice(["f32", "f16"]), how=rng.choice(["full", "causal", "causal", "mask"]))
    elif kind == "rope":
        c.update(tokens=_between(rng, 1, 32768), hq=hq, hkv=hkv, bs=bs, dtype=dtype, neox=rng.random() < 0.7)
    else:
        hi = _between(rng, 100, 16384)
        c.update(seqs=_between(rng, 1, 32), ctx_lo=max(1, hi // 4), ctx_hi=hi, hkv=hkv, bs=bs,
                 form=rng.choice(["rows", "planar"]))
    return c


# --- sizes and inputs ----------------------------------------------------------------------------
def _lens(case):
    """(context lengths, query lengths) of the case's sequences, prompts first."""
    rng = random.Random(case["lens"])
    kind = case["kind"]
    if kind == "decode":
        return ([max(case["nq"], _between(rng, case["ctx_lo"], case["ctx_hi"])) for _ in range(case["seqs"])],
                [case["nq"]] * case["seqs"])
    if kind == "prefill":
        q = [rng.randint(case["len_lo"], case["len_hi"]) for _ in range(case["prompts"])]
        prior = [rng.randint(case["prior_lo"], case["prior_hi"]) for _ in q]
        ctx = [a + b for a, b in zip(q, prior)]
        more = [_between(rng, case["ctx_lo"], case["ctx_hi"]) for _ in range(case["decodes"])]
        return ctx + more, q + [1] * len(more)
    if kind == "padded":
        return ([max(case["sq"], rng.randint(case["ctx_lo"], case["ctx_hi"])) for _ in range(case["batch"])],
                [case["sq"]] * case["batch"])
    if kind == "gather":
        return [rng.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["seqs"])], []
    raise KeyError(kind)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _raw_paged(case, seed):
    """K and V of every cached token (sequence-major) and the queries."""
    g, td = _gen(seed), TYPES[case["dtype"]]
    ctx, nq = _lens(case)
    kvt = torch.float16 if case["dtype"] == "f32" else td
    k = _randn(g, (sum(ctx), case["hkv"], D), kvt)
    v = _randn(g, (sum(ctx), case["hkv"], D), kvt)
    q = _randn(g, (sum(nq), case["hq"], D), td)
    return k, v, q


def _pages(g, ctx, bs):
    """Permuted block table and the slot of every cached token."""
    need = [(n + bs - 1) // bs for n in ctx]
    total = sum(need)
    perm = torch.randperm(total + 1, generator=g, device="cuda")[:total]
    bt = torch.full((len(ctx), max(need)), -1, dtype=torch.int32, device="cuda")
    slots, at = [], 0
    for s, (n, m) in enumerate(zip(ctx, need)):
        mine = perm[at:at + m]
        bt[s, :m] = mine.to(torch.int32)
        slots.append((mine[:, None] * bs + torch.arange(bs, device="cuda")).reshape(-1)[:n])
        at += m
    return bt, torch.cat(slots), total + 1


def _int32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _mask(g, batch, sq, cols):
    """An additive mask as the reference's callers build: rows that see a causal range, the rest far below."""
    j = torch.arange(sq, device="cuda")[:, None] + (cols - sq)
    seen = torch.arange(cols, device="cuda")[None] <= j
    m = torch.zeros((batch, sq, cols), dtype=torch.float16, device="cuda")
    m += 0.25 * _randn(g, (batch, sq, cols), torch.float16)
    return m.masked_fill_(~seen, -math.inf)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _prepare_step(case, seed)
    if kind == "forward":
        return _prepare_forward(case, seed)
    if kind == "padded":
        return _prepare_padded(case, seed)
    if kind == "rope":
        return _prepare_rope(case, seed)
    return _prepare_gather(case, seed)


def _fill_cache(k, v, slots, nb, bs, hkv):
    cache = gfx906_fa.new_kv_cache(nb, bs, hkv, D, device="cuda")
    gfx906_fa.reshape_and_cache_q8_kv(k, v, slots, cache[:, 0], cache[:, 1])
    return cache


def _prepare_step(case, seed):
    ctx, nq = _lens(case)
    k, v, q = _raw_paged(case, seed)
    bt, slots, nb = _pages(_gen(seed + 7919), ctx, case["bs"])
    cache = _fill_cache(k, v, slots, nb, case["bs"], case["hkv"])
    new, at = [], 0
    for n, m in zip(ctx, nq):  # the step's own tokens: the last of each sequence
        at += n
        new.append(torch.arange(at - m, at, device="cuda"))
    new = torch.cat(new)
    qsl = [0]
    for m in nq:
        qsl.append(qsl[-1] + m)
    size = gfx906_fa.workspace_size(len(ctx), sum(nq), case["hq"], case["hkv"], max(nq), max(ctx))
    return dict(case=case, q=q, k=k[new].contiguous(), v=v[new].contiguous(), slots=slots[new].contiguous(),
                cache=cache, bt=bt, ctx=_int32(ctx), qsl=_int32(qsl), max_q=max(nq), max_k=max(ctx),
                out=torch.empty_like(q), ws=gfx906_fa.new_workspace(size, q.device))


def _prepare_forward(case, seed):
    g = _gen(seed)
    b, sq, skv, hq, hkv = (case[n] for n in ("batch", "sq", "skv", "hq", "hkv"))
    q = _randn(g, (b, hq, sq, D), torch.float32)
    k = _randn(g, (b, hkv, skv, D), torch.float16)
    v = _randn(g, (b, hkv, skv, D), torch.float16)
    st = dict(case=case, q=q, k=k, v=v, off=None, mask=None)
    if not case["quantize"]:
        st["kq"] = gfx906_fa.quantize_q8_0(k)
    if case["how"] == "causal":
        st["off"] = torch.full((b,), skv - sq, dtype=torch.int32, device="cuda")
    elif case["how"] == "mask":
        st["mask"] = _mask(g, b, sq, skv)
    return st


def _prepare_padded(case, seed):
    ctx, nq = _lens(case)
    k, v, q = _raw_paged(case, seed)
    bt, slots, nb = _pages(_gen(seed + 7919), ctx, case["bs"])
    cache = _fill_cache(k, v, slots, nb, case["bs"], case["hkv"])
    b, sq = case["batch"], case["sq"]
    st = dict(case=case, q=q.view(b, sq, case["hq"], D).transpose(1, 2).contiguous(), cache=cache, bt=bt,
              ctx=_int32(ctx), off=None, mask=None)
    if case["how"] == "causal":
        st["off"] = _int32([n - sq for n in ctx])
    elif case["how"] == "mask":
        st["mask"] = _mask(_gen(seed + 104729), b, sq, max(ctx))
    return st


def _raw_rope(case, seed):
    g, td, t = _gen(seed), TYPES[case["dtype"]], case["tokens"]
    q = _randn(g, (t, case["hq"], D), td)
    k = _randn(g, (t, case["hkv"], D), td)
    v = _randn(g, (t, case["hkv"], D), td)
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))
    f = torch.outer(torch.arange(32768, device="cuda", dtype=torch.float32), inv)
    table = torch.cat([f.cos(), f.sin()], dim=-1).to(td)
    pos = (torch.arange(t, device="cuda") + int(seed) % 64) % 32768
    return q, k, v, table, pos


def _prepare_rope(case, seed):
    q, k, v, table, pos = _raw_rope(case, seed)
    _, slots, nb = _pages(_gen(seed + 7919), [case["tokens"]], case["bs"])
    cache = gfx906_fa.new_kv_cache(nb, case["bs"], case["hkv"], D, device="cuda")
    return dict(case=case, q=q, k=k, v=v, table=table, pos=pos, slots=slots, cache=cache)


def _prepare_gather(case, seed):
    g = _gen(seed)
    ctx, _ = _lens(case)
    hkv, bs = case["hkv"], case["bs"]
    k = _randn(g, (sum(ctx), hkv, D), torch.float16)
    v = _randn(g, (sum(ctx), hkv, D), torch.float16)
    bt, slots, nb = _pages(_gen(seed + 7919), ctx, bs)
    sk = (max(ctx) + 31) // 32 * 32
    st = dict(case=case, bt=bt, ctx=_int32(ctx), sk=sk)
    st["k_out"] = torch.zeros((len(ctx), hkv, sk, ROW), dtype=torch.uint8, device="cuda")
    if case["form"] == "planar":
        st["cache"] = _fill_cache(k, v, slots, nb, bs, hkv)
        st["v_out"] = torch.zeros_like(st["k_out"])
    else:
        st["kc"] = torch.zeros((nb, bs, hkv, ROW), dtype=torch.uint8, device="cuda")
        gfx906_fa.reshape_and_cache_q8(k, slots, st["kc"])
        st["vc"] = torch.zeros((nb, bs, hkv, D), dtype=torch.float16, device="cuda")
        st["vc"].view(-1, hkv, D)[slots] = v
        st["v_out"] = torch.zeros((len(ctx), hkv, sk, D), dtype=torch.float16, device="cuda")
    return st


# --- one pass ----------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        kp, vp = state["cache"][:, 0], state["cache"][:, 1]
        if case.get("fused"):
            out = gfx906_fa.paged_attention(
                state["q"], kp, vp, state["bt"], state["ctx"], state["qsl"], state["max_q"], state["max_k"], SCALE,
                out=state["out"], workspace=state["ws"], new_key=state["k"], new_value=state["v"],
                slot_mapping=state["slots"])
        else:
            gfx906_fa.reshape_and_cache_q8_kv(state["k"], state["v"], state["slots"], kp, vp)
            out = gfx906_fa_paged.forward_paged(
                state["q"], kp, vp, state["bt"], state["ctx"], state["qsl"], state["max_q"], state["max_k"], SCALE,
                out=state["out"], workspace=state["ws"])
        return {"cache": state["cache"], "out": out.view(-1, case["hq"], D)}
    if kind == "forward":
        kq = gfx906_fa.quantize_q8_0(state["k"]) if case["quantize"] else state["kq"]
        out = gfx906_fa.forward(state["q"], kq, state["v"], SCALE, mask=state["mask"], q_abs_offset=state["off"])
        return {"k_q8": kq, "out": out} if case["quantize"] else {"out": out}
    if kind == "padded":
        out = gfx906_fa.forward_paged_direct(state["q"], state["cache"][:, 0], state["cache"][:, 1], state["bt"],
                                             state["ctx"], SCALE, mask=state["mask"], q_abs_offset=state["off"])
        return {"out": out}
    if kind == "rope":
        gfx906_fa.rope_and_cache_q8_kv(state["pos"], state["q"], state["k"], state["v"], state["table"], case["neox"],
                                       state["slots"], state["cache"][:, 0], state["cache"][:, 1])
        return {"cache": state["cache"], "key": state["k"], "query": state["q"]}
    if case["form"] == "planar":
        k, v = gfx906_fa.gather_paged_kv_q8q8(state["cache"][:, 0], state["cache"][:, 1], state["bt"], state["ctx"],
                                              state["sk"], state["k_out"], state["v_out"])
    else:
        k, v = gfx906_fa.gather_paged_kv_q8(state["kc"], state["vc"], state["bt"], state["ctx"], state["sk"],
                                            state["k_out"], state["v_out"])
    return {"k": k, "v": v}


# --- work and tolerance --------------------------------------------------------------------------
def _pairs(case):
    """Visible (query token, key) pairs and the keys that some query sees."""
    if case["kind"] == "forward":
        ctx, nq = [case["skv"]] * case["batch"], [case["sq"]] * case["batch"]
    else:
        ctx, nq = _lens(case)
    if case.get("how") == "full":
        return sum(n * m for n, m in zip(ctx, nq)), sum(ctx)
    if case.get("how") == "mask":  # the mask's columns end where the longest sequence does
        top = max(ctx)
        return sum(min(n, top - m + j + 1) for n, m in zip(ctx, nq) for j in range(m)), sum(ctx)
    return sum(m * (n - m) + m * (m + 1) // 2 for n, m in zip(ctx, nq)), sum(ctx)


def work(case):
    kind = case["kind"]
    if kind == "rope":
        t, hq, hkv = case["tokens"], case["hq"], case["hkv"]
        return {"bytes": t * ((hq + hkv) * D * 4 + hkv * D * 2 + hkv * 2 * ROW + D * 2 + 16), "flops": 0}
    if kind == "gather":
        ctx, _ = _lens(case)
        vb = ROW if case["form"] == "planar" else 2 * D
        sk = (max(ctx) + 31) // 32 * 32
        pages = sum((n + case["bs"] - 1) // case["bs"] for n in ctx)
        # rows of valid tokens read, their K written, and every V row written (zeros past the length)
        return {"bytes": case["hkv"] * (sum(ctx) * (2 * ROW + vb) + len(ctx) * sk * vb) + 4 * pages, "flops": 0}
    pairs, keys = _pairs(case)
    flops = 4 * D * case["hq"] * pairs
    if kind == "forward":
        rows = case["batch"] * case["sq"]
        b = keys * case["hkv"] * (ROW + 2 * D) + rows * case["hq"] * D * 8
        if case["quantize"]:
            b += keys * case["hkv"] * 2 * D
        if case["how"] == "mask":
            b += rows * case["skv"] * 2
        return {"bytes": b, "flops": flops}
    ctx, nq = _lens(case)
    b = keys * case["hkv"] * 2 * ROW + 4 * sum((n + case["bs"] - 1) // case["bs"] for n in ctx)
    if kind == "padded":
        b += sum(nq) * case["hq"] * D * (SIZE[case["dtype"]] + 4)
        if case["how"] == "mask":
            b += sum(nq) * max(ctx) * 2
    else:
        b += sum(nq) * case["hq"] * D * 2 * SIZE[case["dtype"]]
        b += sum(nq) * case["hkv"] * 2 * D * SIZE[case["dtype"]]  # the step's own K and V read
    return {"bytes": b, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gather", "rope"):  # copies; products and sums each rounded to the model type
        return "exact"
    # Four times what the path shows against 64 bits (K^ and V^ or P rounded to fp16, the output to its type):
    # rel 4.2e-4 and max 8.9e-3 with fp16 or fp32 outputs, 1.7e-3 and 2.4e-2 with bf16 ones.
    if case.get("dtype") == "bf16":
        return {"rel": 7e-3, "max": 1e-1}
    return {"rel": 1.7e-3, "max": 3.5e-2}


# --- the same in 64 bits ---------------------------------------------------------------------------
def _dequantized(x):
    """Q8_0 values of x: blocks of 32 along the last dim, an fp16 scale of amax / 127 each."""
    b = x.float().view(*x.shape[:-1], x.shape[-1] // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    d = amax / torch.full_like(amax, 127.0)
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    q = (b * inv).round().clamp(-128, 127)
    return (q.double() * d.half().double()).view(x.shape)


def _attend(q, k, v, first, mask=None):
    """q [n, G, D], k and v [keys, D], all in 64 bits: query j sees keys up to first + j (None: all)."""
    n, grp, _ = q.shape
    keys = k.shape[0]
    out = torch.zeros_like(q)
    step = max(1, (1 << 27) // max(1, keys * grp))
    for a in range(0, n, step):
        b = min(n, a + step)
        top = keys if first is None else min(keys, max(0, first + b))
        if top <= 0:
            continue
        s = torch.mm(q[a:b].reshape(-1, D), k[:top].t().contiguous()).view(b - a, grp, top) * SCALE
        if first is not None:
            lim = torch.arange(a, b, device=q.device) + first
            s.masked_fill_((torch.arange(top, device=q.device)[None] > lim[:, None])[:, None], -math.inf)
        if mask is not None:
            s += mask[a:b, :top].double()[:, None]
        m = s.amax(-1, keepdim=True)
        p = torch.exp(s - torch.where(torch.isfinite(m), m, torch.zeros_like(m)))
        p = p / p.sum(-1, keepdim=True).clamp_min(1e-300)
        out[a:b] = torch.mm(p.view(-1, top), v[:top]).view(b - a, grp, D)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "gather":
        return None
    if kind == "rope":
        return _exact_rope(case, seed)
    if kind == "forward":
        return _exact_forward(case, seed)
    ctx, nq = _lens(case)
    k, v, q = _raw_paged(case, seed)
    grp = case["hq"] // case["hkv"]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    mask = _mask(_gen(seed + 104729), case["batch"], case["sq"], max(ctx)) if case.get("how") == "mask" else None
    at = qa = 0
    for s, (n, m) in enumerate(zip(ctx, nq)):
        first = None if case.get("how") in ("full", "mask") else n - m
        for h in range(case["hkv"]):
            kd, vd = _dequantized(k[at:at + n, h]), _dequantized(v[at:at + n, h])
            rows = slice(h * grp, (h + 1) * grp)
            out[qa:qa + m, rows] = _attend(q[qa:qa + m, rows].double(), kd, vd, first,
                                           None if mask is None else mask[s])
        at += n
        qa += m
    if kind == "padded":
        return {"out": out.view(case["batch"], case["sq"], case["hq"], D).transpose(1, 2)}
    return {"cache": None, "out": out}


def _exact_forward(case, seed):
    st = _prepare_raw_forward(case, seed)
    b, sq, skv, hq, hkv = (case[n] for n in ("batch", "sq", "skv", "hq", "hkv"))
    grp = hq // hkv
    out = torch.empty((b, hq, sq, D), dtype=torch.float64, device="cuda")
    for s in range(b):
        for h in range(hkv):
            rows = slice(h * grp, (h + 1) * grp)
            got = _attend(st["q"][s, rows].double().transpose(0, 1), _dequantized(st["k"][s, h]), st["v"][s, h].double(),
                          skv - sq if case["how"] == "causal" else None,
                          None if st["mask"] is None else st["mask"][s])
            out[s, rows] = got.transpose(0, 1)
    return {"k_q8": None, "out": out} if case["quantize"] else {"out": out}


def _prepare_raw_forward(case, seed):
    """The tensors of _prepare_forward, none of them from the framework."""
    return _prepare_forward(dict(case, quantize=True), seed)


def _exact_rope(case, seed):
    q, k, _, table, pos = _raw_rope(case, seed)
    cos, sin = table[pos].double().chunk(2, dim=-1)

    def turned(x):
        x = x.double()
        c, s = cos[:, None], sin[:, None]
        y = torch.empty_like(x)
        if case["neox"]:
            a, b = x[..., :D // 2], x[..., D // 2:]
            y[..., :D // 2], y[..., D // 2:] = a * c - b * s, b * c + a * s
        else:
            a, b = x[..., 0::2], x[..., 1::2]
            y[..., 0::2], y[..., 1::2] = a * c - b * s, b * c + a * s
        return y

    return {"cache": None, "key": turned(k), "query": turned(q)}
