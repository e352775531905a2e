"""What is measured when the speed of this framework is measured: one attention layer's
calls as a serving program makes them, over the range of sizes, types and options that the
public entry points take.

Four kinds of case:
  decode   attention.decode_attention over a paged cache (one new token per sequence)
  layer    paging.append_kv (rotary embedding + cache write), then decode_attention
  step     SplitKVHipBackend: the batch's page table, then every layer's decode call
  prefill  SplitKVHipBackend.forward_extend: new tokens over each request's cached prefix
"""
import math
import os
import random
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.abspath("decode-kernel_amd")      # the working folder is the repository's root
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import attention  # noqa: E402
import paging  # noqa: E402
from sglang_backend import SplitKVHipBackend  # noqa: E402

DEV = "cuda"
TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}
THETA = 500000.0                                 # rotary base of the repository's Llama-shaped step
K_SCALE, V_SCALE = 0.5, 0.25                     # an fp8 cache's per-tensor scales


def _case(kind, name=None, **kw):
    """A case with every field, so that two cases of a kind always have the same keys."""
    base = {
        "decode": dict(batch=1, lo=512, hi=512, hq=32, hkv=8, d=128, dtype="fp16", cache="same",
                       split=0, page=16, window=0, cap=0.0, sinks=False),
        "layer": dict(batch=1, lo=512, hi=512, hq=32, hkv=8, d=64, dtype="bf16", cache="same",
                      style=0),
        "step": dict(batch=1, lo=512, hi=512, hq=32, hkv=8, d=128, dtype="fp16", layers=2),
        "prefill": dict(batch=1, new_lo=512, new_hi=512, pre_lo=0, pre_hi=0, hq=32, hkv=8, d=128,
                        dtype="bf16", cache="same", window=0, cap=0.0, sinks=False),
    }[kind]
    out = {} if name is None else {"name": name}
    out["kind"] = kind
    out.update(base)
    out.update(kw)
    return out


def listed():
    return [
        # the smallest call: two short conversations, the reference's CPU-sized configuration
        # with its stated split; launches and host time count
        _case("decode", "decode_small", batch=2, lo=512, hi=512, split=4),
        # the benchmark's own workload: a full batch of long conversations, automatic schedule
        _case("decode", "decode_batch", batch=32, lo=8192, hi=8192),
        # a server's mixed batch: lengths anywhere from 128 to 8192 (the largest call)
        _case("decode", "decode_ragged", batch=128, lo=128, hi=8192),
        # one very long document
        _case("decode", "decode_long", batch=1, lo=131072, hi=131072, dtype="bf16"),
        # the benchmark's workload over an fp8 cache
        _case("decode", "decode_fp8", batch=32, lo=8192, hi=8192, cache="fp8"),
        # 16 q heads per kv head (the matrix-core q.k path), lengths that are no page multiple
        _case("decode", "decode_gqa16", batch=16, lo=4001, hi=4001, hq=128, dtype="bf16"),
        # soft-capped scores over head_dim 256 with a sliding window (Gemma 2's options)
        _case("decode", "decode_softcap", batch=16, lo=3000, hi=8000, hq=16, d=256, dtype="bf16",
              window=4096, cap=50.0),
        # attention sinks with a 128-token window (gpt-oss's layers)
        _case("decode", "decode_sinks", batch=32, lo=1000, hi=6000, hq=64, d=64, dtype="bf16",
              window=128, sinks=True),
        # one layer of the repository's Llama-3.2-1B-shaped step: rotary embedding, cache write,
        # attention
        _case("layer", "layer_append", batch=32, lo=2048, hi=2048),
        # a serving step through the SGLang backend: page table, then two layers
        _case("step", "backend_step", batch=16, lo=300, hi=4000),
        # prompts arriving together, some with a cached prefix
        _case("prefill", "prefill_batch", batch=8, new_lo=33, new_hi=777, pre_lo=0, pre_hi=500,
              d=64),
        # one chunk of a long prompt over what is cached of it
        _case("prefill", "prefill_chunk", batch=1, new_lo=2048, new_hi=2048, pre_lo=6144,
              pre_hi=6144),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _heads(rng):
    return rng.choice([(32, 8), (32, 8), (16, 8), (64, 8), (128, 8), (28, 4), (8, 8), (32, 16)])


def draw(rng: random.Random):
    kind = rng.choice(["decode", "decode", "decode", "layer", "step", "prefill", "prefill"])
    hq, hkv = _heads(rng)
    d = rng.choice([64, 128, 128, 256])
    dtype = rng.choice(["fp16", "bf16"])
    cache = rng.choice(["same", "same", "fp8"])
    if kind == "prefill":
        window = rng.choice([0, 0, 0, 1024])
        cap = rng.choice([0.0, 0.0, 0.0, 30.0])
        sinks = rng.random() < 0.2
        while True:
            batch = _log(rng, 1, 8)
            new, pre = _log(rng, 1, 2048), _log(rng, 1, 8192) - 1
            c = _case("prefill", batch=batch, new_lo=max(1, new // 4), new_hi=new, pre_lo=pre // 4,
                      pre_hi=pre, hq=hq, hkv=hkv, d=d, dtype=dtype, cache=cache, window=window,
                      cap=cap, sinks=sinks)
            # scores of one call (the largest listed chunk: 32 heads x 2048 x 8192), and of one
            # request where they are held whole
            if batch * hq * new * (new + pre) * max(d, 128) <= 32 * 2048 * 8192 * 128 and (
                    not (cap or sinks) or hq * new * (new + pre) <= 2 ** 28):
                return c
    top = 1 << 30 if kind == "step" else 2200 << 20          # bytes of one layer's K and V
    es = 1 if cache == "fp8" and kind != "step" else 2
    while True:
        batch, ctx = _log(rng, 1, 256), _log(rng, 16, 131072)
        if batch * ctx * hkv * d * 2 * es <= top:
            break
    lo = ctx if rng.random() < 0.5 else max(1, ctx // 16)
    if kind == "layer":
        return _case("layer", batch=batch, lo=lo, hi=ctx, hq=hq, hkv=hkv, d=d, dtype=dtype,
                     cache=cache, style=rng.choice([0, 0, 1]))
    if kind == "step":
        return _case("step", batch=batch, lo=lo, hi=ctx, hq=hq, hkv=hkv, d=d, dtype=dtype)
    return _case("decode", batch=batch, lo=lo, hi=ctx, hq=hq, hkv=hkv, d=d, dtype=dtype,
                 cache=cache, split=rng.choice([0, 0, 0, 0, 1, 4, 8]),
                 page=rng.choice([16, 16, 16, 32, 64]), window=rng.choice([0, 0, 0, 1024]),
                 cap=rng.choice([0.0, 0.0, 0.0, 30.0]), sinks=rng.random() < 0.2)


def _lengths(case, lo, hi, salt):
    """The case's lengths: the same for every seed but for their order."""
    rng = random.Random("%s %s %s %s" % (case["batch"], lo, hi, salt))
    return [rng.randint(lo, hi) for _ in range(case["batch"])]


def _generators(seed):
    cpu, gpu = torch.Generator(), torch.Generator(device=DEV)
    cpu.manual_seed(seed)
    gpu.manual_seed(seed)
    return cpu, gpu


def _rows(gen, shape, dtype, scale=1.0):
    x = torch.randn(shape, device=DEV, generator=gen, dtype=torch.float16)
    if dtype == torch.float8_e4m3fn:
        return (x / scale).clamp_(-448, 448).to(dtype)
    return x.to(dtype)


def _scales(case):
    return {"k_scale": K_SCALE, "v_scale": V_SCALE} if case.get("cache") == "fp8" else {}


def _table(lens, page, cpu):
    """A page table whose pages were handed out by a free list, and its host copies."""
    pages = [-(-n // page) for n in lens]
    ids = torch.randperm(sum(pages), generator=cpu).to(torch.int32)
    indptr = torch.zeros(len(lens) + 1, dtype=torch.int32)
    indptr[1:] = torch.tensor(pages).cumsum(0)
    last = torch.tensor([n - (p - 1) * page for n, p in zip(lens, pages)], dtype=torch.int32)
    return indptr, ids, last


def _prepare_paged(case, seed, page):
    cpu, gpu = _generators(seed)
    lens = _lengths(case, case["lo"], case["hi"], "ctx")
    random.Random(seed).shuffle(lens)
    indptr, ids, last = _table(lens, page, cpu)
    dtype = TYPES[case["dtype"]]
    shape = (ids.numel(), 1, page, case["hkv"], case["d"])
    if case["cache"] == "fp8":
        kv = torch.cat([_rows(gpu, shape, TYPES["fp8"], s).view(torch.uint8)
                        for s in (K_SCALE, V_SCALE)], dim=1).view(TYPES["fp8"])
    else:
        kv = _rows(gpu, (shape[0], 2) + shape[2:], dtype)
    return SimpleNamespace(case=case, lens=lens, kv=kv, indptr=indptr.to(DEV), ids=ids.to(DEV),
                           last=last.to(DEV), hint=attention.plan_hint(indptr), dtype=dtype,
                           gen=gpu, host=(indptr.tolist(), ids))


def _prepare_pool(case, seed, lens, extend):
    """What SGLang hands an attention backend: per-layer K and V buffers of token slots, the
    request-to-token map of a paged allocator (16 slots a page), the forward batch."""
    cpu, gpu = _generators(seed)
    dtype = TYPES[case["dtype"]]
    cdtype = TYPES["fp8"] if case.get("cache") == "fp8" else dtype
    indptr, ids, _ = _table(lens, 16, cpu)
    batch, slots = len(lens), ids.numel() * 16
    rows = torch.randperm(batch + 3, generator=cpu)[:batch]
    table = torch.zeros(batch + 3, max(lens) + 16, dtype=torch.int32)
    for b, n in enumerate(lens):
        pages = ids[indptr[b]:indptr[b + 1]]
        table[rows[b], :n] = (pages[:, None] * 16 + torch.arange(16)).reshape(-1)[:n]
    layers = case.get("layers", 1)
    shape = (slots, case["hkv"], case["d"])
    pool = _Pool([_rows(gpu, shape, cdtype, K_SCALE) for _ in range(layers)],
                 [_rows(gpu, shape, cdtype, V_SCALE) for _ in range(layers)])
    new = extend or [1] * batch
    loc = torch.cat([table[rows[b], n - m:n] for b, (n, m) in enumerate(zip(lens, new))]).long()
    fb = SimpleNamespace(
        forward_mode=SimpleNamespace(is_decode=lambda: extend is None), batch_size=batch,
        req_pool_indices=rows.to(DEV), seq_lens=torch.tensor(lens, device=DEV),
        seq_lens_sum=sum(lens), seq_lens_cpu=torch.tensor(lens), out_cache_loc=loc.to(DEV),
        extend_seq_lens_cpu=list(new),
        req_to_token_pool=SimpleNamespace(req_to_token=table.to(DEV)), token_to_kv_pool=pool)
    sc = _scales(case)
    layer = [SimpleNamespace(layer_id=i, tp_q_head_num=case["hq"], tp_k_head_num=case["hkv"],
                             tp_v_head_num=case["hkv"], head_dim=case["d"],
                             scaling=case["d"] ** -0.5, logit_cap=case.get("cap", 0.0),
                             sliding_window_size=(case.get("window") or 0) - 1,
                             k_scale=sc.get("k_scale"), v_scale=sc.get("v_scale"))
             for i in range(layers)]
    n = sum(new)
    q = [_rows(gpu, (n, case["hq"] * case["d"]), dtype) for _ in range(layers)]
    k = [_rows(gpu, (n, case["hkv"], case["d"]), dtype) for _ in range(layers)]
    v = [_rows(gpu, (n, case["hkv"], case["d"]), dtype) for _ in range(layers)]
    return SimpleNamespace(case=case, lens=lens, new=new, fb=fb, layer=layer, pool=pool, q=q, k=k,
                           v=v, loc=loc, table=table, rows=rows, gen=gpu,
                           backend=SplitKVHipBackend(None))


class _Pool:
    """A token pool as SGLang's: K and V buffers per layer, written at the batch's slots."""

    def __init__(self, k, v):
        self.k, self.v = k, v

    def get_key_buffer(self, layer_id):
        return self.k[layer_id]

    def get_value_buffer(self, layer_id):
        return self.v[layer_id]

    def set_kv_buffer(self, layer, loc, k, v, k_scale=None, v_scale=None):
        kb, vb = self.k[layer.layer_id], self.v[layer.layer_id]
        if kb.dtype == torch.float8_e4m3fn:
            kb.view(torch.uint8)[loc] = (k / k_scale).to(kb.dtype).view(torch.uint8)
            vb.view(torch.uint8)[loc] = (v / v_scale).to(vb.dtype).view(torch.uint8)
        else:
            kb[loc], vb[loc] = k, v


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        st = _prepare_paged(case, seed, case["page"])
        st.q = _rows(st.gen, (case["batch"], case["hq"], case["d"]), st.dtype)
        st.sinks = torch.randn(case["hq"], device=DEV, generator=st.gen) if case["sinks"] else None
        st.options = dict(max_pages_per_seq=st.hint, window=case["window"] or None,
                          logit_cap=case["cap"] or None, sinks=st.sinks, **_scales(case))
        return st
    if kind == "layer":
        st = _prepare_paged(case, seed, 16)
        st.qkv = _rows(st.gen, (case["batch"], case["hq"] + 2 * case["hkv"], case["d"]), st.dtype)
        st.inv_freq = paging.rope_inv_freq(case["d"], THETA, device=DEV)
        return st
    if kind == "step":
        lens = _lengths(case, case["lo"], case["hi"], "ctx")
        random.Random(seed).shuffle(lens)
        return _prepare_pool(case, seed, lens, None)
    new = _lengths(case, case["new_lo"], case["new_hi"], "new")
    pre = _lengths(case, case["pre_lo"], case["pre_hi"], "pre")
    order = list(range(case["batch"]))
    random.Random(seed).shuffle(order)
    st = _prepare_pool(case, seed, [new[i] + pre[i] for i in order], [new[i] for i in order])
    st.sinks = torch.randn(case["hq"], device=DEV, generator=st.gen) if case["sinks"] else None
    return st


def run(st):
    c = st.case
    if c["kind"] == "decode":
        return attention.decode_attention(st.q, st.kv, st.indptr, st.ids, st.last, c["split"],
                                          **st.options)
    if c["kind"] == "layer":
        # the projection's output, new in every step: append_kv rotates q where it lies
        qkv = st.qkv.clone()
        q, k, v = qkv.split([c["hq"], c["hkv"], c["hkv"]], dim=1)
        paging.append_kv(q, k, v, st.kv, st.indptr, st.ids, st.last, inv_freq=st.inv_freq,
                         rope_style=c["style"], **_scales(c))
        out = attention.decode_attention(q, st.kv, st.indptr, st.ids, st.last, 0,
                                         max_pages_per_seq=st.hint, **_scales(c))
        return {"out": out, "q": q, "kv": st.kv}
    if c["kind"] == "step":
        st.backend.init_forward_metadata(st.fb)
        return [st.backend.forward_decode(st.q[i], st.k[i], st.v[i], st.layer[i], st.fb)
                for i in range(c["layers"])] + st.pool.k + st.pool.v
    more = {} if st.sinks is None else {"sinks": st.sinks}
    out = st.backend.forward_extend(st.q[0], st.k[0], st.v[0], st.layer[0], st.fb, **more)
    return {"out": out, "k": st.pool.k[0], "v": st.pool.v[0]}


def _totals(case):
    """(attended (query, key) pairs of one q head, K and V rows read, new tokens, rows held)."""
    w = case.get("window") or 1 << 60
    if case["kind"] == "prefill":
        new = _lengths(case, case["new_lo"], case["new_hi"], "new")
        pre = _lengths(case, case["pre_lo"], case["pre_hi"], "pre")
        pairs = sum(min(p + i + 1, w) for n, p in zip(new, pre) for i in range(n))
        return pairs, sum(min(n + p, n + w - 1) for n, p in zip(new, pre)), sum(new)
    lens = _lengths(case, case["lo"], case["hi"], "ctx")
    seen = sum(min(n, w) for n in lens)
    return seen, seen, len(lens)


def work(case):
    pairs, rows, new = _totals(case)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    es = 1 if case.get("cache") == "fp8" else 2
    layers = case.get("layers", 1)
    nbytes = 2 * rows * hkv * d * es + 2 * new * hq * d * 2            # K, V; q and the output
    if case["kind"] == "decode":
        nbytes += 4 * (rows // case["page"]) + 12 * new                # the page table
    else:
        nbytes += 2 * new * hkv * d * (2 + es)                         # the new K and V rows
        if case["kind"] != "layer":
            nbytes += 4 * rows // layers                               # the token map
    return {"bytes": layers * nbytes, "flops": layers * 4 * d * hq * pairs}


def tolerance(case):
    # about four times the distance to exact(), which is the output's own rounding (fp16 keeps
    # 11 bits: 2.1e-4; bf16 8: 1.7e-3) and, in a layer, the rounding of the rotated q and K too
    # (2.9e-4 and 2.4e-3)
    fp16, bf16 = (1.2e-3, 1e-2) if case["kind"] == "layer" else (9e-4, 7e-3)
    return {"rel": fp16 if case["dtype"] == "fp16" else bf16}


def _attend(q, k, v, scale, window=0, cap=0.0, sinks=None):
    """q (n, hq, d): the last n tokens; k, v (t, hkv, d); causal; all float64."""
    n, hq, _ = q.shape
    t, hkv, _ = k.shape
    g = hq // hkv
    pos = torch.arange(t - n, t, device=q.device)[:, None]
    key = torch.arange(t, device=q.device)[None, :]
    mask = key <= pos
    if window:
        mask &= key > pos - window
    out = torch.empty_like(q)
    for h in range(hq):
        s = q[:, h] @ k[:, h // g].T * scale
        if cap:
            s = torch.tanh(s / cap) * cap
        s = s.masked_fill(~mask, float("-inf"))
        if sinks is not None:
            s = torch.cat([s, sinks[h].double().expand(n, 1)], dim=1)
        p = torch.softmax(s, dim=1)[:, :t]
        out[:, h] = p @ v[:, h // g]
    return out


def _rotate(x, pos, inv_freq, style):
    ang = pos.double()[:, None, None] * inv_freq.double()
    c, s = ang.cos(), ang.sin()
    y = torch.empty_like(x)
    half = x.shape[-1] // 2
    a, b = (slice(0, half), slice(half, None)) if style == 0 else (slice(0, None, 2), slice(1, None, 2))
    y[..., a] = x[..., a] * c - x[..., b] * s
    y[..., b] = x[..., b] * c + x[..., a] * s
    return y


def _new_rows(x, dtype, scale):
    """New K or V rows as an fp8 cache holds them (float64 otherwise)."""
    return (x / scale).clamp(-448, 448).float().to(dtype).double() if dtype == TYPES["fp8"] else x


def exact(case, seed):
    st = prepare(case, seed)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    scale = d ** -0.5
    sc = _scales(case)
    ks, vs = sc.get("k_scale", 1.0), sc.get("v_scale", 1.0)
    more = dict(window=case.get("window", 0), cap=case.get("cap", 0.0),
                sinks=getattr(st, "sinks", None))
    if case["kind"] in ("decode", "layer"):
        kv, (indptr, ids) = st.kv, st.host
        page = kv.shape[2]
        q = None
        if case["kind"] == "decode":
            q = st.q.double()
        else:
            # the sizes at which a float64 copy of the whole cache fits beside it
            if kv.numel() > 1 << 29:
                return None
            pos = torch.tensor(st.lens, device=DEV) - 1
            x = st.qkv.double()
            q = _rotate(x[:, :hq], pos, st.inv_freq, case["style"])
            kn = _rotate(x[:, hq:hq + hkv], pos, st.inv_freq, case["style"])
            at = st.ids[(st.indptr[1:] - 1).long()].long()
            slot = (st.last - 1).long()
            kv = torch.stack([kv[:, r].double() for r in (0, 1)], dim=1)
            kv[at, 0, slot] = _new_rows(kn, st.kv.dtype, ks)
            kv[at, 1, slot] = _new_rows(x[:, hq + hkv:], st.kv.dtype, vs)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, n in enumerate(st.lens):
            pages = ids[indptr[b]:indptr[b + 1]].to(DEV).long()
            rows = kv[pages].double().transpose(0, 1).reshape(2, -1, hkv, d)[:, :n]
            out[b] = _attend(q[b:b + 1], rows[0] * ks, rows[1] * vs, scale, **more)[0]
        return out if case["kind"] == "decode" else {"out": out, "q": q, "kv": kv}
    outs, kbs, vbs = [], [], []
    for i in range(len(st.layer)):
        loc = st.loc.to(DEV)
        kb, vb = st.pool.k[i].double(), st.pool.v[i].double()
        kb[loc] = _new_rows(st.k[i].double(), st.pool.k[i].dtype, ks)
        vb[loc] = _new_rows(st.v[i].double(), st.pool.v[i].dtype, vs)
        q = st.q[i].double().view(-1, hq, d)
        out, at = torch.empty_like(q), 0
        for b, (n, m) in enumerate(zip(st.lens, st.new)):
            slots = st.table[st.rows[b], :n].to(DEV).long()
            out[at:at + m] = _attend(q[at:at + m], kb[slots] * ks, vb[slots] * vs, scale, **more)
            at += m
        outs.append(out.view(-1, hq * d))
        kbs.append(kb)
        vbs.append(vb)
    if case["kind"] == "prefill":
        return {"out": outs[0], "k": kbs[0], "v": vbs[0]}
    return outs + kbs + vbs
