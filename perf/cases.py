"""Performance cases of the paged KV-cache path: what an engine has it do, layer by layer.

Every case is one call, or the calls of one layer in one step, through ``firefly_amd``'s functions on one layer's
pools.  ``op`` says which:

  step     a decode step: append one token per row and attend its whole context
           (``append_paged_attention``; with ``rope``: ``rope_append_kv_cache`` then ``paged_attention``)
  shared   the attention of a decode step whose rows share their first pages (``paged_attention_shared_prefix``)
  prefill  a prompt chunk: append its K/V, then causal attention over the cached prefix and the chunk
           (``append_kv_cache`` then ``paged_prefill``), or, with ``ctx_hi`` 0 and ``contiguous``, the causal
           prefill of a whole prompt over its own K/V
  append   a chunk's K/V into the pages (quantizing caches quantize), with ``rope`` after rotating q and k

Context lengths are spread evenly over [ctx_lo, ctx_hi] and dealt to the rows in an order drawn from the seed, so
the work of a case does not depend on the seed.  Pages are scattered over a pool 10 % larger than needed, as an
allocator in use leaves them; ``wide`` block tables have the row stride of an engine whose context limit is well
above the contexts at hand.  Values are N(0, 1); quantized caches hold them with 1 % of the elements 8 times larger.
"""

from __future__ import annotations

import math
import random

import torch

import firefly_amd as ff

BLOCK = ff.BLOCK_SIZE
THETA = 1e6
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8, "fp8": torch.uint8}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1, "fp8": 1}


def _case(op, batch, heads, kv_heads, head_dim, ctx_lo, ctx_hi, q="bf16", kv="bf16", seq=1, shared=0, rope=False,
          contiguous=False, wide=False, **name):
    return {**name, "op": op, "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "q": q, "kv": kv, "seq": seq, "shared": shared, "rope": rope,
            "contiguous": contiguous, "wide": wide}


def listed():
    return [
        # A few short chats on a small model (16 query heads, 8 KV heads): the smallest step, all launch and latency.
        _case("step", 4, 16, 8, 128, 17, 255, name="step_small"),
        # An ordinary decode step of an 8B-class layer at moderate load, with the rotary embedding in the append.
        _case("step", 16, 32, 8, 128, 256, 2048, rope=True, wide=True, name="step_rope_b16"),
        # The headline decode step: 64 rows of 512 to 4096 tokens.
        _case("step", 64, 32, 8, 128, 512, 4096, name="step_b64"),
        # Long documents: few rows of 32k tokens, 7 query heads per KV head.
        _case("step", 8, 28, 4, 128, 32768, 32768, name="step_long"),
        # A full server on an int8 cache (the largest case), and a busy one on an fp8 cache.
        _case("step", 256, 32, 8, 128, 1024, 8192, kv="i8", name="step_int8_b256"),
        _case("step", 48, 32, 8, 128, 1024, 8192, kv="fp8", wide=True, name="step_fp8_b48"),
        # fp32 activations and cache, as a numerically conservative deployment or a debugging run has them.
        _case("step", 32, 32, 8, 128, 512, 4096, q="f32", kv="f32", name="step_f32"),
        # 120 chats behind one 2048-token system prompt whose pages the radix tree shares.
        _case("shared", 120, 32, 8, 128, 2048 + 64, 2048 + 1024, shared=128, name="decode_shared_prefix"),
        # Eight prompts' 512-token chunks over what they have cached.
        _case("prefill", 8, 32, 8, 128, 2048 + 64, 2048 + 1024, seq=512, name="prefill_chunks_b8"),
        # One request's 256-token chunk (the scheduler's default) deep in a long prompt: one prompt at a time is how
        # the reference engine prefills.
        _case("prefill", 1, 32, 8, 128, 7919, 7919, seq=256, wide=True, name="prefill_one_chunk"),
        # A whole prompt with nothing cached, over its own contiguous K/V.
        _case("prefill", 1, 32, 8, 128, 0, 0, q="f16", kv="f16", seq=2000, contiguous=True, name="prefill_prompt"),
        # Prompt chunks into an int8 cache.
        _case("append", 64, 32, 8, 128, 0, 4096, kv="i8", seq=512, name="append_int8"),
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choices(["step", "prefill", "shared", "append"], [5, 4, 1, 2])[0]
    kv_heads = rng.choice([2, 4, 8, 8, 8])
    group = rng.choice([1, 2, 4, 4, 5, 7, 8])
    heads = kv_heads * group
    rope = False
    if op == "step":
        kv = rng.choices(["bf16", "f16", "i8", "fp8", "f32"], [5, 2, 2, 2, 1])[0]
        rope = rng.random() < 0.4
        head_dim = rng.choice([64, 128, 128, 128, 256] if rope else [64, 80, 96, 112, 128, 128, 128, 128, 256])
        batch, hi = _log(rng, 1, 256), _log(rng, 64, 32768)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        most = 2.4e9 / (kv_heads * head_dim * _BYTES[kv] * 2) / batch  # mean tokens per row that the largest case allows
        hi = max(32, min(hi, int(most)))
        return _case("step", batch, heads, kv_heads, head_dim, min(lo, hi), hi, q=kv if kv in ("f16", "f32") else "bf16",
                     kv=kv, rope=rope, wide=rng.random() < 0.5)
    if op == "shared":
        kv = rng.choices(["bf16", "f16", "i8", "fp8"], [5, 2, 2, 2])[0]
        shared = _log(rng, 4, 256)
        head_dim = rng.choice([64, 128, 128, 128])
        lo = shared * BLOCK + rng.randrange(0, 65)
        return _case("shared", _log(rng, 8, 128), heads, kv_heads, head_dim, lo, lo + _log(rng, 64, 1024),
                     q="f16" if kv == "f16" else "bf16", kv=kv, shared=shared)
    if op == "prefill":
        contiguous = rng.random() < 0.25
        kv = rng.choices(["bf16", "f16"] if contiguous else ["bf16", "f16", "i8", "fp8"],
                         [1, 1] if contiguous else [5, 2, 2, 2])[0]
        head_dim = rng.choice([64, 128, 128, 128, 256])
        batch, seq = _log(rng, 1, 4 if contiguous else 16), _log(rng, 16, 2048)
        hi = 0 if contiguous else _log(rng, 64, 16384)
        lo = int(hi * rng.uniform(0.1, 1.0))
        if contiguous:
            seq = max(seq, 64)
        while 4.0 * batch * seq * (0.5 * (lo + hi) + 0.5 * seq) * heads * head_dim > 2.0e11:
            batch, seq, lo, hi = max(1, batch // 2), max(64, seq * 3 // 4), lo * 3 // 4, hi * 3 // 4
        return _case("prefill", batch, heads, kv_heads, head_dim, lo, hi, q="f16" if kv == "f16" else "bf16", kv=kv,
                     seq=seq, contiguous=contiguous, wide=not contiguous and rng.random() < 0.5)
    kv = rng.choices(["bf16", "f16", "i8", "fp8"], [4, 2, 3, 3])[0]
    head_dim = rng.choice([64, 128, 128, 128, 256])
    batch = _log(rng, 1, 64)
    seq = _log(rng, 16, max(16, 65536 // batch))
    hi = _log(rng, 64, 8192)
    return _case("append", batch, heads, kv_heads, head_dim, int(hi * rng.uniform(0.0, 1.0)), hi,
                 q="f16" if kv == "f16" else "bf16", kv=kv, seq=seq, rope=rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------------------------------------------


def _lens(case):
    """Cached tokens of the rows before the call, evenly spread over [ctx_lo, ctx_hi]."""
    n, lo, hi = case["batch"], case["ctx_lo"], case["ctx_hi"]
    if n == 1:
        return [hi if lo == hi else (lo + hi) // 2]
    return [lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _randn(shape, dtype, gen):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _outliers(shape, gen):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return x.mul_(torch.rand(shape, generator=gen, device="cuda").lt_(0.01).mul_(7.0).add_(1.0))


def _pool(pages, case, gen):
    """One pool of K or V pages and its scales, as a cache in use holds them."""
    hkv, d, kv = case["kv_heads"], case["head_dim"], case["kv"]
    pool = torch.empty((pages, BLOCK, hkv, d), dtype=_TORCH[kv], device="cuda")
    scale = None
    if kv == "i8":
        scale = torch.empty((pages, BLOCK, hkv), dtype=torch.float32, device="cuda")
    elif kv == "fp8":
        scale = torch.empty(hkv, device="cuda").uniform_(0.08, 0.1, generator=gen)
    slab = max(1, (1 << 26) // (BLOCK * hkv * d))
    for p in range(0, pages, slab):
        shape = (min(slab, pages - p), BLOCK, hkv, d)
        if kv in ("i8", "fp8"):
            x = _outliers(shape, gen)
            if kv == "i8":
                s = x.abs().amax(dim=-1) / 127.0
                scale[p:p + slab] = s
                pool[p:p + slab] = torch.round(x / s[..., None]).to(torch.int8)
            else:
                y = (x / scale[None, None, :, None]).clamp_(-448.0, 448.0)
                pool[p:p + slab] = y.to(torch.float8_e4m3fn).view(torch.uint8)
        else:
            pool[p:p + slab] = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return pool, scale


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 7919 + 17)
    order = random.Random(seed * 31 + 5)
    b, s, hq, hkv, d = case["batch"], case["seq"], case["heads"], case["kv_heads"], case["head_dim"]
    act = _TORCH[case["q"]]
    st = {"q": _randn((b, s, hq, d), act, gen)}
    if case["op"] == "shared":
        st["k"] = st["v"] = None
    elif case["kv"] in ("i8", "fp8"):
        st["k"], st["v"] = _outliers((b, s, hkv, d), gen).to(act), _outliers((b, s, hkv, d), gen).to(act)
    else:
        st["k"], st["v"] = _randn((b, s, hkv, d), act, gen), _randn((b, s, hkv, d), act, gen)
    if case["contiguous"]:
        return st
    lens = _lens(case)
    order.shuffle(lens)
    shared = case["shared"]
    need = [(n + s + BLOCK - 1) // BLOCK for n in lens]
    pages = math.ceil((shared + sum(n - shared for n in need)) * 1.1)
    perm = list(range(pages))
    order.shuffle(perm)
    width = max(need)
    if case["wide"]:
        width = max(256, 2 * width)
    rows, at = [], shared
    for n in need:
        rows.append(perm[:shared] + perm[at:at + n - shared] + [-1] * (width - n))
        at += n - shared
    st["table"] = torch.tensor(rows, dtype=torch.int32, device="cuda")
    st["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    st["k_cache"], st["k_scale"] = _pool(pages, case, gen)
    st["v_cache"], st["v_scale"] = _pool(pages, case, gen)
    return st


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    b, s, hq, hkv, d = case["batch"], case["seq"], case["heads"], case["kv_heads"], case["head_dim"]
    if case["op"] != "append":
        st["out"] = torch.empty((b, s, hq * d), dtype=_TORCH[case["q"]], device="cuda")
    if case["op"] == "step":
        st["workspace"] = ff.decode_workspace(b, hq, d, st["table"].shape[1])
    elif case["op"] == "shared":
        st["workspace"] = ff.shared_prefix_workspace(b, hq, hkv, d, st["table"].shape[1], case["shared"])
    return st


# ---- one pass ----------------------------------------------------------------------------------------------------


def _caches(st):
    got = {"k_cache": st["k_cache"], "v_cache": st["v_cache"]}
    if st["case"]["kv"] == "i8":
        got.update(k_scale=st["k_scale"], v_scale=st["v_scale"])
    return got


def run(st):
    case = st["case"]
    op = case["op"]
    if case["contiguous"]:
        return {"out": ff.paged_prefill(st["q"], st["k"], st["v"], None, None, out=st["out"])}
    kc, vc, bt, cx = st["k_cache"], st["v_cache"], st["table"], st["lens"]
    scales = {"k_scale": st["k_scale"], "v_scale": st["v_scale"]}
    if op == "shared":
        return {"out": ff.paged_attention_shared_prefix(st["q"], kc, vc, bt, cx, case["shared"], out=st["out"],
                                                        workspace=st["workspace"], **scales)}
    if op == "step":
        if not case["rope"]:
            out = ff.append_paged_attention(st["k"], st["v"], st["q"], kc, vc, bt, cx, out=st["out"],
                                            workspace=st["workspace"], **scales)
            return {"out": out, **_caches(st)}
        ff.rope_append_kv_cache(st["q"], st["k"], st["v"], kc, vc, bt, cx, theta=THETA, **scales)
        out = ff.paged_attention(st["q"], kc, vc, bt, cx, out=st["out"], workspace=st["workspace"], **scales)
        return {"out": out, "q": st["q"], "k": st["k"], **_caches(st)}
    if op == "append":
        if case["rope"]:
            ff.rope_append_kv_cache(st["q"], st["k"], st["v"], kc, vc, bt, cx, theta=THETA, **scales)
            return {"q": st["q"], "k": st["k"], **_caches(st)}
        ff.append_kv_cache(st["k"], st["v"], kc, vc, bt, cx, **scales)
        return _caches(st)
    ff.append_kv_cache(st["k"], st["v"], kc, vc, bt, cx, **scales)
    return {"out": ff.paged_prefill(st["q"], kc, vc, bt, cx, out=st["out"], **scales), **_caches(st)}


# ---- what a pass cannot do without, and how far two correct ones may lie apart --------------------------------------


def work(case):
    b, s, hq, hkv, d = case["batch"], case["seq"], case["heads"], case["kv_heads"], case["head_dim"]
    es, qs, op = _BYTES[case["kv"]], _BYTES[case["q"]], case["op"]
    row = 2 * (hkv * d * es + (4 * hkv if case["kv"] == "i8" else 0))  # a cached token's K and V, with scales
    source = 2 * b * s * hkv * d * qs  # the new tokens' K and V
    lens = [0] * b if case["contiguous"] else _lens(case)
    seen = sum(lens) + b * s  # tokens attended
    pages = 0 if case["contiguous"] else 4 * sum((n + s + BLOCK - 1) // BLOCK for n in lens) + 4 * b
    nbytes = flops = 0.0
    if op == "append":
        nbytes = source + b * s * row + 4 * b * ((s + BLOCK - 1) // BLOCK) + 4 * b
    else:
        nbytes = 2 * b * s * hq * d * qs + pages
        flops = 4.0 * hq * d * sum(s * n + s * (s + 1) / 2 for n in lens)
        if case["contiguous"]:
            nbytes += source
        elif op == "shared":
            nbytes += (seen - (b - 1) * case["shared"] * BLOCK) * row
        else:  # the cached tokens are read, the new ones come from their source and are written
            nbytes += (seen - b * s) * row + source + b * s * row
    if case["rope"]:  # q (unless the attention reads it anyway) and k written back rotated
        nbytes += b * s * (hq + hkv) * d * qs + (b * s * hq * d * qs if op == "append" else 0)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["op"] == "append" and not case["rope"]:
        return "exact"
    return {"rel": {"f32": 1e-5, "f16": 1.5e-3, "bf16": 1e-2}[case["q"]]}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------


def _value(pool, scale, kv):
    """Cached rows [..., Hkv, D] in 64 bits."""
    if kv == "fp8":
        return pool.view(torch.float8_e4m3fn).to(torch.float32).double() * scale.double()[:, None]
    return pool.double() * (scale.double()[..., None] if kv == "i8" else 1.0)


def _rotate(x, lens):
    """Rotary embedding of x [B, S, H, D] at positions lens[b] + t: inverse frequencies and angles are single
    precision by definition, the rest is 64 bits; rounded to x's type, as it is stored."""
    b, s, _, d = x.shape
    inv = torch.pow(torch.tensor(THETA, dtype=torch.float64, device=x.device),
                    -2.0 * torch.arange(d // 2, dtype=torch.float64, device=x.device) / d).float()
    pos = (lens.long()[:, None] + torch.arange(s, device=x.device)).float()
    ang = (pos[..., None] * inv).double()[:, :, None, :]
    lo, hi = x[..., :d // 2].double(), x[..., d // 2:].double()
    return torch.cat((lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()), dim=-1).to(x.dtype)


def _attend(q, k, v, first):
    """q [S, Hq, D] at positions first .. first + S - 1 over k, v [L, Hkv, D]; 64 bits."""
    s, hq, d = q.shape
    hkv, n = k.shape[1], k.shape[0]
    qd = q.double().reshape(s, hkv, hq // hkv, d).permute(1, 2, 0, 3).reshape(hkv, -1, d)
    p = torch.matmul(qd, k.permute(1, 2, 0).contiguous()) / math.sqrt(d)
    if s > 1:
        seen = torch.arange(n, device=q.device)[None, :] <= first + torch.arange(s, device=q.device)[:, None]
        p = p.reshape(hkv, -1, s, n).masked_fill_(~seen, -math.inf).reshape(hkv, -1, n)
    o = torch.matmul(torch.softmax(p, dim=-1), v.permute(1, 0, 2).contiguous())
    return o.reshape(hkv, hq // hkv, s, d).permute(2, 0, 1, 3).reshape(s, hq * d)


def exact(case, seed):
    if case["op"] == "append" and case["kv"] == "fp8" and not case["rope"]:
        return None  # codes alone
    st = _inputs(case, seed)
    b, s, kv = case["batch"], case["seq"], case["kv"]
    if case["contiguous"]:
        return {"out": torch.stack([_attend(st["q"][i], st["k"][i].double(), st["v"][i].double(), 0)
                                    for i in range(b)])}
    got, quant = {}, kv in ("i8", "fp8")
    if case["rope"]:
        st["q"], st["k"] = _rotate(st["q"], st["lens"]), _rotate(st["k"], st["lens"])
        got.update(q=st["q"].double(), k=st["k"].double())
    if st["k"] is not None:
        pos = st["lens"].long()[:, None] + torch.arange(s, device="cuda")
        page = torch.gather(st["table"].long(), 1, pos // BLOCK)
        for name in ("k", "v"):
            x, pool, scale = st[name], st[name + "_cache"], st[name + "_scale"]
            if kv == "i8":
                sc = x.float().abs().amax(dim=-1) / 127.0
                scale[page, pos % BLOCK] = sc
                x = torch.round(x.float() / sc[..., None]).to(torch.int8)
            elif kv == "fp8":
                y = (x.float() / scale[:, None]).clamp(-448.0, 448.0)
                x = y.to(torch.float8_e4m3fn).view(torch.uint8)
            pool[page, pos % BLOCK] = x
        # codes are whole numbers: no 64-bit value stands for them
        got.update(k_cache=None if quant else st["k_cache"], v_cache=None if quant else st["v_cache"])
        if kv == "i8":
            got.update(k_scale=st["k_scale"], v_scale=st["v_scale"])
    if case["op"] == "append":
        return got
    out = []
    for i, n in enumerate(st["lens"].tolist()):
        live = n + s
        pages = st["table"][i, :(live + BLOCK - 1) // BLOCK].long()
        k, v = ((_value(st[c + "_cache"][pages], st[c + "_scale"][pages] if kv == "i8" else st[c + "_scale"], kv)
                 .reshape(-1, case["kv_heads"], case["head_dim"])[:live]) for c in "kv")
        out.append(_attend(st["q"][i], k, v, n))
    return {"out": torch.stack(out), **got}
