"""NaN and infinite scores through every form of the kernels: a row is NaN where its softmax is, whether one workgroup
sees all its keys, several launches share them, or a merge folds them.

A query with a NaN, a key with one and a score that overflows to +inf make the outputs that attend them NaN and leave
all others alone; a score of -inf weighs nothing.  The decode is held to that in float64, the split prefill also to the
unsplit call.
"""

import numpy as np
import pytest

import cases
import gpu_util as gu
import oracle as O
from test_gpu_parity import half_ulp
from test_gpu_prefill import _case
from test_gpu_prefill_split import _both

pytestmark = pytest.mark.gpu
NAN = {O.DTYPE_F32: np.float32(np.nan), O.DTYPE_BF16: 0x7FC0, O.DTYPE_F16: 0x7E00, O.DTYPE_FP8: 0x7F}
BIG = 1e30  # in bf16 and fp32: BIG * BIG is beyond fp32


def _values(c, pool, scale):
    x = {O.DTYPE_I8: lambda: pool.astype(np.float64), O.DTYPE_FP8: lambda: O.e4m3_to_f32(pool).astype(np.float64)}.get(
        c.kv, lambda: cases.decode(pool, c.kv).astype(np.float64))()
    if c.kv == O.DTYPE_I8:
        return x * scale[..., None].astype(np.float64)
    return x * scale[:, None].astype(np.float64) if c.kv == O.DTYPE_FP8 else x


def _expected(c):
    """softmax(q k^T / sqrt(D)) v in float64, where a NaN or a score past fp32 makes the row NaN and one below it
    weighs nothing."""
    q = cases.decode(c.q, c.act).astype(np.float64)[:, 0]
    kf, vf = _values(c, c.k_pool, c.k_scale), _values(c, c.v_pool, c.v_scale)
    out = np.zeros((c.B, c.Hq, c.D))
    G = c.Hq // c.Hkv
    for b in range(c.B):
        n = int(c.ctx[b]) + 1
        pages = c.block_table[b, :(n + 15) // 16]
        k, v = kf[pages].reshape(-1, c.Hkv, c.D)[:n], vf[pages].reshape(-1, c.Hkv, c.D)[:n]
        for h in range(c.Hq):
            s = k[:, h // G] @ q[b, h] / np.sqrt(c.D)
            if np.isnan(s).any() or (s > 3.4e38).any():
                out[b, h] = np.nan
                continue
            p = np.where(s < -3.4e38, 0.0, np.exp(s - s.max()))
            out[b, h] = (p / p.sum()) @ v[:, h // G]
    return out


def _one(value, dt):
    """`value` in storage."""
    return NAN[dt] if np.isnan(value) else cases.encode(np.array([value], np.float32), dt)[0]


def _set_key(c, b, t, head, value):
    """Token t of row b, KV head `head`: dim 0 (or the int8 scale) becomes `value`."""
    page, slot = int(c.block_table[b, t // 16]), t % 16
    if not np.isnan(value):
        c.k_pool[page, slot, head, 0] = _one(value, c.kv)
    elif c.kv == O.DTYPE_I8:
        c.k_scale[page, slot, head] = np.nan
    else:
        c.k_pool[page, slot, head, 0] = NAN[c.kv]


def _clear_dim0(c, q):
    """Dim 0 of every query and key is 0, so that one BIG in a query meets only the keys that have one."""
    q[..., 0] = 0
    c.k_pool[..., 0] = 0
    c.k_new[..., 0] = 0


def _plant(c, kind):
    G = c.Hq // c.Hkv
    if kind == "nan query":
        c.q[1, 0, G, 3] = NAN[c.act]
    elif kind == "nan key":
        _set_key(c, 1, 45, 1, np.nan)
        _set_key(c, 0, int(c.ctx[0]), 0, np.nan)
    else:  # the scores of head G of row 1 with these keys pass fp32, all others are ordinary
        _clear_dim0(c, c.q)
        c.q[1, 0, G, 0] = _one(BIG, c.act)
        for t in [45] if kind == "+inf" else list(range(16)) + list(range(32, 48)):
            _set_key(c, 1, t, 1, BIG if kind == "+inf" else -BIG)


FORMS = [("bf16", "bf16", k) for k in ("nan query", "nan key", "+inf", "-inf")] + [
    ("f32", "f32", k) for k in ("nan query", "nan key", "+inf", "-inf")] + [
    (a, kv, k) for a, kv in (("f16", "f16"), ("bf16", "i8"), ("bf16", "fp8"), ("f32", "bf16"))
    for k in ("nan query", "nan key")]


def _check(got, want, c, tol):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    excess = np.abs(got - want)[ok] - half_ulp(np.maximum(np.abs(got), np.abs(want))[ok], c.act)
    assert float(excess.max()) <= tol


def _decode(ff, dev, c, table, shared=0):
    import torch

    up = lambda x: None if x is None else torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    args = (gu.to_dev(c.q, c.act, dev), gu.to_dev(c.k_pool, c.kv, dev), gu.to_dev(c.v_pool, c.kv, dev), up(table), up(c.ctx))
    kw = {"k_scale": up(c.k_scale), "v_scale": up(c.v_scale)}
    out = ff.paged_attention_shared_prefix(*args, shared, **kw) if shared else ff.paged_attention(*args, **kw)
    return out.double().cpu().numpy().reshape(c.B, c.Hq, c.D)


@pytest.mark.parametrize("act,kv,kind", FORMS)
@pytest.mark.parametrize("B,ctx", [(3, 250), (2, 900), (40, 90)])
def test_decode(ff, gpu, act, kv, kind, B, ctx):
    """Behind its own table (one launch where the rule takes it) and behind a wide one (pieces of a page or a few, merged
    by 16 waves per head, by fewer, and by one thread)."""
    c = cases.make_case(8000 + B, B, 8, 2, 128, [ctx - 7 * (b % 5) for b in range(B)], act=act, kv=kv)
    _plant(c, kind)
    want = _expected(c)
    wide = np.full((c.B, 600), -1, dtype=np.int32)
    wide[:, :c.max_blocks] = c.block_table
    for table in (c.block_table, wide):
        _check(_decode(ff, gpu, c, table), want, c, 2e-2 if kv in ("i8", "fp8") else 2e-3)


@pytest.mark.parametrize("act,kv,kind", FORMS)
@pytest.mark.parametrize("Hq,D", [(8, 88), (16, 128)])
def test_vector_decode(ff, gpu, act, kv, kind, Hq, D):
    """The vector kernel where its lanes past the head load like the others (a head dim of no instance of its own), and with
    eight heads per KV head (fp32 pages)."""
    c = cases.make_case(8300 + D, 3, Hq, 2, D, [300, 250, 90], act=act, kv=kv)
    _plant(c, kind)
    _check(_decode(ff, gpu, c, c.block_table), _expected(c), c, 2e-2 if kv in ("i8", "fp8") else 2e-3)


@pytest.mark.parametrize("act,kv", [("bf16", "bf16"), ("f16", "f16"), ("bf16", "i8"), ("bf16", "fp8")])
@pytest.mark.parametrize("kind", ["nan query", "nan key"])
@pytest.mark.parametrize("B", [3, 40])
def test_shared_prefix(ff, gpu, act, kv, kind, B):
    """In the shared pages (token 45) and in a row's own."""
    c = cases.make_case(8100 + B, B, 8, 2, 128, [330 + 7 * (b % 5) for b in range(B)], act=act, kv=kv,
                        shared_prefix_blocks=16)
    _plant(c, kind)
    _check(_decode(ff, gpu, c, c.block_table, shared=16), _expected(c), c, 2e-2 if kv in ("i8", "fp8") else 2e-3)


@pytest.mark.parametrize("act,kv,kind", FORMS[:4] + FORMS[8:])
@pytest.mark.parametrize("t", [45, 1400, 1510])
def test_split_prefill(ff, gpu, act, kv, kind, t):
    """A prompt chunk of 20 tokens over 1500: the same rows NaN as in the unsplit call, for a key that all queries see (in
    the first and in the last piece) or, at 1510, only the later ones."""
    c, qn = _case(8200, 1, 8, 2, 128, [1500], 20, act=act, kv=kv)
    hit = np.zeros((1, 20, 8), dtype=bool)
    if kind == "nan query":
        qn[0, 7, 5, 3] = NAN[c.act]
        hit[0, 7, 5] = True
    else:
        if kind != "nan key":
            _clear_dim0(c, qn)
            qn[0, 12, 5, 0] = _one(BIG, c.act)
        value = {"nan key": np.nan, "+inf": BIG, "-inf": -BIG}[kind]
        if t < 1500:
            _set_key(c, 0, t, 1, value)
        else:  # a token of the chunk, in the source's type: quantizing keeps no NaN, so only float caches hold one
            if kv in ("i8", "fp8"):
                pytest.skip("a quantized token holds no NaN")
            c.k_new[0, t - 1500, 1, 0] = _one(value, c.act)
        if kind == "nan key":
            hit[0, max(0, t - 1500):, 4:] = True
        elif kind == "+inf":
            hit[0, 12, 5] = True
    got, whole, _, split = _both(ff, gpu, c, qn, False)
    assert split
    assert np.array_equal(np.isnan(got).all(axis=-1), hit) and np.array_equal(np.isnan(got), np.isnan(whole))
    ok = ~np.isnan(whole)
    tol = 2e-2 if kv in ("i8", "fp8") else 2e-3
    d = np.abs(got - whole)[ok] - 2 * half_ulp(np.maximum(np.abs(got), np.abs(whole))[ok], c.act)
    assert float(d.max()) <= 2 * tol
