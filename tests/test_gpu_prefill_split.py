"""Prefill split over its keys (few blocks of 128 query rows over many keys) against the CPU closed form and against
the unsplit call.

Bar against the closed form as in test_gpu_prefill.py.  Split and unsplit differ by the order of fp32 sums and the
reference maxima of P's rounding to 11 bits: both lie within the bar, so their difference is held to the sum of two.
Each case says whether the library plans to split it (``ffkv_prefill_workspace_bytes``) at the edges of the rule on the
bound of a row (12 steps of 64 keys at five pieces and more), or, behind a wide table, whether it is split at the edges of
the rule on the longest row's own length (8 steps at eight pieces and more, 9 from five, 13 from three, 19 at two).
"""

import numpy as np
import pytest

import cases
import gpu_util as gu
import oracle as O
from test_gpu_prefill import _case, _check, half_ulp

pytestmark = pytest.mark.gpu


def _both(ff, dev, c, qn, contiguous):
    """(split output, unsplit output, closed form, split?) of the case's chunk."""
    import torch

    q = gu.to_dev(qn, c.act, dev)
    B, S, Hq, D = q.shape
    if contiguous:
        k, v = gu.to_dev(c.k_new, c.act, dev), gu.to_dev(c.v_new, c.act, dev)
        ks = vs = bt = cx = None
        ref = O.paged_prefill_f64(qn, c.act, c.k_new, c.v_new, c.act, None, None)
    else:
        k, v = gu.to_dev(c.k_pool, c.kv, dev), gu.to_dev(c.v_pool, c.kv, dev)
        ks = None if c.k_scale is None else torch.from_numpy(c.k_scale.copy()).to(dev)
        vs = None if c.v_scale is None else torch.from_numpy(c.v_scale.copy()).to(dev)
        bt, cx = torch.from_numpy(c.block_table).to(dev), torch.from_numpy(c.ctx).to(dev)
        ff.append_kv_cache(gu.to_dev(c.k_new, c.act, dev), gu.to_dev(c.v_new, c.act, dev), k, v, bt, cx, ks, vs)
        rk, rv = c.k_pool.copy(), c.v_pool.copy()
        rks = None if c.k_scale is None else c.k_scale.copy()
        rvs = None if c.v_scale is None else c.v_scale.copy()
        O.append(c.k_new, c.v_new, c.act, rk, rv, c.kv, c.block_table, c.ctx, rks, rvs)
        ref = O.paged_prefill_f64(qn, c.act, rk, rv, c.kv, c.block_table, c.ctx, rks, rvs)
    mb = 0 if contiguous else c.max_blocks
    qt, ct = ff.torch_dtype_code(q), ff.torch_dtype_code(k)
    need = ff.lib.ffkv_prefill_workspace_bytes(qt, ct, B, S, Hq, c.Hkv, D, int(not contiguous), mb, 0)
    split = ff.paged_prefill(q, k, v, bt, cx, k_scale=ks, v_scale=vs)
    whole = torch.full_like(split, float("nan"))
    ff.check(ff.lib.ffkv_paged_prefill(ff._ptr(q), ff._ptr(whole), qt, ff._ptr(k), ff._ptr(v), ct, ff._ptr(ks),
                                       ff._ptr(vs), ff._ptr(bt), ff._ptr(cx), B, S, Hq, c.Hkv, D, 16, mb,
                                       0 if contiguous else c.num_blocks, 0, 0.0, ff._stream(None)))
    torch.cuda.synchronize()
    f = lambda t: t.float().cpu().numpy().reshape(ref.shape)
    return f(split), f(whole), ref, need > 0


@pytest.mark.parametrize("B,Hq,Hkv,D,ctx,S,act,kv,splits", [
    (1, 32, 8, 128, [1500], 33, "bf16", "bf16", True),    # a remainder of a row block, pieces of 4 and 5 steps
    (1, 32, 8, 128, [703], 1, "bf16", "bf16", False),     # 11 steps: whole
    (1, 32, 8, 128, [704], 1, "bf16", "bf16", True),      # 12 steps, the last of one key
    (1, 2, 2, 128, [4000], 128, "f16", "f16", True),      # two groups over eight XCDs, one full row block each
    (2, 32, 8, 128, [0, 1200], 130, "f16", "f16", True),  # one row too short to split beside one that is split
    (3, 10, 2, 64, [900, 1111, 17], 50, "bf16", "bf16", True),
    (1, 8, 4, 256, [1000], 20, "bf16", "bf16", True),
    (1, 28, 4, 128, [1000], 70, "f32", "bf16", True),
    (2, 16, 4, 128, [1000, 850], 40, "bf16", "i8", True),
    (2, 16, 4, 128, [1000, 850], 40, "bf16", "fp8", True),
    (1, 8, 4, 64, [2100], 30, "f16", "i8", True),
])
def test_split_prefill(ff, gpu, B, Hq, Hkv, D, ctx, S, act, kv, splits):
    c, qn = _case(900 + S + D, B, Hq, Hkv, D, ctx, S, act=act, kv=kv)
    got, whole, ref, split = _both(ff, gpu, c, qn, False)
    assert split == splits
    tol = 2e-2 if kv in ("i8", "fp8") else 2e-3
    _check(got, ref, c.act, tol)
    d = np.abs(got - whole) - 2 * half_ulp(np.maximum(np.abs(got), np.abs(whole)), c.act)
    assert float(d.max()) <= 2 * tol


@pytest.mark.parametrize("S,Hq,Hkv,splits", [(770, 4, 2, True), (700, 4, 2, False)])
def test_split_prompt(ff, gpu, S, Hq, Hkv, splits):
    """A whole prompt (contiguous K/V): its late row blocks are split, the early ones are not."""
    c, qn = _case(950 + S, 1, Hq, Hkv, 128, [0], S, act="f16")
    got, whole, ref, split = _both(ff, gpu, c, qn, True)
    assert split == splits
    _check(got, ref, c.act, 2e-3)


def _pieces(ff, dev, c, qn, max_context_len=0):
    """(output, pieces of every block or None) of the case's chunk behind a table of 300 blocks, over a workspace that
    holds all ones before the call."""
    import torch

    wide = np.full((c.B, 300), -1, dtype=np.int32)
    wide[:, :c.max_blocks] = c.block_table
    q = gu.to_dev(qn, c.act, dev)
    kp, vp = gu.to_dev(c.k_pool, c.kv, dev), gu.to_dev(c.v_pool, c.kv, dev)
    bt, cx = torch.from_numpy(wide).to(dev), torch.from_numpy(c.ctx).to(dev)
    B, S, Hq, D = q.shape
    out = torch.full((B, S, Hq * D), float("nan"), dtype=q.dtype, device=dev)
    qt, ct = ff.torch_dtype_code(q), ff.torch_dtype_code(kp)
    need = ff.lib.ffkv_prefill_workspace_bytes(qt, ct, B, S, Hq, c.Hkv, D, 1, 300, max_context_len)
    ws = torch.full((max(need, 256),), 255, dtype=torch.uint8, device=dev)
    ff.check(ff.lib.ffkv_paged_prefill_ws(ff._ptr(q), ff._ptr(out), qt, ff._ptr(kp), ff._ptr(vp), ct, None, None,
                                          ff._ptr(bt), ff._ptr(cx), B, S, Hq, c.Hkv, D, 16, 300, c.num_blocks,
                                          max_context_len, 0.0, ff._ptr(ws), ws.numel(), ff._stream(None)))
    torch.cuda.synchronize()
    blocks = B * c.Hkv * ((S * Hq // c.Hkv + 127) // 128)
    return out.float().cpu().numpy(), None if need == 0 else ws[:4 * blocks].view(torch.int32).cpu().numpy()


@pytest.mark.parametrize("B,Hq,Hkv,S,rule", [(1, 32, 8, 33, 8), (1, 32, 8, 256, 8), (1, 32, 8, 350, 9), (3, 32, 8, 160, 13),
                                             (3, 32, 8, 256, 19)])
def test_wide_table(ff, gpu, B, Hq, Hkv, S, rule):
    """32, 8, 5, 4 and 2 pieces planned for: a call whose longest row is one step short of the rule is whole, one at it is
    split in every block of more than four steps, also in a shorter row, and a bound below the rule's own plans nothing."""
    for steps in (rule - 1, rule):
        ctx = [0, 64 * 7 - S, 64 * steps - S][-B:] if B > 1 else [64 * steps - S]
        c, qn = _case(1000 + S + steps, B, Hq, Hkv, 128, ctx, S)
        # the pools hold the chunk's keys as well: nothing is appended
        ref = O.paged_prefill_f64(qn, c.act, c.k_pool, c.v_pool, c.kv, c.block_table, c.ctx)
        got, pieces = _pieces(ff, gpu, c, qn)
        _check(got.reshape(ref.shape), ref, c.act, 2e-3)
        split = pieces.reshape(B, -1) > 1
        assert (pieces >= 1).all() and split[-1].all() == split.any() == (steps == rule)
        assert B == 1 or split[-2].any() == split.any()
        assert not split[:-2].any()
        got, pieces = _pieces(ff, gpu, c, qn, max_context_len=64 * 11)
        assert pieces is None


@pytest.mark.parametrize("B,Hq,Hkv,D,S,lo", [
    (3, 4, 2, 128, 20, 900),    # fewer groups than XCDs
    (16, 16, 4, 128, 8, 0),     # 64 group slots of an XCD, all ranked together
    (21, 6, 3, 64, 5, 0),       # groups that no XCD boundary divides
    (33, 8, 2, 64, 30, 0),
    (70, 2, 2, 64, 3, 0),       # more rows than lanes
    (13, 16, 8, 256, 9, 0),
    (30, 16, 8, 64, 2, 2400),   # rows alike: the order of the pieces
    (9, 16, 4, 128, 8, -300),   # a call that stays whole
])
def test_rows_of_many_lengths(ff, gpu, B, Hq, Hkv, D, S, lo):
    """Pieces dealt by their rows' lengths: each block's are done once, whatever the lengths and their order."""
    rng = np.random.default_rng(1100 + B)
    ctx = rng.integers(lo, 2500, size=B) if lo >= 0 else rng.integers(0, -lo, size=B)
    ctx[B // 2] = 0 if lo <= 0 else lo
    c, qn = _case(1100 + B, B, Hq, Hkv, D, [int(x) for x in ctx], S)
    ref = O.paged_prefill_f64(qn, c.act, c.k_pool, c.v_pool, c.kv, c.block_table, c.ctx)
    got, pieces = _pieces(ff, gpu, c, qn)
    _check(got.reshape(ref.shape), ref, c.act, 2e-3)
    assert (pieces >= 1).all() and (pieces > 1).any() == (lo >= 0)


def test_split_prefill_reuses_scratch(ff, gpu):
    """Calls of different sizes in a row, their scratch handed on by the allocator with the former call's contents
    (test_wide_table has a workspace of all ones)."""
    for seed, ctx, S in ((1, [3000], 8), (2, [900, 1400], 100), (3, [1300], 3)):
        c, qn = _case(960 + seed, len(ctx), 8, 2, 128, ctx, S)
        got, _, ref, split = _both(ff, gpu, c, qn, False)
        assert split
        _check(got, ref, c.act, 2e-3)


def test_split_prefill_masks(ff, gpu):
    """Absent pages across pieces (a whole piece among them) and a value that only some queries may see."""
    c, qn = _case(970, 1, 8, 2, 128, [1500], 20)
    c.block_table[0, 8:30] = -1
    c.block_table[0, 60] = c.num_blocks + 5
    got, _, ref, split = _both(ff, gpu, c, qn, False)
    assert split
    _check(got, ref, c.act, 2e-3)


def test_split_prefill_large_v(ff, gpu):
    """V beyond f16 in one piece only: that piece's rerun on bf16 products, the others' f16 tiles."""
    c, qn = _case(980, 1, 8, 2, 128, [1500], 20)
    page = int(c.block_table[0, 3])
    v = cases.decode(c.v_pool, c.kv)
    v[page, 5] *= 1e5
    c.v_pool = cases.encode(v, c.kv)
    got, _, ref, split = _both(ff, gpu, c, qn, False)
    assert split
    err = np.abs(got - ref)
    assert float((err / np.maximum(np.abs(ref), 1.0)).max()) < 1e-2


def test_unsplit_under_capture(ff, gpu):
    """A captured call allocates nothing: it runs unsplit, and its replays give the unsplit call's bits, between eager
    calls that are split."""
    import torch

    c, qn = _case(990, 1, 8, 2, 128, [1500], 20)
    q = gu.to_dev(qn, c.act, gpu)
    kp, vp = gu.to_dev(c.k_pool, c.kv, gpu), gu.to_dev(c.v_pool, c.kv, gpu)
    bt, cx = torch.from_numpy(c.block_table).to(gpu), torch.from_numpy(c.ctx).to(gpu)
    eager = ff.paged_prefill(q, kp, vp, bt, cx).clone()
    whole, out = torch.empty_like(eager), torch.empty_like(eager)
    ff.check(ff.lib.ffkv_paged_prefill(ff._ptr(q), ff._ptr(whole), ff.torch_dtype_code(q), ff._ptr(kp), ff._ptr(vp),
                                       ff.torch_dtype_code(kp), None, None, ff._ptr(bt), ff._ptr(cx), 1, 20, 8, 2, 128, 16,
                                       c.max_blocks, c.num_blocks, 0, 0.0, ff._stream(None)))
    assert not torch.equal(eager, whole)  # the eager call is split
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ff.paged_prefill(q, kp, vp, bt, cx, out=out)
        assert ff._prefill_scratch(256, q, None) is None
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, whole)
        assert torch.equal(ff.paged_prefill(q, kp, vp, bt, cx), eager)


@pytest.mark.parametrize("form", ["stream", "handle", "object", "external"])
def test_streams(ff, gpu, form):
    """Split calls that name their stream, as a torch stream, its handle, an object with one, or a stream torch did not
    make: two streams in turn, each with scratch of its own, give the current stream's bits."""
    import torch

    class Holder:
        pass

    def named(s):
        if form == "object":
            h = Holder()
            h.cuda_stream = s.cuda_stream
            return h
        return {"stream": s, "handle": s.cuda_stream, "external": torch.cuda.ExternalStream(s.cuda_stream)}[form]

    c, qn = _case(995, 1, 8, 2, 128, [1500], 20)
    d, pn = _case(996, 2, 16, 4, 128, [2000, 900], 70)
    calls = []
    for x, n in ((c, qn), (d, pn)):
        args = (gu.to_dev(n, x.act, gpu), gu.to_dev(x.k_pool, x.kv, gpu), gu.to_dev(x.v_pool, x.kv, gpu),
                torch.from_numpy(x.block_table).to(gpu), torch.from_numpy(x.ctx).to(gpu))
        B, S, Hq, D = args[0].shape
        code = ff.torch_dtype_code(args[0])
        assert ff.lib.ffkv_prefill_workspace_bytes(code, code, B, S, Hq, x.Hkv, D, 1, x.max_blocks, 0) > 0
        calls.append((args, ff.paged_prefill(*args).clone()))
    torch.cuda.synchronize()
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for i in range(12):
        args, want = calls[i % 2]
        out = torch.full_like(want, float("nan"))
        sides[i // 2 % 2].wait_stream(torch.cuda.current_stream())  # the fill
        outs.append((ff.paged_prefill(*args, out=out, stream=named(sides[i // 2 % 2])), want))
    torch.cuda.synchronize()
    assert all(torch.equal(got, want) for got, want in outs)
