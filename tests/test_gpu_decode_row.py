"""The decode of a small batch in one launch (a workgroup per row and KV head), against the CPU checker and against the
split decode, at the edges of the rule that chooses between them.

The rule goes by the bound on the row length (the table's width, or max_context_len): the same rows behind a table
padded with -1 to 8192 tokens take the split decode.  Both lie within the bar of the checker, so they differ by twice
that at most.
"""

import numpy as np
import pytest

import cases
import gpu_util as gu
import oracle as O
from test_gpu_append_decode import _run
from test_gpu_parity import TOL, _check, half_ulp

pytestmark = pytest.mark.gpu
NAME = {O.DTYPE_F32: "f32", O.DTYPE_F16: "f16", O.DTYPE_BF16: "bf16", O.DTYPE_I8: "i8", O.DTYPE_FP8: "fp8"}


def _both_routes(ff, dev, c, max_context_len=0):
    """Decode over the case's own table and, without max_context_len, over one padded to 512 blocks; each against the
    checker."""
    import torch

    wide = np.full((c.B, 512), -1, dtype=np.int32)
    wide[:, :c.max_blocks] = c.block_table
    kp, vp = c.k_pool.copy(), c.v_pool.copy()
    ks = None if c.k_scale is None else c.k_scale.copy()
    vs = None if c.v_scale is None else c.v_scale.copy()
    O.append(c.k_new, c.v_new, c.act, kp, vp, c.kv, c.block_table, c.ctx, ks, vs)
    _, ref = O.paged_decode(c.q, c.act, kp, vp, c.kv, c.block_table, c.ctx, ks, vs, max_context_len=max_context_len)
    up = lambda x: None if x is None else torch.from_numpy(x).to(dev)
    dk, dv, q = gu.to_dev(kp, c.kv, dev), gu.to_dev(vp, c.kv, dev), gu.to_dev(c.q, c.act, dev)
    got = []
    for table in (c.block_table, wide)[:1 if max_context_len else 2]:
        out = torch.full((c.B, 1, c.Hq * c.D), float("nan"), dtype=q.dtype, device=dev)
        ff.paged_attention(q, dk, dv, up(np.ascontiguousarray(table)), up(c.ctx), out=out, k_scale=up(ks), v_scale=up(vs),
                           max_context_len=max_context_len, num_blocks=c.num_blocks)
        got.append(out.float().cpu().numpy().reshape(ref.shape).astype(np.float64))
    tol = TOL.get((NAME[c.act], NAME[c.kv]), 2e-3)
    for g in got:
        excess = np.abs(g - ref) - half_ulp(np.maximum(np.abs(g), np.abs(ref)), c.act)
        assert float(excess.max()) <= tol
    if max_context_len == 0:
        d = np.abs(got[0] - got[1]) - 2 * half_ulp(np.maximum(*map(np.abs, got)), c.act)
        assert float(d.max()) <= 2 * tol


@pytest.mark.parametrize("act,kv", [("bf16", "bf16"), ("f16", "f16"), ("f32", "bf16"), ("bf16", "f16"), ("bf16", "i8"),
                                    ("f16", "i8"), ("bf16", "fp8"), ("f32", "fp8")])
@pytest.mark.parametrize("D,G", [(64, 1), (80, 4), (96, 7), (112, 2), (128, 4), (128, 20), (256, 16)])
def test_row_forms(ff, gpu, act, kv, D, G):
    """Rows of no page, one page, fewer pages than waves, as many, and more, at every head_dim; a group of 20 takes two
    blocks of query heads."""
    c = cases.make_case(5000 + D + G, 7, 2 * G, 2, D, [-1, 0, 15, 16, 100, 127, 249], act=act, kv=kv,
                        input_scale=1 / np.sqrt(D), max_blocks=16)
    _both_routes(ff, gpu, c)


@pytest.mark.parametrize("B,tokens", [(1, 511), (1, 512), (16, 1023), (16, 1024), (32, 1000), (33, 1000), (64, 511),
                                      (65, 511)])
def test_rule_edges(ff, gpu, B, tokens):
    """512 and 1024 tokens of bf16 at head_dim 128 are the 256 and 512 KiB of the rule; 16 rows of 8 KV heads are its
    128 workgroups, 32 its 256, 64 its 512."""
    ctx = np.full(B, tokens)
    ctx[B // 2:] //= 3
    c = cases.make_case(5100 + B, B, 8, 8, 128, ctx, act="bf16", input_scale=1 / np.sqrt(128))
    _both_routes(ff, gpu, c)


@pytest.mark.parametrize("cap", [16, 130, 400])
def test_truncated(ff, gpu, cap):
    """Rows longer than max_context_len, in the plain decode and with the new token appended (it is written to its slot
    without being attended)."""
    c = cases.make_case(5200 + cap, 9, 16, 8, 128, [3, 129, 130, 131, 399, 400, 401, 15, 16], act="bf16")
    _both_routes(ff, gpu, c, max_context_len=cap)
    _run(ff, gpu, c, max_context_len=cap)


def test_absent_pages(ff, gpu):
    """Absent pages at the start, between and at the end of rows, one row of nothing else, and one under a new token."""
    c = cases.make_case(5300, 5, 16, 8, 128, [200, 310, 90, 64, 47], act="bf16")
    c.block_table[0, 0] = -1
    c.block_table[1, 3:9] = c.num_blocks + 1
    c.block_table[2, 90 // 16] = -1
    c.block_table[3, :] = -1
    _both_routes(ff, gpu, c)
    _run(ff, gpu, c)


def test_any_workspace(ff, gpu):
    """The one launch writes no partials, but a workspace that the split would refuse is refused here too, and none
    given is none allocated under capture."""
    import torch

    c = cases.config1(act="bf16")
    _check(ff, gpu, c, 2e-3, workspace=True)
    q, dk, dv = gu.to_dev(c.q, c.act, gpu), gu.to_dev(c.k_pool, c.kv, gpu), gu.to_dev(c.v_pool, c.kv, gpu)
    bt, cx = torch.from_numpy(c.block_table).to(gpu), torch.from_numpy(c.ctx).to(gpu)
    with pytest.raises(ff.FFKVError, match="smaller than"):
        ff.paged_attention(q, dk, dv, bt, cx, workspace=torch.empty(64, dtype=torch.uint8, device=gpu))
    eager = ff.paged_attention(q, dk, dv, bt, cx).clone()
    out = torch.empty_like(eager)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ff.paged_attention(q, dk, dv, bt, cx, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        ff.paged_attention(q, dk, dv, bt, cx)
