"""Decode over fp32 pages: the lanes' split of a row's dims over its two halves, the loads that go past the caches
(rows with pages of their own) and those that do not (rows that share their first pages), and the merge of one to many
chunks (chunks of 256 tokens here, merged eight at a time).  Against the CPU checker, 1e-4 as in test_gpu_parity.py.
"""

import math

import numpy as np
import pytest

import cases
from test_gpu_parity import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,G,ctx", [
    (128, 4, [0, 255, 256, 2046, 2047, 2048, 2049, 4200]),  # 1, 1, 2, 8, 8, 9, 9 and 17 chunks
    (64, 1, [300, 2100]),
    (256, 8, [17, 700, 1025]),
    (8, 2, [600, 5]),
    (88, 16, [515, 2300]),
])
def test_decode_f32(ff, gpu, D, G, ctx):
    c = cases.make_case(700 + D + G, len(ctx), 2 * G, 2, D, ctx, act="f32", input_scale=1 / math.sqrt(D))
    _check(ff, gpu, c, 1e-4)


@pytest.mark.parametrize("shared", [1, 20])
def test_decode_f32_shared_pages(ff, gpu, shared):
    """Rows that share their first pages with a neighbour, and one in between that ends inside them."""
    c = cases.make_case(720 + shared, 5, 16, 4, 128, [700, 16 * shared - 1, 900, 333, 16 * shared + 1], act="f32",
                        input_scale=1 / math.sqrt(128), shared_prefix_blocks=shared)
    c.ctx[1] = 16 * shared - 2  # its new token stays out of the shared pages' last slot
    _check(ff, gpu, c, 1e-4)


@pytest.mark.parametrize("B", [6, 300])
def test_decode_f32_prefixes_in_turn(ff, gpu, B):
    """Rows over two prefixes in turn, so that no row shares pages with its neighbours, and rows of their own at the ends;
    more rows than one workgroup looks at."""
    ctx = [330 + 16 * (b % 3) for b in range(B)]
    c = cases.make_case(730 + B, B, 4, 2, 64, ctx, act="f32", input_scale=1 / 8)
    for b in range(3, B - 2):
        c.block_table[b, :18] = c.block_table[1 + b % 2, :18]
    _check(ff, gpu, c, 1e-4)


@pytest.mark.parametrize("kv,tol", [("bf16", 2e-3), ("i8", 2e-2)])
def test_vector_decode_merge(ff, gpu, kv, tol):
    """The same merge behind the vector kernel's other caches (head_dim 88)."""
    c = cases.make_case(740, 3, 12, 3, 88, [2047, 90, 3000], act="bf16", kv=kv, input_scale=1 / math.sqrt(88))
    _check(ff, gpu, c, tol)


@pytest.mark.parametrize("act,kv,G,D", [("f32", "f32", 8, 128), ("f32", "f32", 5, 64), ("f32", "f32", 2, 80),
                                        ("bf16", "bf16", 8, 88), ("bf16", "i8", 1, 40), ("f32", "f32", 3, 128)])
def test_absent_pages_read_nothing(ff, gpu, act, kv, G, D):
    """Page 0, which tokens of no page may load from, holds NaN and belongs to no row: no output shows it, a row without
    any page is zero."""
    c = cases.make_case(750 + D + G, 4, 2 * G, 2, D, [500, 37, 300, 64], act=act, kv=kv, input_scale=1 / math.sqrt(D))
    c.block_table[c.block_table == 0] = -1
    c.block_table[0, 5:9] = -1
    c.block_table[0, 12] = c.num_blocks
    c.block_table[3, :] = -1
    if kv == "i8":
        c.k_scale[0] = c.v_scale[0] = np.nan
    else:
        c.k_pool[0] = c.v_pool[0] = np.nan if kv == "f32" else 0x7FC0
    _check(ff, gpu, c, 2e-2 if kv == "i8" else 2e-3 if kv == "bf16" else 1e-4)
