"""The decode step in one call on the vector kernel (fp32 pages, and head dims that the matrix cores do not take): the
append kernel, then the decode.  Pages byte for byte as the append kernel writes them, outputs within the bar of the CPU
checker."""

import numpy as np
import pytest

import cases
from test_gpu_append_decode import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,G,act", [(128, 4, "f32"), (64, 1, "f32"), (256, 16, "f32"), (8, 2, "f32"), (88, 8, "f32"),
                                     (88, 5, "bf16"), (40, 2, "f16")])
def test_forms(ff, gpu, D, G, act):
    """The new token first or last in its page and its chunk of 256 tokens, in a one-token row, and after none."""
    ctx = [0, 15, 16, 254, 255, 256, 257, 700, -1]
    c = cases.make_case(7000 + D + G, len(ctx), 2 * G, 2, D, ctx, act=act)
    _run(ff, gpu, c)


@pytest.mark.parametrize("cap", [16, 300, 1000])
def test_truncated(ff, gpu, cap):
    c = cases.make_case(7100 + cap, 6, 16, 4, 128, [15, 16, 299, 300, 301, 900], act="f32")
    _run(ff, gpu, c, max_context_len=cap)


def test_absent_pages(ff, gpu):
    c = cases.make_case(7200, 4, 16, 4, 128, [40, 95, 200, 16], act="f32")
    table = c.block_table.copy()
    table[0, 40 // 16] = -1
    table[2, 200 // 16] = c.num_blocks + 2
    table[3, :] = -1
    _run(ff, gpu, c, table=table)


@pytest.mark.parametrize("act,kv", [("bf16", "f32"), ("f32", "bf16")])
def test_other_source_types(ff, gpu, act, kv):
    """Tokens of another type than the cache's: the append kernel, then the decode."""
    rng = np.random.default_rng(73)
    c = cases.make_case(7300, 5, 16, 4, 128, rng.integers(0, 600, size=5), act=act, kv=kv)
    _run(ff, gpu, c)


@pytest.mark.parametrize("D,act,kv", [(88, "bf16", "i8"), (40, "bf16", "fp8"), (88, "f32", "fp8")])
@pytest.mark.parametrize("cap", [0, 16, 300])
def test_quantized(ff, gpu, D, act, kv, cap):
    """8-bit pages of the vector kernel's head dims, with and without rows cut short by max_context_len."""
    c = cases.make_case(7400 + D, 6, 8, 2, D, [15, 16, 299, 300, 301, 700], act=act, kv=kv)
    _run(ff, gpu, c, max_context_len=cap)
