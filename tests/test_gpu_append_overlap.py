"""The decode step in one call where rows attend each other's new tokens: several consecutive tokens of one sequence, each
a row over the same block table (as a draft is verified).  Every token is in its page before any row attends it, so the
call equals the append followed by the decode.  (16-bit caches fed in their own type write the tokens in the decode's own
launch and ask for slots of their own; their rows here come in another type.)
"""

import numpy as np
import pytest

import cases
from test_gpu_append_decode import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,kv", [("f32", "f32"), ("bf16", "i8"), ("f32", "i8"), ("bf16", "fp8"), ("f32", "bf16")])
@pytest.mark.parametrize("D,G", [(128, 4), (64, 16), (88, 2)])
@pytest.mark.parametrize("base", [0, 90, 1270])
def test_rows_of_one_sequence(ff, gpu, act, kv, D, G, base):
    """Eight rows from token `base` on (90: over the end of a page; 1270: of the vector kernel's chunk of 256 tokens),
    behind their own table and a wide one."""
    ctx = base + np.arange(8)
    c = cases.make_case(9000 + base + D, 8, 2 * G, 2, D, ctx, act=act, kv=kv, shared_prefix_blocks=int(ctx[-1]) // 16 + 1)
    assert (c.block_table[:, 0] == c.block_table[0, 0]).all()
    wide = np.full((c.B, 600), -1, dtype=np.int32)
    wide[:, :c.max_blocks] = c.block_table
    for table in (c.block_table, wide):
        _run(ff, gpu, c, table=table)
