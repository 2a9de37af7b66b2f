"""The decode step on quantized caches in one call: pages, codes and int8 scales byte for byte as the append kernel
writes them, outputs within the bar of the CPU checker.  Both forms of the decode after the append launch: one workgroup
per row behind the narrow table, the split behind one padded with -1.
"""

import numpy as np
import pytest

import cases
from test_gpu_append_decode import _run

pytestmark = pytest.mark.gpu


def _wide(c, blocks):
    t = np.full((c.B, blocks), -1, dtype=np.int32)
    t[:, :c.max_blocks] = c.block_table
    return t


@pytest.mark.parametrize("kv", ["i8", "fp8"])
@pytest.mark.parametrize("D,G,act", [(64, 1, "bf16"), (64, 20, "f16"), (80, 4, "bf16"), (96, 7, "f16"), (112, 2, "bf16"),
                                     (128, 4, "bf16"), (128, 17, "f32"), (256, 8, "bf16")])
def test_forms(ff, gpu, kv, D, G, act):
    """Every head_dim and source type; a group of 17 or 20 has two blocks of query heads; odd KV-head counts put two heads
    of a token on one cache line."""
    if (act, kv) == ("f16", "fp8") and D == 96:
        act = "f32"
    c = cases.make_case(6000 + D + G, 6, 3 * G, 3, D, [0, 15, 16, 31, 200, 333], act=act, kv=kv)
    for table in (c.block_table, _wide(c, 700)):
        _run(ff, gpu, c, table=table)


@pytest.mark.parametrize("kv", ["i8", "fp8"])
def test_many_rows(ff, gpu, kv):
    """Several windows of rows; many rows' ends in one wave's share of pages; 8 KV heads in workgroups of 4 or 8."""
    rng = np.random.default_rng(61)
    c = cases.make_case(6100, 150, 16, 8, 128, rng.integers(0, 300, size=150), act="bf16", kv=kv)
    for table in (c.block_table, _wide(c, 100), _wide(c, 3500)):  # row or split, split, split over a bound of more than 1 GiB
        _run(ff, gpu, c, table=table)


@pytest.mark.parametrize("kv", ["i8", "fp8"])
@pytest.mark.parametrize("cap", [16, 500, 1000])
def test_truncated(ff, gpu, kv, cap):
    """Rows cut short by max_context_len: their tokens are quantized into their slots without being attended."""
    rng = np.random.default_rng(62)
    c = cases.make_case(6200 + cap, 70, 16, 4, 128, rng.integers(200, 900, size=70), act="bf16", kv=kv)
    _run(ff, gpu, c, max_context_len=cap)


@pytest.mark.parametrize("kv", ["i8", "fp8"])
def test_absent_page_and_zero_row(ff, gpu, kv):
    """No page under a new token: nothing is written or attended; an all-zero token row has scale 0."""
    c = cases.make_case(6300, 4, 16, 4, 128, [40, 95, 200, 16], act="bf16", kv=kv)
    c.k_new[1] = 0
    c.v_new[3] = 0
    table = c.block_table.copy()
    table[0, 40 // 16] = -1
    table[2, 200 // 16] = c.num_blocks + 2
    _run(ff, gpu, c, table=table)
    wide = np.full((c.B, 600), -1, dtype=np.int32)
    wide[:, :c.max_blocks] = table
    _run(ff, gpu, c, table=wide)
