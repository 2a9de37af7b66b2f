"""The merge of a split decode at the edges of its forms: one thread per output chunk for rows of few pieces, workgroups
of 4, 8 and 16 waves per (row, head) for more.  A launch has up to 256 work items per pair of 4-head groups here, so the
batch sizes put the mean number of pieces on both sides of 4, 8 and 16; one long row among short ones has more pieces
than the mean, and rows of one piece are left to the decode kernel.  Against the CPU checker."""

import math

import numpy as np
import pytest

import cases
from test_gpu_parity import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 16, 17, 32, 33, 64, 65, 130])
def test_pieces(ff, gpu, B):
    rng = np.random.default_rng(B)
    ctx = rng.integers(40, 400, size=B)
    ctx[B // 2] = 3000
    ctx[-1] = 0
    c = cases.make_case(4000 + B, B, 16, 8, 128, ctx, act="bf16", input_scale=1 / math.sqrt(128))
    _check(ff, gpu, c, 2e-3)


@pytest.mark.parametrize("D,kv,act", [(64, "f16", "f16"), (80, "bf16", "bf16"), (256, "bf16", "bf16"),
                                      (128, "i8", "bf16"), (96, "fp8", "f32")])
@pytest.mark.parametrize("B", [2, 20, 70])
def test_pieces_head_dims(ff, gpu, D, kv, act, B):
    """head_dim 64 and 80 leave lanes of a wave with one dim or none, 256 gives them four."""
    rng = np.random.default_rng(D + B)
    c = cases.make_case(4100 + D + B, B, 6, 2, D, rng.integers(1, 900, size=B), act=act, kv=kv,
                        input_scale=1 / math.sqrt(D))
    _check(ff, gpu, c, 2e-3 if kv in ("bf16", "f16") else 2e-2)


@pytest.mark.parametrize("B,Hq,Hkv,D,ctx,kv", [
    (1, 10, 2, 64, 20000, "bf16"), (2, 10, 2, 64, 5900, "f16"), (3, 8, 2, 128, 5897, "bf16"),
    (1, 32, 8, 128, 9000, "i8"), (21, 10, 2, 64, 1500, "bf16"), (22, 10, 2, 64, 1500, "bf16")])
def test_few_long_rows(ff, gpu, B, Hq, Hkv, D, ctx, kv):
    """Fewer work items than workgroups fit the chip, by the rows' pages: above and below the least of them per row (96, 369
    pages), and where the rows are as many that it limits nothing."""
    act = "f16" if kv == "f16" else "bf16"
    c = cases.make_case(4300 + B + D, B, Hq, Hkv, D, [ctx - 17 * (b % 7) for b in range(B)], act=act, kv=kv,
                        input_scale=1 / math.sqrt(D))
    _check(ff, gpu, c, 2e-2 if kv == "i8" else 2e-3)


def test_few_long_rows_workspace(ff, gpu):
    """The bound on work items leaves the workspace's limit where it is without: one that only the bounded items' partials
    would fit is refused."""
    import torch

    B, Hq, Hkv, D, blocks = 1, 10, 2, 64, 1250  # 5 sqrt(1250) = 176 of at least 1024 resident workgroups
    q = torch.zeros((B, 1, Hq, D), dtype=torch.bfloat16, device=gpu)
    k = torch.zeros((1, 16, Hkv, D), dtype=torch.bfloat16, device=gpu)
    table = torch.full((B, blocks), -1, dtype=torch.int32, device=gpu)
    ctx = torch.full((B,), 19999, dtype=torch.int32, device=gpu)
    ws = torch.empty((176 + B + 8) * Hq * (D + 2) * 4 + 4096, dtype=torch.uint8, device=gpu)
    with pytest.raises(ff.FFKVError):
        ff.paged_attention(q, k, k, table, ctx, workspace=ws)
    out = ff.paged_attention(q, k, k, table, ctx, workspace=ff.decode_workspace(B, Hq, D, blocks, device=gpu))
    torch.cuda.synchronize()
    assert not out.any()
