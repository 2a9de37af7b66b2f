"""The native Python front end without a GPU: what it reads from its tensors, and the errors it hands on.  Calls that
need no launch (empty batches) or that the library rejects return before touching a device; ``stream`` is given, since
there is no current one."""

import threading

import numpy as np
import pytest
import torch

HKV, D = 2, 64


def _args(B=0, S=1, dtype=torch.bfloat16, cache=torch.bfloat16):
    k = torch.zeros(B, S, HKV, D, dtype=dtype)
    pool = torch.zeros(4, 16, HKV, D, dtype=cache)
    return k, k.clone(), pool, pool.clone(), torch.zeros(B, 3, dtype=torch.int32), torch.zeros(B, dtype=torch.int32)


class Stream:
    cuda_stream = 0


@pytest.mark.parametrize("stream", [0, Stream()])
def test_empty_batch(ff, stream):
    k, v, kc, vc, bt, cx = _args()
    q = torch.zeros(0, 1, 2 * HKV, D, dtype=torch.bfloat16)
    ff.append_kv_cache(k, v, kc, vc, bt, cx, stream=stream)
    ff.apply_rope(q, k, cx, stream=stream)
    ff.apply_rope(None, k, None, theta=10, stream=stream)
    ff.rope_append_kv_cache(q, k, v, kc, vc, bt, cx, stream=stream)
    ws = torch.zeros(256, dtype=torch.uint8)
    for out in (ff.paged_attention(q, kc, vc, bt, cx, stream=stream),
                ff.paged_attention(q[:, 0], kc, vc, bt, cx, workspace=ws, num_blocks=2, stream=stream),
                ff.append_paged_attention(k, v, q, kc, vc, bt, cx, stream=stream),
                ff.paged_attention_shared_prefix(q, kc, vc, bt, cx, 1, stream=stream)):
        assert out.shape == (0, 1, 2 * HKV * D) and out.dtype == q.dtype
    given = torch.empty(0, 1, 2 * HKV * D, dtype=q.dtype)
    assert ff.paged_attention_noalloc(q, kc, vc, bt, cx, given, stream=stream) is given
    assert ff.paged_prefill(q, kc, vc, bt, cx, out=given, stream=stream) is given
    assert ff.paged_prefill(q, k, v, None, None, stream=stream).shape == (0, 1, 2 * HKV * D)


def test_library_errors(ff):
    k, v, kc, vc, bt, cx = _args(B=1)
    q = torch.zeros(1, 1, 3 * HKV + 1, D, dtype=torch.bfloat16)
    with pytest.raises(ff.FFKVError, match="multiple of num_kv_heads"):
        ff.paged_attention(q, kc, vc, bt, cx, stream=0)
    with pytest.raises(ff.FFKVError, match="k_scale"):
        ff.append_kv_cache(k, v, kc.to(torch.int8), vc.to(torch.int8), bt, cx, stream=0)
    with pytest.raises(ff.FFKVError, match="16-byte aligned"):
        ff.append_kv_cache(torch.zeros(HKV * D + 1, dtype=k.dtype)[1:].view(1, 1, HKV, D), v, kc, vc, bt, cx, stream=0)
    with pytest.raises(ff.FFKVError, match="shared_blocks 7"):
        ff.paged_attention_shared_prefix(q[:, :, :4].contiguous(), kc, vc, bt, cx, 7, stream=0)


def test_argument_errors(ff):
    k, v, kc, vc, bt, cx = _args()
    with pytest.raises(TypeError, match="unsupported dtype torch.float64"):
        ff.append_kv_cache(k.double(), v, kc, vc, bt, cx, stream=0)
    with pytest.raises(ValueError, match="not enough values"):
        ff.append_kv_cache(k[0:0, 0], v, kc, vc, bt, cx, stream=0)
    with pytest.raises(IndexError):
        ff.paged_attention(k, kc[0, 0], vc, bt, cx, stream=0)
    with pytest.raises(AttributeError):
        ff.append_kv_cache(k, v, kc, vc, [[0]], cx, stream=0)
    with pytest.raises(TypeError):
        ff.append_kv_cache(k, v, kc, vc, bt, cx, num_blocks="4", stream=0)
    with pytest.raises((TypeError, ValueError)):
        ff.append_kv_cache(k, v, kc, vc, bt, cx, stream="x")


@pytest.mark.parametrize("n", [4.0, torch.tensor(4), np.int64(4)])
def test_integers_are_ints(ff, n):
    """num_blocks and max_context_len take a Python int (or a bool), as ctypes' c_int does, and no value that converts to
    one; scale and theta take what float() takes."""
    k, v, kc, vc, bt, cx = _args()
    q = torch.zeros(0, 1, 2 * HKV, D, dtype=torch.bfloat16)
    with pytest.raises(TypeError):
        ff.append_kv_cache(k, v, kc, vc, bt, cx, num_blocks=n, stream=0)
    with pytest.raises(TypeError):
        ff.paged_attention(q, kc, vc, bt, cx, max_context_len=n, stream=0)
    ff.append_kv_cache(k, v, kc, vc, bt, cx, num_blocks=True, stream=0)
    ff.paged_attention(q, kc, vc, bt, cx, scale=n, stream=0)
    ff.paged_attention(q, kc, vc, bt, cx, scale="0.5", stream=0)
    ff.apply_rope(q, k, cx, theta=n, stream=0)
    with pytest.raises(ValueError):
        ff.paged_attention(q, kc, vc, bt, cx, scale="x", stream=0)


def test_prefill_scratch_without_memory(ff, monkeypatch):
    """No memory for a split prefill's scratch: the call runs unsplit, as it does while its stream is captured."""
    def full(*a, **kw):
        raise torch.OutOfMemoryError("full")

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert ff._prefill_scratch(64, torch.empty(1), None).numel() == 64
    monkeypatch.setattr(torch, "empty", full)
    assert ff._prefill_scratch(64, torch.zeros(1), None) is None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: pytest.fail("allocated under capture"))
    assert ff._prefill_scratch(64, torch.zeros(1), None) is None


def test_threads(ff):
    """The interpreter lock is given up around the library's call; its error message is the calling thread's."""
    k, v, kc, vc, bt, cx = _args(B=1)
    seen = []

    def work(i):
        q = torch.zeros(1, 1, HKV * 2 + 1, D, dtype=torch.bfloat16) if i % 2 else None
        for _ in range(200):
            try:
                if i % 2:
                    ff.paged_attention(q, kc, vc, bt, cx, stream=0)
                else:
                    ff.append_kv_cache(k, v, kc.to(torch.int8), vc.to(torch.int8), bt, cx, stream=0)
            except ff.FFKVError as e:
                seen.append(("num_kv_heads" if i % 2 else "k_scale") in str(e))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert len(seen) == 800 and all(seen)
