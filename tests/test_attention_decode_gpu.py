"""The few-rows attention path (attention_decode.hip: at most 16 new tokens and
64 query rows per KV head) against the oracle's float64 softmax(S) V, at the
edges of its row blocks, key tiles and chunks, and over every way a new row
reaches a tile: appended in the launch (aligned K / V, at most 32 rows) or by
the separate append, plain and ring caches, each dtype pair. Held to the tier
the flash kernel is held to: operands and probabilities enter as fp16."""
import ctypes

import numpy as np
import pytest

from helpers import FP16, assert_close, draw
from oracle import oracle
from test_attention_gpu import _cache_planes

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


@pytest.mark.parametrize("b, hq, hkv, tq, tkv, d, causal, span, dt, odt", [
    (1, 1, 1, 1, 1, 64, True, 0, F16, F32),          # one key
    (1, 4, 4, 1, 32, 64, False, 0, F16, F32),        # one whole tile
    (1, 4, 1, 4, 129, 128, True, 0, F16, F32),       # 16 rows; one key past the first unit's four tiles
    (1, 17, 1, 1, 500, 64, False, 0, F16, F16),      # 17 rows: the 32-row kernel
    (1, 4, 1, 16, 1000, 64, True, 0, F16, F32),      # 64 rows in two blocks
    (1, 5, 1, 13, 700, 128, True, 0, F16, F32),      # 65 rows: past the path's last
    (1, 2, 2, 17, 700, 64, True, 0, F16, F32),       # 17 tokens: past the path's last
    (3, 6, 2, 2, 333, 72, False, 0, F16, F32),       # batch, head dim padded to 128
    (2, 4, 2, 5, 4100, 16, True, 0, F32, F32),       # smallest head dim, fp32
    (1, 8, 1, 8, 2500, 256, True, 0, F32, F16),      # D = 256 in 16-row blocks, fp32
    (1, 4, 2, 3, 900, 200, True, 100, F16, F32),     # window, padded D = 256
    (1, 2, 1, 9, 5, 64, True, 0, F16, F32),          # Tq > Tkv: four queries see no key
    (40, 8, 8, 1, 600, 64, False, 0, F16, F16),      # no workspace: the heads alone fill the GPU
])
def test_decode_rows(gpu, b, hq, hkv, tq, tkv, d, causal, span, dt, odt):
    rng = np.random.default_rng(d + tkv)
    q, k, v = draw((b, hq, tq, d), rng, dt), draw((b, hkv, tkv, d), rng, dt), draw((b, hkv, tkv, d), rng, dt)
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((b, tq, hq, d), odt)
    print(f"decode rows b={b} hq={hq} hkv={hkv} tq={tq} tkv={tkv} d={d} span={span}", flush=True)
    got = gpu.attention(out, D(q), D(k), D(v), causal=causal, span=span).numpy().astype(np.float32)
    want = oracle.attention(q, k, v, causal=causal, span=span, out_dtype=np.float32)
    assert_close(got, want, FP16)


@pytest.mark.parametrize("d, hq, hkv, tq, tkv, count, size, ring, span, cdt, kdt", [
    (64, 8, 2, 1, 1, 0, 4096, False, 0, F16, F16),       # an empty cache: one unit of many has work
    (64, 8, 2, 1, 1, 31, 4096, False, 0, F16, F16),      # the new row ends a tile
    (64, 8, 2, 1, 1, 32, 4096, False, 0, F16, F16),      # ... starts one
    (128, 4, 2, 16, 16, 120, 1024, False, 0, F16, F32),  # new rows over two tiles and two units, converted
    (128, 4, 2, 3, 3, 253, 256, False, 0, F16, F16),     # the cache filled to its last row
    (64, 4, 4, 2, 32, 100, 512, False, 0, F32, F16),     # more new keys than queries, fp16 rows into an fp32 cache
    (64, 4, 4, 2, 33, 100, 512, False, 0, F16, F16),     # too many new rows to append in the launch
    (64, 4, 2, 8, 8, 252, 256, True, 60, F16, F16),      # the new rows wrap the ring
    (128, 4, 2, 5, 5, 1000, 64, True, 30, F32, F32),     # the smallest ring, wrapped many times
    (72, 4, 1, 4, 4, 700, 1024, False, 300, F16, F32),   # window, padded head dim
    (256, 8, 1, 2, 2, 3000, 8192, False, 0, F16, F16),   # many units at D = 256
])
def test_decode_cache(gpu, d, hq, hkv, tq, tkv, count, size, ring, span, cdt, kdt):
    rng = np.random.default_rng(count + size + d)
    kc, vc = _cache_planes(rng, hkv, size, d, count, ring, cdt)
    q = draw((1, hq, tq, d), rng, F16)
    k, v = draw((1, hkv, tkv, d), rng, kdt), draw((1, hkv, tkv, d), rng, kdt)
    D = gpu.DeviceArray.from_numpy
    dkc, dvc = D(kc), D(vc)
    out = gpu.DeviceArray((1, tq, hq, d), F32)
    print(f"decode cache d={d} hq={hq} hkv={hkv} tq={tq} tkv={tkv} count={count} size={size} ring={ring}", flush=True)
    got = gpu.attention(out, D(q), D(k), D(v), causal=True, span=span,
                        cache=(dkc, dvc, D(np.array([count], np.uint32)), ring)).numpy()
    want, wkc, wvc = oracle.attention_cached(q[0], k, v, kc, vc, count, ring=ring, causal=True, span=span)
    assert_close(got[0], want, FP16)
    np.testing.assert_array_equal(dkc.numpy(), wkc)
    np.testing.assert_array_equal(dvc.numpy(), wvc)


def test_decode_cache_unaligned_new_rows(gpu):
    """New rows that are not 16-byte aligned are appended by the separate launch."""
    rng = np.random.default_rng(3)
    hq, hkv, d, size, count = 4, 2, 64, 256, 77
    kc, vc = _cache_planes(rng, hkv, size, d, count, False, F16)
    q, k, v = draw((1, hq, 1, d), rng, F16), draw((1, hkv, 1, d), rng, F16), draw((1, hkv, 1, d), rng, F16)
    D = gpu.DeviceArray.from_numpy
    pad = np.zeros(1, F16)
    dk, dv = D(np.concatenate([pad, k.ravel()])), D(np.concatenate([pad, v.ravel()]))
    dkc, dvc, dq, cnt = D(kc), D(vc), D(q), D(np.array([count], np.uint32))
    out = gpu.DeviceArray((1, 1, hq, d), F32)
    a = gpu.attention_args(out, dq, D(k), D(v), causal=True, cache=(dkc, dvc, cnt, False))
    a.k, a.v = dk.ptr + 2, dv.ptr + 2
    need = gpu.lib().vai_attention_workspace_size(ctypes.byref(a))
    ws = gpu.DeviceArray((max(need, 1),), np.uint8)
    a.workspace, a.workspace_bytes = ws.ptr, ws.nbytes
    gpu.check(gpu.lib().vai_attention_launch(ctypes.byref(a), None), "attention")
    gpu.synchronize()
    want, wkc, wvc = oracle.attention_cached(q[0], k, v, kc, vc, count, causal=True)
    assert_close(out.numpy()[0], want, FP16)
    np.testing.assert_array_equal(dkc.numpy(), wkc)
    np.testing.assert_array_equal(dvc.numpy(), wvc)


def test_decode_graph_follows_the_count(gpu):
    """One recorded step replayed while the count grows past a unit's keys:
    the kernels read the count when they run."""
    rng = np.random.default_rng(9)
    hq, hkv, d, size = 8, 2, 64, 1024
    kc, vc = _cache_planes(rng, hkv, size, d, 600, False, F16)
    q, k, v = draw((1, hq, 1, d), rng, F16), draw((1, hkv, 1, d), rng, F16), draw((1, hkv, 1, d), rng, F16)
    D = gpu.DeviceArray.from_numpy
    dkc, dvc, dq, dk, dv = D(kc), D(vc), D(q), D(k), D(v)
    cnt, out = gpu.DeviceArray((1,), np.uint32), gpu.DeviceArray((1, 1, hq, d), F32)
    cnt.fill_(0)
    a = gpu.attention_args(out, dq, dk, dv, causal=True, cache=(dkc, dvc, cnt, False))
    need = gpu.lib().vai_attention_workspace_size(ctypes.byref(a))
    ws = gpu.DeviceArray((max(need, 1),), np.uint8)
    a.workspace, a.workspace_bytes = ws.ptr, ws.nbytes
    gpu.synchronize()
    stream = gpu.Stream()
    graph = gpu.Graph(stream, lambda: gpu.check(gpu.lib().vai_attention_launch(ctypes.byref(a), stream.ptr), "step"))
    for count in (0, 5, 127, 128, 600, 40):
        gpu.lib().vai_memcpy_h2d(cnt.ptr, np.array([count], np.uint32).ctypes.data, 4, None)
        gpu.lib().vai_memcpy_h2d(dkc.ptr, kc.ctypes.data, kc.nbytes, None)
        gpu.lib().vai_memcpy_h2d(dvc.ptr, vc.ctypes.data, vc.nbytes, None)
        graph.launch()
        stream.synchronize()
        want, wkc, _ = oracle.attention_cached(q[0], k, v, kc, vc, count, causal=True)
        assert_close(out.numpy()[0], want, FP16)
        np.testing.assert_array_equal(dkc.numpy(), wkc)
