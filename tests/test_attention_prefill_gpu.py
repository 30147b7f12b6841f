"""Prefill attention at the edges of its workgroup order and tiles, against
float64. Bound, with A = sum p |v| of the row: P is rounded to fp16 (2^-11 A), a
score's D products are summed in fp32 (D 2^-24 sum |q k| scale, which moves p
and 1 / l by that much each), exp2 and the sums over keys (32 + T / 64 steps of
2^-24 each side), and the output rounding."""
import numpy as np
import pytest

from helpers import draw

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


@pytest.mark.parametrize("b, hq, hkv, tq, tkv, d, causal, span, odt", [
    (1, 256, 32, 130, 130, 64, True, 0, F32),      # a multiple of 8 pairs, unsplit, two query tiles
    (2, 132, 44, 129, 129, 64, True, 0, F16),      # 264 pairs of two batches
    (1, 150, 50, 300, 300, 128, True, 0, F16),     # pairs not a multiple of 8: heads spread over the XCDs
    (1, 131, 131, 257, 200, 128, True, 0, F32),    # rows that see no key
    (1, 90, 30, 385, 450, 128, False, 0, F32),     # no mask, a key tail of two rows
    (1, 72, 24, 520, 520, 80, True, 70, F16),      # window, padded head dim
    (3, 43, 43, 300, 300, 256, True, 0, F32),
    (1, 24, 8, 1000, 1000, 128, True, 0, F32),     # fewer tiles than CUs: split
    (1, 24, 8, 1400, 1400, 128, True, 0, F32),     # two wave groups share the keys, unsplit, odd and even walks
    (1, 40, 40, 833, 900, 64, True, 0, F16),
    (1, 2, 2, 640, 640, 72, False, 0, F32),        # ... and split
    (1, 16, 2, 256, 2111, 128, True, 0, F16),      # long walks, an odd number of tiles
    (1, 4, 4, 64, 65, 64, False, 0, F32),
    (1, 2, 2, 100, 64, 128, False, 0, F16),        # one key tile
])
def test_prefill(gpu, b, hq, hkv, tq, tkv, d, causal, span, odt):
    rng = np.random.default_rng(tq + d + hq)
    q, k, v = (draw((b, h, t, d), rng, F16) for h, t in ((hq, tq), (hkv, tkv), (hkv, tkv)))
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((b, tq, hq, d), odt)
    out.fill_(0xFF)
    print(f"prefill b={b} hq={hq} hkv={hkv} tq={tq} tkv={tkv} d={d} causal={causal} span={span}", flush=True)
    got = gpu.attention(out, D(q), D(k), D(v), causal=causal, span=span).numpy().astype(np.float64)
    i, j = np.arange(tq)[:, None] + (tkv - tq), np.arange(tkv)[None, :]
    vis = (j <= i) if causal else np.ones((tq, tkv), bool)
    if span:
        vis = vis & (j > i - span)
    none = ~vis.any(axis=1)
    e = 2.0 ** -24
    for bb in range(b):
        for h in list(range(0, hq, max(1, hq // 9))) + [hq - 1]:
            q64, k64, v64 = (x.astype(np.float64) for x in (q[bb, h], k[bb, h // (hq // hkv)], v[bb, h // (hq // hkv)]))
            s = np.where(vis, q64 @ k64.T / np.sqrt(d), -np.inf)
            mx = np.where(none, 0.0, s.max(axis=1, initial=-np.inf))
            p = np.exp(s - mx[:, None])
            p /= np.maximum(p.sum(axis=1, keepdims=True), 1e-300)
            y, A = p @ v64, p @ np.abs(v64)
            err = d * e * (np.abs(q64) @ np.abs(k64).T / np.sqrt(d)).max() + (32 + tkv / 64 + 8) * e
            tol = A * (2.0 ** -11 + 2 * err) + (2.0 ** -11 * np.abs(y) if odt == F16 else 0) + 2.0 ** -24
            if odt == F16 and tkv > 64:
                tol = tol + 2.0 ** -10 * A       # split walks: partials rounded to fp16 before they are merged
            r = got[bb, :, h]
            assert np.isfinite(r).all() and (np.abs(r - y) <= tol).all(), (h, float((np.abs(r - y) / tol).max()))
            assert (r[none] == 0).all()


@pytest.mark.parametrize("hq, hkv, t, d", [(2, 1, 200, 64), (24, 8, 1400, 128), (3, 3, 300, 256)])
def test_prefill_nan_key(gpu, hq, hkv, t, d):
    """A NaN score makes its own row NaN and no other: the rows before the key
    (they may share a wave, and so the moves of the running maximum, with NaN
    rows) stay within two roundings of P to fp16, other KV heads keep their bits."""
    rng = np.random.default_rng(t)
    q, k, v = (draw((1, h, t, d), rng, F16) for h in (hq, hkv, hkv))
    D = gpu.DeviceArray.from_numpy
    outs = []
    j = t // 2 + 3
    for bad in (False, True):
        if bad:
            k[0, 0, j, 5] = np.nan
        out = gpu.DeviceArray((1, t, hq, d), F32)
        out.fill_(0xFF)
        print(f"prefill nan={bad} hq={hq} t={t} d={d}", flush=True)
        outs.append(gpu.attention(out, D(q), D(k), D(v), causal=True).numpy())
    g = hq // hkv
    assert np.isfinite(outs[0]).all()
    assert np.isnan(outs[1][0, j:, :g]).all()
    assert np.allclose(outs[1][0, :j], outs[0][0, :j], rtol=0, atol=2.0 ** -10 * np.abs(v.astype(F32)).max())
    assert (outs[1][0, :, g:] == outs[0][0, :, g:]).all()


@pytest.mark.parametrize("d, count", [(64, 0), (128, 0), (128, 12), (128, 70), (64, 200)])
def test_prefill_into_a_large_cache(gpu, d, count):
    """A chunk over a cache that holds little of what it was made for: planned in long walks for two wave groups,
    of which the second has nothing (one tile), or the last tile nothing for it."""
    from oracle import oracle
    rng = np.random.default_rng(d + count)
    hq, hkv, t, size = 4, 2, 52, 8192
    kc, vc = (draw((hkv, size, d), rng, F16) for _ in range(2))
    kc[:, count:], vc[:, count:] = np.nan, np.nan          # rows never written
    q, k, v = (draw((1, h, t, d), rng, F16) for h in (hq, hkv, hkv))
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((1, t, hq, d), F32)
    out.fill_(0xFF)
    print(f"prefill chunk d={d} count={count}", flush=True)
    got = gpu.attention(out, D(q), D(k), D(v), causal=True,
                        cache=(D(kc), D(vc), D(np.array([count], np.uint32)), False)).numpy()
    want, _, _ = oracle.attention_cached(q[0], k, v, kc, vc, count, causal=True)
    # P to fp16 (2^-11 of sum p |v| <= max |v|), scores of D products in fp32
    vmax = max(np.abs(vc[:, :count]).max(initial=0), np.abs(v).max())
    assert np.isfinite(got).all() and np.abs(got[0] - want).max() <= float(vmax) * (2.0 ** -11 + 64 * d * 2.0 ** -24)
