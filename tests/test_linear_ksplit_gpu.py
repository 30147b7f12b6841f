"""The small-tile Linear (gemm_ksplit.hip) against float64, at the edges of its
tiles, k chunks and both staging forms. The bound is the rounding an fp32 sum
of K products can make, (K + 1) 2^-24 sum |x w|, plus one fp16 rounding of each
fp32 activation that meets fp16 weights (2^-11 sum |x w|) and of the output
(2^-11 |y|)."""
import ctypes

import numpy as np
import pytest

from helpers import draw, normal

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


def silu(v):
    return v / (1 + np.exp(-v))


def check(gpu, m, k, n, xdt, odt, tile, bias=None, residual=None, gated=False, off=0, wdt=F16):
    rng = np.random.default_rng(m + k + n)
    w, x = draw(normal((n, k), 0.05), rng, wdt), draw((m, k), rng, xdt)
    b = draw(normal((n,) if bias == "row" else (m, n), 0.05), rng, F16) if bias else None
    r = draw((n,) if residual == "row" else (m, n), rng, odt) if residual else None
    D = gpu.DeviceArray.from_numpy
    dw = D(np.concatenate([np.zeros(off, wdt), w.ravel()]))
    dx, db, dr = D(x), None if b is None else D(b), None if r is None else D(r)
    out = gpu.DeviceArray((m, n // 2 if gated else n), odt)
    out.fill_(0xFF)
    a = gpu.linear_args(out, dx, D(w), db, dr, gated=gated, gate_epi="SILU")
    a.weight = dw.ptr + w.itemsize * off
    name, splits = gpu.linear_plan(a)
    print(f"ksplit m={m} k={k} n={n} {np.dtype(xdt)} -> {np.dtype(odt)} gated={gated} plan={name}", flush=True)
    assert name == f"tile_f{8 * w.itemsize}_{tile}_kwaves" + ("_gated" if gated else "") and splits == 1
    assert gpu.lib().vai_linear_workspace_size(ctypes.byref(a)) == 0
    gpu.check(gpu.lib().vai_linear_launch(ctypes.byref(a), None), "linear")
    gpu.synchronize()
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    mag = np.abs(x64) @ np.abs(w64).T
    tol = mag * ((k + 1) * 2.0 ** -24 + (2.0 ** -11 if xdt == F32 and wdt == F16 else 0)) + 1e-6
    y = x64 @ w64.T + (0 if b is None else b.astype(np.float64))
    if gated:
        h = n // 2
        g, u = y[:, :h], y[:, h:]
        y = silu(g) * u
        tol = 1.1 * tol[:, :h] * np.abs(u) + np.abs(silu(g)) * tol[:, h:] + 2e-6 * np.abs(y)   # |silu'| <= 1.1
    elif r is not None:
        y = y + r.astype(np.float64)
    if odt == F16:
        tol = tol + 2.0 ** -11 * np.abs(y)
    got = out.numpy().astype(np.float64)
    assert np.isfinite(got).all() and (np.abs(got - y) <= tol).all(), float((np.abs(got - y) / tol).max())


@pytest.mark.parametrize("m, k, n, xdt, odt, tile, kw", [
    (9, 32, 33, F16, F32, "32x32", {}),                             # one chunk, half of it past K; one column in the second tile
    (32, 4096, 128, F16, F32, "32x32", {"bias": "row"}),            # every wave of eight runs whole trips
    (33, 1032, 100, F16, F16, "32x32", {"residual": "full"}),       # a k tail of one 16-byte piece, a second row tile of one row
    (50, 1000, 77, F32, F32, "32x32", {"bias": "row"}),             # fp32 X, odd N
    (61, 1147, 96, F16, F32, "32x32", {"residual": "row"}),         # odd K: staged through registers
    (70, 333, 40, F32, F16, "32x32", {"bias": "full"}),             # odd K, fp32 X, a bias of its own repeat
    (64, 2048, 8192, F16, F16, "32x64", {"bias": "row", "residual": "full"}),
    (90, 2040, 7000, F32, F32, "64x64", {}),
    (61, 1148, 8191, F16, F32, "32x64", {"residual": "full"}),      # K % 8 = 4, odd N
    (100, 1024, 5000, F16, F32, "64x64", {"residual": "full"}),
    (300, 512, 4100, F16, F16, "64x128", {"bias": "row"}),          # quadrant tiles, ragged M and N
    (300, 515, 4100, F32, F32, "64x128", {"residual": "full"}),     # ... through registers
    (400, 576, 8192, F16, F32, "128x128", {"bias": "row"}),
    (400, 571, 8192, F16, F16, "128x128", {}),
    (511, 640, 8200, F32, F32, "128x128", {"residual": "full"}),
])
def test_ksplit(gpu, m, k, n, xdt, odt, tile, kw):
    check(gpu, m, k, n, xdt, odt, tile, **kw)


@pytest.mark.parametrize("m, k, h, xdt, odt, tile", [
    (9, 256, 17, F16, F32, "32x32"),          # H one past a tile's 16 outputs
    (40, 1000, 2050, F32, F16, "32x64"),
    (61, 1021, 700, F16, F32, "32x32"),       # odd K
    (300, 512, 2100, F16, F16, "64x128"),
])
def test_ksplit_gated(gpu, m, k, h, xdt, odt, tile):
    check(gpu, m, k, 2 * h, xdt, odt, tile, bias="row", gated=True)


@pytest.mark.parametrize("m, k, n, odt, tile, kw", [
    (1024, 768, 3072, F32, "64x64", {"bias": "row"}),          # whole tiles
    (1000, 100, 3201, F16, "64x64", {"residual": "full"}),     # a short last chunk, one column past a tile
    (900, 301, 3100, F32, "64x64", {"bias": "full"}),         # odd K: through registers
    (9, 33, 40, F32, "32x32", {}),                            # two chunks for eight waves, the second of one k
    (33, 1147, 96, F16, "32x32", {"bias": "row", "residual": "row"}),
    (70, 1028, 1000, F32, "32x32", {"residual": "full"}),     # K % 4 == 0: direct copies, a short last chunk
    (64, 516, 64, F32, "32x32", {"off": 1}),                  # W off a 16-byte boundary
])
def test_ksplit_f32(gpu, m, k, n, odt, tile, kw):
    check(gpu, m, k, n, F32, odt, tile, wdt=F32, **kw)


def test_ksplit_unaligned_weight(gpu):
    """A weight two bytes off a 16-byte boundary is staged through registers."""
    check(gpu, 20, 512, 64, F16, F32, "32x32", off=1)


@pytest.mark.parametrize("m, k, n, gated, tile", [
    (9, 256, 33, False, "32x32"), (61, 3072, 5120, False, "32x64"), (100, 1024, 5000, False, "64x64"),
    (300, 512, 4100, False, "64x128"), (400, 384, 8192, False, "128x128"),
    (9, 256, 34, True, "32x32"), (40, 1024, 4100, True, "32x64"), (300, 512, 4200, True, "64x128"),
])
def test_ksplit_packed_weight(gpu, m, k, n, gated, tile):
    """The packed weight takes the same k order: the same bits, from the packed
    copy alone (the weight it was packed from is overwritten with NaNs)."""
    rng = np.random.default_rng(n)
    D = gpu.DeviceArray.from_numpy
    dw, dx = D(draw(normal((n, k), 0.05), rng, F16)), D(draw((m, k), rng, F16))
    outs = [gpu.DeviceArray((m, n // 2 if gated else n), F32) for _ in range(2)]
    for i, out in enumerate(outs):
        out.fill_(0xFF)
        a = gpu.linear_args(out, dx, dw, None, None, gated=gated, gate_epi="SILU")
        if i:
            packed = gpu.linear_pack_weight(a)
            a.packed_weight = packed.ptr
            dw.fill_(0xFF)
        name = gpu.linear_plan(a)[0]
        print(f"ksplit packed={i} m={m} k={k} n={n} gated={gated} plan={name}", flush=True)
        assert name == f"tile_f16_{tile}_kwaves" + ("_gated" if gated else "")
        gpu.check(gpu.lib().vai_linear_launch(ctypes.byref(a), None), "linear")
        gpu.synchronize()
    got, want = outs[1].numpy(), outs[0].numpy()
    assert np.isfinite(got).all() and (got == want).all()


def chain_error(k, step, chain, n=4096):
    """Relative error (2-norm) of fp32 sums of k normal products, added `step` at a time to chains of `chain` k
    whose totals are added in turn."""
    rng = np.random.default_rng(k)
    parts = rng.standard_normal((k // step, n)) * np.sqrt(step)   # one step's products, summed exactly
    total = np.zeros(n, F32)
    for c in range(0, k // step, chain // step):
        run = np.zeros(n, F32)
        for p in parts[c:c + chain // step].astype(F32):
            run += p
        total += run
    want = parts.astype(F32).astype(np.float64).sum(axis=0)
    return float(np.linalg.norm(total - want) / np.linalg.norm(want))


@pytest.mark.parametrize("m, k, n, xdt, tile, kw", [
    (500, 4096, 4096, F16, "64x128", {}),
    (400, 8192, 8192, F16, "128x128", {}),
    (300, 8192, 2048, F16, "64x64", {}),
    (300, 8191, 2048, F16, "64x64", {}),           # through registers
    (61, 8192, 5120, F16, "32x64", {}),
    (64, 8192, 1024, F16, "32x32", {}),
    (500, 4096, 4096, F32, "64x128", {}),
    (64, 4095, 1000, F32, "32x32", {"wdt": F32}),
])
def test_ksplit_long_k(gpu, m, k, n, xdt, tile, kw):
    """The sums run in chains of at most 256 k (512 in 128x128 tiles from K = 3584, 128 with fp32 weights), the
    shortest that a K split had at these sizes: the error against float64 is that of such chains, with a matrix
    instruction's k taken 8 (fp32: 1) at a time. One chain over K has 2.5 times as much at K = 4096, sums over
    a sixteenth of K = 8192 1.1 times."""
    wdt = kw.get("wdt", F16)
    rng = np.random.default_rng(m + k + n)
    w, x = draw(normal((n, k), 0.05), rng, wdt), draw((m, k), rng, F16).astype(xdt)
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((m, n), F32)
    a = gpu.linear_args(out, D(x), D(w))
    name = gpu.linear_plan(a)[0]
    print(f"ksplit chains m={m} k={k} n={n} plan={name}", flush=True)
    assert name == f"tile_f{8 * w.itemsize}_{tile}_kwaves"
    gpu.check(gpu.lib().vai_linear_launch(ctypes.byref(a), None), "linear")
    gpu.synchronize()
    cols = slice(n // 2, n // 2 + 64)
    want = x.astype(np.float64) @ w[cols].astype(np.float64).T
    err = float(np.linalg.norm(out.numpy()[:, cols] - want) / np.linalg.norm(want))
    bound = chain_error((k + 511) // 512 * 512, *((1, 128) if wdt == F32 else (8, 512 if tile == "128x128" else 256)))
    print(f"  error {err:.2e}, chains {bound:.2e}", flush=True)
    assert err <= 1.04 * bound


@pytest.mark.parametrize("m, k, n, xdt, wdt, off, tile", [
    (22, 7864, 256, F32, F32, 0, "64x64"),
    (9, 4095, 130, F32, F32, 0, "64x64"),
    (40, 8200, 96, F32, F16, 0, "64x64"),
    (33, 16384, 40, F16, F16, 1, "64x64"),
])
def test_long_k_over_few_tiles(gpu, m, k, n, xdt, wdt, off, tile):
    """K split over workgroups where the small tiles are too few for the chip; without the workspace for that
    (or with one too small) the small tiles run."""
    rng = np.random.default_rng(k)
    w, x = draw(normal((n, k), 0.05), rng, wdt), draw((m, k), rng, F16).astype(xdt)
    D = gpu.DeviceArray.from_numpy
    dw = D(np.concatenate([np.zeros(off, wdt), w.ravel()]))
    out = gpu.DeviceArray((m, n), F32)
    a = gpu.linear_args(out, D(x), D(w))
    a.weight = dw.ptr + w.itemsize * off
    name, splits = gpu.linear_plan(a)
    need = gpu.linear_workspace_size(a)
    print(f"few tiles m={m} k={k} n={n} plan={name} splits={splits}", flush=True)
    assert name == f"tile_f{8 * w.itemsize}_{tile}" and splits > 1 and need == splits * m * n * 4
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    want, tol = x64 @ w64.T, (np.abs(x64) @ np.abs(w64).T) * (k + 1) * 2.0 ** -24
    ws = gpu.DeviceArray((need,), np.uint8)
    errs = []
    for ptr, size in ((ws.ptr, need), (None, 0), (ws.ptr, need - 4)):
        out.fill_(0xFF)
        a.workspace, a.workspace_bytes = ptr, size
        gpu.check(gpu.lib().vai_linear_launch(ctypes.byref(a), None), "linear")
        gpu.synchronize()
        got = out.numpy().astype(np.float64)
        assert np.isfinite(got).all() and (np.abs(got - want) <= tol).all()
        errs.append(got)
    assert (errs[1] == errs[2]).all()
