"""The M <= 8 Linear over rows that are not whole 16-byte chunks or operands off
a 16-byte boundary, against float64: within the rounding of an fp32 sum of K
products, (K + 1) 2^-24 sum |x w|, and of the output."""
import ctypes

import numpy as np
import pytest

from helpers import draw, normal

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


def run(gpu, x, w, odt, xoff=0, woff=0, plan="slab_any"):
    D = gpu.DeviceArray.from_numpy
    dx = D(np.concatenate([np.full(xoff, np.nan, x.dtype), x.ravel(), np.full(9, np.nan, x.dtype)]))
    dw = D(np.concatenate([np.full(woff, np.nan, w.dtype), w.ravel(), np.full(9, np.nan, w.dtype)]))
    out = gpu.DeviceArray((x.shape[0], w.shape[0]), odt)
    out.fill_(0xFF)
    a = gpu.linear_args(out, D(x), D(w))
    a.inp, a.weight = dx.ptr + x.itemsize * xoff, dw.ptr + w.itemsize * woff
    name = gpu.linear_plan(a)[0]
    print(f"slab m={x.shape[0]} k={x.shape[1]} n={w.shape[0]} {x.dtype} x {w.dtype} -> {name}", flush=True)
    assert name == plan
    gpu.check(gpu.lib().vai_linear_launch(ctypes.byref(a), None), "linear")
    gpu.synchronize()
    return out.numpy().astype(np.float64)


@pytest.mark.parametrize("m, k, n, xdt, wdt, odt, off", [
    (1, 7, 5, F16, F16, F32, (0, 0)),            # shorter than a chunk
    (1, 9, 3, F16, F16, F32, (0, 0)),            # one chunk and one element
    (2, 513, 9, F16, F16, F32, (0, 0)),          # one element past a block
    (1, 1147, 1001, F32, F16, F32, (0, 0)),
    (3, 2047, 33, F16, F16, F16, (0, 0)),        # one element short of whole blocks
    (4, 1025, 18, F32, F32, F32, (0, 0)),
    (5, 333, 16, F16, F16, F32, (0, 0)),
    (8, 1148, 100, F16, F16, F32, (0, 0)),       # K % 8 = 4, whole and part groups of rows
    (8, 767, 15, F32, F32, F16, (0, 0)),
    (7, 90, 31, F16, F32, F32, (0, 0)),
    (1, 2048, 40, F16, F16, F32, (0, 1)),        # whole chunks, W off a boundary
    (8, 512, 40, F32, F16, F32, (1, 0)),         # X off a boundary
    (6, 260, 21, F32, F32, F32, (3, 2)),
])
def test_slab_any(gpu, m, k, n, xdt, wdt, odt, off, plan=None):
    plan = plan or ("slab_any" if k >= 8 else "slab_scalar")
    rng = np.random.default_rng(m + k + n)
    x, w = draw((m, k), rng, xdt), draw(normal((n, k), 0.1), rng, wdt)
    got = run(gpu, x, w, odt, *off, plan=plan)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    y = x64 @ w64.T
    tol = (np.abs(x64) @ np.abs(w64).T) * (k + 1) * 2.0 ** -24 + (2.0 ** -11 * np.abs(y) + 2.0 ** -24 if odt == F16 else 1e-30)
    assert np.isfinite(got).all() and (np.abs(got - y) <= tol).all(), float((np.abs(got - y) / tol).max())


@pytest.mark.parametrize("m, k, n, xdt, wdt, odt", [
    (8, 1000, 1023, F16, F16, F32),       # one row a wave
    (5, 520, 1024, F32, F16, F32),        # two
    (8, 1000, 2050, F16, F16, F16),       # four, the last wave's partly past N
    (8, 1024, 2047, F32, F32, F32),       # fp32 rows: two a wave ...
    (6, 1028, 2049, F32, F32, F32),       # ... and X through LDS
    (4, 1032, 1030, F32, F16, F32),
    (3, 516, 17, F32, F32, F32),
    (4, 3504, 3075, F32, F16, F32),       # three and four rows staged in LDS: long rows ...
    (3, 2052, 12291, F32, F32, F16),
    (4, 1000, 33, F32, F32, F32),         # ... and rows of one K block
    (5, 600, 2049, F32, F32, F32),
    (8, 516, 2060, F16, F32, F32),
    (7, 4096, 1537, F32, F32, F32),
])
def test_slab_whole_chunks(gpu, m, k, n, xdt, wdt, odt):
    """Rows of whole chunks with more activations than a lane holds ahead."""
    test_slab_any(gpu, m, k, n, xdt, wdt, odt, (0, 0), plan="slab")


def test_slab_any_infinity(gpu):
    """An infinite activation in the elements that the short last chunk reads twice counts once."""
    x, w = np.ones((2, 77), F16), np.ones((5, 77), F16)
    x[0, 72] = np.inf
    w[:, 70] = 2.0
    got = run(gpu, x, w, F32)
    assert (got[0] == np.inf).all() and (got[1] == 78.0).all()
