"""The convolution over the weight as stored (conv_direct.hip: rows wider than
128 outputs, kernels over 3x3) against the float64 sum, at the edges of its
column pieces, row and channel tiles and channel blocks. The bound: the fp32
sum of K exact products, K 2^-24 sum |x w|, one fp16 rounding of an fp32 input
and of an fp16 output."""
import ctypes

import numpy as np
import pytest

from helpers import draw, normal

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


def conv64(x, w, stride):
    k, (co, ci) = w.shape[2], w.shape[:2]
    b, _, h, wi = x.shape
    xp = np.pad(x, ((0, 0), (0, 0), (k // 2, k // 2), (k // 2, k // 2)))
    ho, wo = (h - 1) // stride + 1, (wi - 1) // stride + 1
    out = np.zeros((b, co, ho, wo))
    for kh in range(k):
        for kw in range(k):
            v = xp[:, :, kh:kh + (ho - 1) * stride + 1:stride, kw:kw + (wo - 1) * stride + 1:stride]
            out += np.einsum("bchw,oc->bohw", v, w[:, :, kh, kw], optimize=True)
    return out


@pytest.mark.parametrize("b, ci, co, h, w, k, stride, xdt, odt, epi, residual, order", [
    (1, 3, 16, 9, 136, 3, 1, F16, F32, "SILU", False, "AFTER_EPILOGUE"),    # one octet of 3 channels, 32-channel tiles of 8 rows
    (1, 32, 64, 13, 264, 3, 2, F16, F16, "SILU", False, "AFTER_EPILOGUE"),  # stride 2, whole octets: no zero fill
    (2, 17, 70, 5, 333, 3, 1, F16, F32, "RELU", True, "AFTER_EPILOGUE"),    # odd width: pieces moved down, one channel past two octets
    (1, 40, 33, 6, 200, 3, 1, F32, F32, "NONE", True, "BEFORE_EPILOGUE"),   # fp32 image, one channel past a 32-channel tile
    (1, 130, 65, 4, 262, 3, 2, F16, F16, "GELU", False, "AFTER_EPILOGUE"),  # several channel blocks, the last one short
    (1, 200, 20, 3, 160, 3, 1, F32, F16, "SIGMOID", False, "AFTER_EPILOGUE"),
    (1, 8, 64, 7, 145, 1, 1, F16, F32, "SILU", True, "AFTER_EPILOGUE"),     # pointwise, one piece of weights a row
    (1, 700, 40, 5, 160, 1, 1, F16, F32, "NONE", False, "AFTER_EPILOGUE"),  # pointwise, blocks, 4 of 8 channels in the last octet
    (1, 515, 64, 3, 301, 1, 2, F32, F32, "NONE", False, "AFTER_EPILOGUE"),  # ... from an odd-width fp32 image, stride 2
    (1, 5, 10, 20, 30, 5, 1, F16, F32, "RELU", False, "AFTER_EPILOGUE"),    # 5x5 on a narrow image
    (1, 24, 48, 17, 40, 7, 2, F16, F16, "NONE", True, "AFTER_EPILOGUE"),    # 7x7, stride 2
    (1, 2, 4, 8, 8, 9, 1, F32, F32, "NONE", False, "AFTER_EPILOGUE"),       # the kernel is wider than the image
    (1, 4, 8, 6, 400, 3, 3, F16, F32, "NONE", False, "AFTER_EPILOGUE"),     # stride 3
])
def test_conv_direct(gpu, b, ci, co, h, w, k, stride, xdt, odt, epi, residual, order):
    rng = np.random.default_rng(ci + co + w)
    wt = draw(normal((co, ci, k, k), 0.1), rng, F16)
    bias, scale = draw(normal((co,), 0.1), rng, F16), draw(lambda g: g.uniform(0.5, 1.5, (co,)), rng, F16) if ci % 2 else None
    x = draw(lambda g: g.uniform(-1, 1, (b, ci, h, w)), rng, xdt)
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    r = draw((b, co, ho, wo), rng, xdt) if residual else None
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((b, co, ho, wo), odt)
    out.fill_(0xFF)
    a = gpu.conv2d_args(out, D(x), D(wt), D(bias), None if scale is None else D(scale), None if r is None else D(r),
                        stride=stride, epi=epi, order=order)
    assert gpu.lib().vai_conv2d_packed_weight_size(ctypes.byref(a)) == 0   # no packed plan for these
    print(f"conv direct b={b} ci={ci} co={co} {h}x{w} k={k} s={stride} {np.dtype(xdt)} -> {np.dtype(odt)}", flush=True)
    gpu.check(gpu.lib().vai_conv2d_launch(ctypes.byref(a), None), "conv")
    gpu.synchronize()
    x64, w64 = x.astype(np.float64), wt.astype(np.float64)
    s = (np.ones(co) if scale is None else scale.astype(np.float64))[:, None, None]
    mag = conv64(np.abs(x64), np.abs(w64), stride) * s
    tol = mag * (ci * k * k * 2.0 ** -24 + (2.0 ** -11 if xdt == F32 else 0)) + 1e-6
    y = conv64(x64, w64, stride) * s + bias.astype(np.float64)[:, None, None]
    if r is not None and order == "BEFORE_EPILOGUE":
        y = y + r.astype(np.float64)
    if epi == "SILU":
        y = y / (1 + np.exp(-y))
    elif epi == "RELU":
        y = np.maximum(y, 0)
    elif epi == "SIGMOID":
        y = 1 / (1 + np.exp(-y))
    elif epi == "GELU":
        from math import erf
        y = y * 0.5 * (1 + np.vectorize(erf)(y / np.sqrt(2)))
        tol = tol + 1e-6 * (1 + np.abs(y))   # the erf polynomial's 1.5e-7, times y
    if r is not None and order == "AFTER_EPILOGUE":
        y = y + r.astype(np.float64)
    tol = 1.2 * tol + 2e-6 * np.abs(y) + (2.0 ** -11 * np.abs(y) if odt == F16 else 0)   # slopes up to 1.13
    got = out.numpy().astype(np.float64)
    assert np.isfinite(got).all() and (np.abs(got - y) <= tol).all(), float((np.abs(got - y) / tol).max())


@pytest.mark.parametrize("xdt, w", [(F16, 136), (F32, 136), (F16, 141)])
def test_conv_direct_infinite_weight(gpu, xdt, w):
    """An infinite weight of a full channel block reaches its own output once: the last block, of one octet where
    the one before has 44, does not multiply it by the zeros of the channels that it lacks."""
    ci, co, h, bad = 360, 64, 5, 200
    rng = np.random.default_rng(w)
    x, wt = draw(lambda g: g.uniform(0.5, 1, (1, ci, h, w)), rng, xdt), draw(normal((co, ci, 1, 1), 0.1), rng, F16)
    wt[7, bad] = np.inf
    D = gpu.DeviceArray.from_numpy
    out = gpu.DeviceArray((1, co, h, w), F32)
    out.fill_(0xFF)
    print(f"conv direct infinity {np.dtype(xdt)} w={w}", flush=True)
    got = gpu.conv2d(out, D(x), D(wt)).numpy()
    x64, w64 = x.astype(np.float64), wt.astype(np.float64)
    assert (got[0, 7] == np.inf).all()
    keep = np.arange(co) != 7
    mag = conv64(np.abs(x64), np.abs(w64[keep]), 1)
    tol = mag * (ci * 2.0 ** -24 + (2.0 ** -11 if xdt == F32 else 0)) + 1e-6
    assert (np.abs(got[:, keep] - conv64(x64, w64[keep], 1)) <= tol).all()
