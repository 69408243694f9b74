"""The prefill GEMM's three tiles and its K splits against the dequantised
product in 64 bits (gemvW4A16Neon per token, xq_gemv_w4a16_neon.cpp:259-291), at
sizes that leave each tile, quad of groups and split partly empty, in the four
metadata forms.

Bound: x carries 22 bits (fp16 hi + lo: 2^-22 of itself), the codes are exact, the
zero-point term's factors carry 22 bits each, and the fp32 sums round once per
MFMA and group: |error| <= (2^-20 + (8 G + 16) 2^-24 / 4) sum |w| |x|, the last
term with its roundings' signs averaging out to a quarter of their worst case."""
import ctypes

import numpy as np
import pytest

import xqbind as xb
from test_decode_ops_gpu import dev

pytestmark = pytest.mark.gpu


def matrix(rng, rows, cols, form):
    """(packed, scales, zeros, affine, dense fp64) in the metadata form: `s16` fp16 scale and zero 8, `f16` fp16
    pairs, `z4` fp32 scale and integer zero, `f32` fp32 pairs (affine)."""
    n = rows * cols // 64
    packed = rng.integers(0, 256, rows * cols // 2, dtype=np.uint8)
    scales = np.abs(rng.normal(0, 0.02, n)).astype(np.float32)
    if form in ("s16", "f16"):
        scales = scales.astype(np.float16).astype(np.float32)
    zeros = {"s16": np.full(n, 8.0), "f16": np.round(rng.normal(0, 4, n)) / 8, "z4": rng.integers(0, 16, n).astype(float),
             "f32": rng.normal(0, 0.1, n)}[form].astype(np.float32)
    affine = 1 if form in ("f16", "f32") else 0
    q = np.stack([packed & 15, packed >> 4], -1).reshape(rows, cols // 64, 64).astype(np.float64)
    s, z = scales.astype(np.float64).reshape(rows, -1, 1), zeros.astype(np.float64).reshape(rows, -1, 1)
    return packed, scales, zeros, affine, (q * s + z if affine else (q - z) * s).reshape(rows, cols)


@pytest.mark.parametrize("form", ["s16", "f16", "z4", "f32"])
@pytest.mark.parametrize("rows,cols,m,epi", [
    (128, 512, 1, "store"), (129, 1024, 32, "add"), (34, 4160, 33, "silu"), (1000, 640, 31, "store"),  # small tile
    (258, 2048, 7, "silu"), (96, 12288, 40, "add"),                                                    # ... split
    (20001, 576, 130, "add"), (20000, 64, 129, "silu"),                                                 # middle tile
    (4098, 3648, 247, "silu"), (1502, 5952, 450, "add"),                                                # ... split
    (24600, 320, 500, "store"), (20002, 192, 257, "store"), (19970, 448, 300, "add"), (20000, 256, 384, "silu")])  # large
def test_matches_64_bit_product(rows, cols, m, epi, form):
    rng = np.random.default_rng(rows + cols + m)
    packed, scales, zeros, affine, W = matrix(rng, rows, cols, form)
    w = xb.DeviceW4(packed, scales, zeros, rows, cols, affine=affine)
    ldx, out = cols + 4, rows // 2 if epi == "silu" else rows
    ldy = out + 3
    x = rng.normal(0, 1, (m, ldx)).astype(np.float32)
    y0 = rng.normal(0, 1, (m, ldy)).astype(np.float32)
    yd = dev(y0)
    ws = xb.DeviceBuffer(xb.hip().xqhip_gemm_workspace_bytes(m, cols, rows))
    code = {"store": xb.EPI_STORE, "add": xb.EPI_ADD, "silu": xb.EPI_SILU_PAIR}[epi]
    xb.ck(xb.hip().xqhip_gemm_w4a16(w.ref, dev(x).ptr, m, ldx, None, 0, yd.ptr, ldy, code, ws.ptr, ws.nbytes, None))
    got = yd.download(np.float32, m * ldy).reshape(m, ldy)
    assert np.array_equal(got[:, out:], y0[:, out:])
    x64 = x[:, :cols].astype(np.float64)
    y, size = x64 @ W.T, np.abs(x64) @ np.abs(W).T
    G = cols // 64
    tol = (2.0**-20 + (8 * G + 16) * 2.0**-26) * size + 1e-7
    if epi == "silu":
        g, u = y[:, 0::2], y[:, 1::2]
        sig = 1 / (1 + np.exp(-g))
        # |silu'| <= 1.1; expf and the divide: 4 ulp
        tol = 1.1 * np.abs(u) * tol[:, 0::2] + (np.abs(g * sig) + tol[:, 0::2]) * tol[:, 1::2] + 2.0**-21 * np.abs(g * sig * u)
        y = g * sig * u
    elif epi == "add":
        y = y0[:, :out] + y
        tol = tol + 2.0**-23 * np.abs(y)
    err = np.abs(got[:, :out] - y)
    assert (err <= tol).all(), (err / tol).max()


@pytest.mark.parametrize("rows,cols,m", [(256, 512, 3), (128, 4096, 2), (24600, 128, 500), (20002, 128, 257)])
def test_columns_beside_an_outlier(rows, cols, m):
    """One weight a row beside a token's outlier of 2^14 times the other values (under the zero point): scaled with the
    outlier to 2^12 .. 2^13, x is off by 2^-22 of itself and 2^-25 (half the smallest fp16) = 2^-37 of the outlier, the
    same in even and odd columns; the sum of hi and lo, the scale and the result round to fp32."""
    rng = np.random.default_rng(cols)
    r = np.arange(rows)
    q = np.full((rows, cols), 8, np.uint8)
    at = 1 + r % (cols - 1)
    q[r, at] = (8 + rng.integers(1, 16, rows)) % 16
    scales = np.abs(rng.normal(0, 0.02, rows * cols // 64)).astype(np.float16).astype(np.float32)
    w = xb.DeviceW4(q[:, 0::2] | q[:, 1::2] << 4, scales, np.full_like(scales, 8.0), rows, cols)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32)
    x[:, 0] = 2.0**14
    yd, xd = xb.DeviceBuffer(4 * m * rows), dev(x)
    ws = xb.DeviceBuffer(xb.hip().xqhip_gemm_workspace_bytes(m, cols, rows))
    xb.ck(xb.hip().xqhip_gemm_w4a16(w.ref, xd.ptr, m, cols, None, 0, yd.ptr, rows, xb.EPI_STORE, ws.ptr, ws.nbytes, None))
    got = yd.download(np.float32, m * rows).reshape(m, rows)
    weight = (q[r, at].astype(np.float64) - 8) * scales.reshape(rows, -1)[r, at // 64]
    xa = x[:, at].astype(np.float64)
    tol = np.abs(weight) * (np.abs(xa) * (2.0**-22 + 3 * 2.0**-24) + 2.0**(14 - 37))
    err = np.abs(got - weight * xa)
    assert (err <= tol).all(), (err / tol).max()


@pytest.mark.parametrize("cols,pro", [(640, "none"), (2048, "none"), (640, "rms"), (4096, "gated")])
def test_rows_of_tiny_values(cols, pro):
    """Rows whose largest magnitude is far below 2^-113, subnormal or 0: the row's power of two stays finite (fp16 then
    holds 2^-152, below fp32's smallest), the result has the precision of any other row down to fp32's subnormals."""
    rows, m = 96, 6
    rng = np.random.default_rng(cols)
    packed, scales, zeros, affine, W = matrix(rng, rows, cols, "z4")
    w = xb.DeviceW4(packed, scales, zeros, rows, cols, affine=affine)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32)
    x = (x * np.array([1e-34, 1e-36, 3e-38, 1e-40, 0.0, 1.0])[:, None]).astype(np.float32)
    x64 = x.astype(np.float64)
    weight, gate, ref = np.ones(cols, np.float32), np.ones((m, cols), np.float32), None
    wd, gd = dev(weight), dev(gate)
    if pro == "rms":  # eps far above the squares: x / 1e-3
        ref = ctypes.byref(xb.Prologue(xb.PRO_RMS, 0, wd.ptr, None, 1e-6))
        x64 = x64 / np.sqrt((x64**2).mean(-1, keepdims=True) + 1e-6)
    elif pro == "gated":
        ref = ctypes.byref(xb.Prologue(xb.PRO_GATED_HEAD, 128, wd.ptr, gd.ptr, 1e-6))
        h = x64.reshape(m, -1, 128)
        x64 = (h / np.sqrt((h**2).mean(-1, keepdims=True) + 1e-6)).reshape(m, cols) / (1 + np.exp(-1.0))
    xd, yd = dev(x), xb.DeviceBuffer(4 * m * rows)
    ws = xb.DeviceBuffer(xb.hip().xqhip_gemm_workspace_bytes(m, cols, rows))
    xb.ck(xb.hip().xqhip_gemm_w4a16(w.ref, xd.ptr, m, cols, ref, cols, yd.ptr, rows, xb.EPI_STORE, ws.ptr, ws.nbytes, None))
    got = yd.download(np.float32, m * rows).reshape(m, rows)
    G = cols // 64
    # a prologue's own roundings: a few of fp32 on each x, and of its subnormals (2^-149) where it ends there
    lift = 2.0**-21 if pro != "none" else 0.0
    tol = (2.0**-20 + lift + (8 * G + 16) * 2.0**-26) * (np.abs(x64) @ np.abs(W).T) + 2.0**-148
    tol += 4 * 2.0**-149 * np.abs(W).sum(-1) if pro != "none" else 0.0
    err = np.abs(got - x64 @ W.T)
    assert (err <= tol).all(), (err / tol).max(-1)


@pytest.mark.parametrize("pro", ["none", "rms", "gated"])
@pytest.mark.parametrize("cols", [2048, 4096, 6144, 8192, 10240, 12288, 2176])
def test_prologues_of_each_width(cols, pro):
    """The preparation's vectorised widths (2048 times 1 to 6) and a general one, each prologue: weights and
    gates that differ in every column.  A prologue rounds x a few times (its sum of squares with errors of either sign),
    silu by 4 ulp: 2^-20 of x more than without."""
    rows, m = 64, 5
    rng = np.random.default_rng(cols)
    packed, scales, zeros, affine, W = matrix(rng, rows, cols, "s16")
    w = xb.DeviceW4(packed, scales, zeros, rows, cols, affine=affine)
    x, gate = (rng.normal(0, 1, (m, cols + 4)).astype(np.float32) for _ in range(2))
    weight = rng.normal(1, 0.3, cols).astype(np.float32)
    xd, gd, wd, ref = dev(x), dev(gate), dev(weight), None
    x64, g64, w64 = x[:, :cols].astype(np.float64), gate[:, :cols].astype(np.float64), weight.astype(np.float64)
    if pro == "rms":
        ref = ctypes.byref(xb.Prologue(xb.PRO_RMS, 0, wd.ptr, None, 1e-6))
        x64 = x64 / np.sqrt((x64**2).mean(-1, keepdims=True) + 1e-6) * w64
    elif pro == "gated":
        ref = ctypes.byref(xb.Prologue(xb.PRO_GATED_HEAD, 128, wd.ptr, gd.ptr, 1e-6))
        h = x64.reshape(m, -1, 128)
        h = h / np.sqrt((h**2).mean(-1, keepdims=True) + 1e-6) * w64[:128]
        x64 = h.reshape(m, cols) * g64 / (1 + np.exp(-g64))
    yd = xb.DeviceBuffer(4 * m * rows)
    ws = xb.DeviceBuffer(xb.hip().xqhip_gemm_workspace_bytes(m, cols, rows))
    xb.ck(xb.hip().xqhip_gemm_w4a16(w.ref, xd.ptr, m, cols + 4, ref, cols + 4, yd.ptr, rows, xb.EPI_STORE, ws.ptr,
                                    ws.nbytes, None))
    got = yd.download(np.float32, m * rows).reshape(m, rows)
    G = cols // 64
    tol = (2.0**-20 + (2.0**-20 if pro != "none" else 0.0) + (8 * G + 16) * 2.0**-26) * (np.abs(x64) @ np.abs(W).T)
    err = np.abs(got - x64 @ W.T)
    assert (err <= tol).all(), (err / tol).max()
