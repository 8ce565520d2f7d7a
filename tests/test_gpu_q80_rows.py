"""GPU: Q8_0 projections of rows of whole blocks whose k is no multiple of 256, and the
fused silu(gate) * up down projection over Q8_0, against the f64 oracle, and over the same
inputs and forms as the element-wise path (a base that is not 2-byte aligned)."""
import numpy as np
import pytest

import laguna_hip as lh
import oracle as orc
import synth
from conftest import parity

pytestmark = pytest.mark.gpu


def call(ctx, raw, x, up, k, n, off=0):
    wb = lh.GpuBuffer(ctx, raw.size + 16)
    wb.upload(raw, offset=off)
    xb, cb = lh.upload_f32(ctx, x), lh.GpuBuffer(ctx, 4 * n)
    if up is None:
        lh.dispatch_proj_quant(ctx, xb, wb.ptr + off, cb, k, n, lh.Q8_0)
    else:
        lh.dispatch_silu_mul_proj_quant(ctx, xb, lh.upload_f32(ctx, up), wb.ptr + off, cb, k, n, lh.Q8_0)
    return cb.read_f32(n)


# one half block and lane edges (1024 elements a wavefront step), odd block counts, rows past
# the last wavefront, two rows a wavefront and rows beyond one round of workgroups, the
# longest staged row and one past it
@pytest.mark.parametrize("k,n", [(32, 1), (96, 9), (992, 17), (1056, 8), (2016, 300), (4128, 31), (288, 4099),
                                 (64, 9000), (160, 20011), (32224, 5), (32288, 3)])
@pytest.mark.parametrize("fuse", [0, 1])
def test_q80_rows(ctx, k, n, fuse):
    print(f"q8_0 rows k={k} n={n} fuse={fuse}", flush=True)
    raw = synth.q8_0_weight(0x5EED0A00 + k, k, n)
    x = synth.normal(0x5EED0A01 + n, k)
    up = synth.normal(0x5EED0A02 + n, k) if fuse else None
    y = call(ctx, raw, x, up, k, n)
    h = x if up is None else (x.astype(np.float64) / (1.0 + np.exp(-x.astype(np.float64))) * up).astype(np.float32)
    y64, a = orc.proj_quant_f64(h, raw, lh.Q8_0, k, n)
    parity(y, y64, a, 1e-6)
    parity(call(ctx, raw, x, up, k, n, off=1), y64, a, 1e-6)  # element by element


@pytest.mark.parametrize("fuse", [0, 1])
def test_q80_rows_nonfinite(ctx, fuse):
    """Activations and scales that are infinite or NaN reach what they reach element by element."""
    k, n = 1056, 40
    print(f"q8_0 rows non-finite fuse={fuse}", flush=True)
    raw = synth.q8_0_weight(0x5EED0A10, k, n).reshape(n, -1).copy()
    raw[3, 34:36] = np.array([0x7C00], np.uint16).view(np.uint8)    # d = inf
    raw[9, 68:70] = np.array([0x7E00], np.uint16).view(np.uint8)    # d = NaN
    raw[11, 0:2] = np.array([0x0001], np.uint16).view(np.uint8)     # the decoder's exponent-0 codes
    x = synth.normal(0x5EED0A11, k)
    up = synth.normal(0x5EED0A12, k) if fuse else None
    for v in (None, np.inf, -np.inf, np.nan):
        if v is not None:
            x[700] = v
        a, b = call(ctx, raw.ravel(), x, up, k, n), call(ctx, raw.ravel(), x, up, k, n, off=1)
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
        ok = np.isfinite(a)
        assert np.allclose(a[ok], b[ok], rtol=1e-5, atol=1e-5) and np.array_equal(a[np.isinf(a)], b[np.isinf(b)])


# rows shared by a workgroup's wavefronts, odd counts among them, a team of wavefronts per row,
# and a wavefront per row or two, on both sides of each line between them (256 CUs); the longest
# staged row
@pytest.mark.parametrize("k,n,fuse", [
    (4352, 256, 0), (4352, 257, 0), (8224, 1025, 0), (992, 4095, 0), (992, 4096, 0), (6144, 2047, 0), (6144, 2048, 0),
    (5120, 4095, 0), (5120, 4096, 0), (5120, 6144, 0), (5120, 6145, 0), (12288, 1024, 0), (16384, 1023, 0),
    (16384, 1024, 0), (16384, 2048, 0), (16384, 2049, 0), (32768, 1, 0), (33024, 5, 0), (4352, 256, 1), (4352, 257, 1),
    (4128, 1024, 1), (4128, 1025, 1), (32224, 1026, 1)])
def test_q80_few_rows(ctx, k, n, fuse):
    print(f"q8_0 few rows k={k} n={n} fuse={fuse}", flush=True)
    raw = synth.q8_0_weight(0x5EED0A20 + k, k, n)
    x = synth.normal(0x5EED0A21 + n, k)
    up = synth.normal(0x5EED0A22 + n, k) if fuse else None
    y = call(ctx, raw, x, up, k, n)
    h = x.astype(np.float64) if up is None else x.astype(np.float64) / (1.0 + np.exp(-x.astype(np.float64))) * up
    y64, a = orc.proj_quant_f64(h.astype(np.float32), raw, lh.Q8_0, k, n)
    # of the sum of magnitudes: the product's two roundings and the input's (the SiLU's four with
    # it), a lane's chain of at most 64 additions for each 4096 elements of its row (a lane takes
    # 64 of them), and the sums over lanes and wavefronts
    assert np.all(np.abs(y - y64) <= (8 + 64 * (1 + k // 4096) + 16) * 2.0 ** -24 * a)
    assert np.max(np.abs(y - y64) / a) <= 1e-6
