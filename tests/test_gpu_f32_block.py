"""GPU: the small-M product over f32 weights (f32 matrix cores; element by element where k
is not a multiple of 4 or an operand is unaligned) against the f64 sum."""
import numpy as np
import pytest

import laguna_hip as lh
import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,m,bf16", [
    (4, 1, 2, 0), (60, 15, 16, 0), (64, 16, 17, 1), (68, 17, 32, 0),     # partial and single blocks, row edges
    (260, 40, 33, 1), (512, 33, 48, 0), (1028, 100, 49, 0), (320, 64, 64, 1),  # each number of token tiles
    (256, 8200, 5, 0), (132, 8209, 31, 1),                               # two row tiles a workgroup
    (62, 9, 3, 0), (2, 5, 64, 0),                                        # k not a multiple of 4
])
def test_f32_block(ctx, k, n, m, bf16):
    print(f"f32 block k={k} n={n} m={m} bf16={bf16}", flush=True)
    w = synth.normal(0x5EED0800 + k, n * k, 0.02).reshape(n, k)
    x = synth.normal(0x5EED0801 + m, m * k).reshape(m, k)
    if bf16:
        u = (x.view(np.uint32) >> 16).astype(np.uint16)
        x = (u.astype(np.uint32) << 16).view(np.float32)
        xb = lh.upload_bytes(ctx, u.view(np.uint8).ravel())
    else:
        xb = lh.upload_f32(ctx, x)
    wb, cb = lh.upload_f32(ctx, w), lh.GpuBuffer(ctx, 4 * m * n)
    cb.fill(0xFF)
    lh.dispatch_proj_quant_batch(ctx, xb, lh.BF16 if bf16 else lh.F32, wb, cb, k, n, m, lh.F32)
    y = cb.read_f32(m * n).reshape(m, n).astype(np.float64)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    mag = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    # k f32 additions of exact products: k 2^-24 of the sum of magnitudes at the most
    assert np.all(np.abs(y - want) <= max(k, 8) * 2.0 ** -24 * mag + 1e-30)


@pytest.mark.parametrize("off", [0, 4])
def test_f32_block_nonfinite_and_unaligned(ctx, off):
    """Each output meets its own row and token only; a weight base off by `off` bytes."""
    k, n, m = 192, 50, 20
    print(f"f32 block non-finite, offset {off}", flush=True)
    w = synth.normal(0x5EED0810, n * k, 0.02).reshape(n, k)
    x = synth.normal(0x5EED0811, m * k).reshape(m, k)
    w[7, 100], x[3, 5] = np.inf, np.nan
    raw = np.zeros(n * k + 4, np.float32)
    raw[off // 4:off // 4 + n * k] = w.ravel()
    wb, xb, cb = lh.upload_f32(ctx, raw), lh.upload_f32(ctx, x), lh.GpuBuffer(ctx, 4 * m * n)
    lh.dispatch_proj_quant_batch(ctx, xb, lh.F32, wb.ptr + off, cb, k, n, m, lh.F32)
    y = cb.read_f32(m * n).reshape(m, n)
    assert np.all(np.isnan(y[3])) and np.all(np.isinf(np.delete(y[:, 7], 3)))
    ok = np.ones((m, n), bool)
    ok[3], ok[:, 7] = False, False
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
    assert np.all(np.isfinite(y[ok])) and np.max(np.abs(y[ok] - want[ok])) < 1e-5


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("k,ops", [(64, 7.5), (512, 10.75)])
def test_f32_block_rounding(ctx, k, ops, bf16):
    """The sum's order: 2-norm error of short rows.  In units of k var(x w), the squared partial
    sums that are rounded add up to `ops`: 4.5 k in chains of eight products, 1 k for each of
    three pairings of a block's eight chains, and at 512 (two blocks a wavefront, four
    wavefronts) 1 k and 2.25 k more; each rounding is 2^-25 of its sum at most."""
    n, m = 200, 16
    print(f"f32 block rounding k={k} bf16={bf16}", flush=True)
    w = synth.normal(0x5EED0820 + k, n * k, 0.02).reshape(n, k)
    u = synth.normal(0x5EED0821 + k, m * k).view(np.uint32) & np.uint32(0xFFFF0000)
    x = u.view(np.float32).reshape(m, k)
    xb = lh.upload_bytes(ctx, (u >> 16).astype(np.uint16).view(np.uint8)) if bf16 else lh.upload_f32(ctx, x)
    wb, cb = lh.upload_f32(ctx, w), lh.GpuBuffer(ctx, 4 * m * n)
    lh.dispatch_proj_quant_batch(ctx, xb, lh.BF16 if bf16 else lh.F32, wb, cb, k, n, m, lh.F32)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    e = np.linalg.norm(cb.read_f32(m * n).reshape(m, n) - want) / np.linalg.norm(want)
    print(f"  {e:.2e}", flush=True)
    assert e <= np.sqrt(ops) * 2.0 ** -25
