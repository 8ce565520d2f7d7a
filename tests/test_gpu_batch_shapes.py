"""GPU: the launch shapes of the small-M products on both sides of each line that the automatic
choice draws (row tiles per wavefront, slices of k, gate/up pairs of whole k)."""
import numpy as np
import pytest

import laguna_hip as lh
import oracle as orc
import synth
from conftest import parity

pytestmark = pytest.mark.gpu


def weights(ctx, dtype, k, n, seed):
    raw = synth.q4k_weight(seed, k, n) if dtype == lh.Q4_K else synth.q8_0_weight(seed, k, n)
    wb = lh.upload_bytes(ctx, raw)
    return raw, wb, lh.repack_tiled(ctx, wb, dtype, k, n)


def close(y, x, raw, dtype, k, n):
    # of the sum of magnitudes |x w|: 2^-22 a product for the parts of x, 32 additions of 2^-24
    # inside a sub-block's matrix product, and as many over a chunk's sub-blocks and the chunks
    y64, a = orc.proj_quant_f64(x, raw, dtype, k, n)
    parity(y, y64, a)
    assert np.all(np.abs(y - y64) <= (2.0 ** -22 + (48 + k // 256) * 2.0 ** -24) * a)


# columns of 128 rows: under and from a quarter of 256 CUs (8064, 8192); of 64 rows: a CU each
# and one more (16384, 16385); 7/8 of the CUs in columns of 128 (28544, 28672); 15 and 16 chunks
# over few rows; Q8_0 rounds of more than 48 rows with a split and without
@pytest.mark.parametrize("dtype", [lh.Q4_K, lh.Q8_0])
@pytest.mark.parametrize("k,n", [(512, 8064), (512, 8192), (512, 16384), (512, 16385), (256, 28544), (256, 28672),
                                 (3840, 40), (4096, 40)])
@pytest.mark.parametrize("m", [16, 17, 32, 49, 64])
def test_shape_edges(ctx, dtype, k, n, m):
    print(f"shape edge dtype={dtype} k={k} n={n} m={m}", flush=True)
    raw, wb, wt = weights(ctx, dtype, k, n, 0x5EED0C00 + k + n)
    x = synth.normal(0x5EED0C01 + m, m * k).reshape(m, k)
    xb, out = lh.upload_f32(ctx, x), []
    for w, t in ((wb, dtype), (wt, lh.TILED[dtype])):
        cb = lh.GpuBuffer(ctx, 4 * m * n)
        cb.fill(0xFF)
        lh.dispatch_proj_quant_batch(ctx, xb, lh.F32, w, cb, k, n, m, t)
        out.append(cb.read_f32(m * n).reshape(m, n))
    assert np.array_equal(out[0], out[1])  # same slices whatever the row tiles
    for r in (0, m - 1):
        close(out[0][r], x[r], raw, dtype, k, n)


# columns of 32 rows of both products: 7/8 of a CU each and fewer, one each and one more; 8
# chunks and 9
@pytest.mark.parametrize("dtype", [lh.Q4_K, lh.Q8_0])
@pytest.mark.parametrize("k,n", [(512, 7136), (512, 7168), (512, 8192), (512, 8193), (2048, 7168), (2304, 7168)])
@pytest.mark.parametrize("m", [16, 32, 40, 64])
def test_pair_edges(ctx, dtype, k, n, m):
    print(f"pair edge dtype={dtype} k={k} n={n} m={m}", flush=True)
    wg, wu = weights(ctx, dtype, k, n, 0x5EED0C10 + n), weights(ctx, dtype, k, n, 0x5EED0C11 + n)
    x = synth.normal(0x5EED0C12 + m, m * k).reshape(m, k)
    xb, out = lh.upload_f32(ctx, x), []
    for i, t in ((1, dtype), (2, lh.TILED[dtype])):
        gb, ub = lh.GpuBuffer(ctx, 4 * m * n), lh.GpuBuffer(ctx, 4 * m * n)
        gb.fill(0xFF)
        lh.dispatch_silu_gate_up_batch(ctx, xb, wg[i], wu[i], gb, ub, k, n, m, t)
        out.append(gb.read_f32(m * n).reshape(m, n).astype(np.float64))
    for r in (0, m - 1):
        g, ga = orc.proj_quant_f64(x[r], wg[0], dtype, k, n)
        u, ua = orc.proj_quant_f64(x[r], wu[0], dtype, k, n)
        e = 2.0 ** -22 + (48 + k // 256) * 2.0 ** -24  # of each product's sum of magnitudes
        s = g / (1 + np.exp(-g))
        # |silu'| < 1.1; the SiLU's own roundings, each a few 2^-24 of the result
        tol = 1.1 * e * ga * np.abs(u) + np.abs(s) * e * ua + 1.1 * e * ga * e * ua + 16 * 2.0 ** -24 * np.abs(s * u)
        for y in out:
            assert np.all(np.abs(y[r] - s * u) <= tol)
