"""GPU: small-M products of 33 to 64 rows (one launch, two passes over each chunk of the
weights), bf16 activations in one f16 part, and the draft blocks whose 2m rows take such a
launch."""
import numpy as np
import pytest

import dflash_oracle as dfo
import laguna_hip as lh
import oracle as orc
import synth
from conftest import parity
from test_gpu_dflash import SMALL, TOL_FWD_TRAINED, build, check

pytestmark = pytest.mark.gpu


def weights(ctx, dtype, k, n, tiled, seed):
    raw = synth.q4k_weight(seed, k, n) if dtype == lh.Q4_K else synth.q8_0_weight(seed, k, n)
    wb = lh.upload_bytes(ctx, raw)
    return raw, (lh.repack_tiled(ctx, wb, dtype, k, n), lh.TILED[dtype]) if tiled else (wb, dtype), wb


def product(ctx, xb, xt, w, k, n, m):
    cb = lh.GpuBuffer(ctx, 4 * m * n)
    cb.fill(0xFF)
    lh.dispatch_proj_quant_batch(ctx, xb, xt, w[0], cb, k, n, m, w[1])
    return cb.read_f32(m * n).reshape(m, n)


# one chunk and many (slices), row tiles that end inside a workgroup's column, each number
# of token tiles and its edges
@pytest.mark.parametrize("dtype", [lh.Q4_K, lh.Q8_0])
@pytest.mark.parametrize("tiled", [0, 1])
@pytest.mark.parametrize("k,n,m", [(256, 16, 33), (1024, 100, 48), (2304, 65, 49), (4096, 200, 64), (512, 1, 47)])
def test_wide_block(ctx, dtype, tiled, k, n, m):
    print(f"wide block dtype={dtype} tiled={tiled} k={k} n={n} m={m}", flush=True)
    raw, w, keep = weights(ctx, dtype, k, n, tiled, 0x5EED0B00 + k + m)
    x = synth.normal(0x5EED0B01 + m, m * k).reshape(m, k)
    y = product(ctx, lh.upload_f32(ctx, x), lh.F32, w, k, n, m)
    assert np.array_equal(y, product(ctx, lh.upload_f32(ctx, x), lh.F32, w, k, n, m))
    # the rows in two calls of at most 32: each sums its slices in its own order
    two = np.vstack([product(ctx, lh.upload_f32(ctx, x[:32]), lh.F32, w, k, n, 32),
                     product(ctx, lh.upload_f32(ctx, x[32:]), lh.F32, w, k, n, m - 32)])
    # of the sum of magnitudes |x w|: 2^-22 a product for the parts of x, 32 additions of 2^-24
    # inside a sub-block's matrix product, and as many over a chunk's sub-blocks and the chunks
    bound = 2.0 ** -22 + (32 + 8 + k // 256 + 8) * 2.0 ** -24
    for r in (0, 15, 31, 32, m - 1):
        y64, a = orc.proj_quant_f64(x[r], raw, dtype, k, n)
        parity(y[r], y64, a)
        assert np.all(np.abs(y[r] - y64) <= bound * a) and np.all(np.abs(two[r] - y[r]) <= 2 * bound * a)


@pytest.mark.parametrize("dtype", [lh.Q4_K, lh.Q8_0])
@pytest.mark.parametrize("m", [2, 16, 31, 48, 64])
def test_bf16_is_one_part(ctx, dtype, m):
    """bf16 activations over 60 binary orders of magnitude: bit for bit the f32 call's result."""
    k, n = 1024, 90
    print(f"bf16 one part dtype={dtype} m={m}", flush=True)
    raw, w, keep = weights(ctx, dtype, k, n, m % 2, 0x5EED0B20)
    x = synth.normal(0x5EED0B21 + m, m * k) * np.exp2((np.arange(m * k) * 7 % 61 - 45).astype(np.float32))
    u = (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    xf = (u.astype(np.uint32) << 16).view(np.float32)
    a = product(ctx, lh.upload_bytes(ctx, u.view(np.uint8)), lh.BF16, w, k, n, m)
    b = product(ctx, lh.upload_f32(ctx, xf), lh.F32, w, k, n, m)
    assert np.all(np.isfinite(a)) and np.array_equal(a, b)


@pytest.mark.parametrize("dtype,m", [(lh.Q4_K, 40), (lh.Q8_0, 64)])
def test_wide_gate_up(ctx, dtype, m):
    k, n = 768, 130
    print(f"wide gate/up dtype={dtype} m={m}", flush=True)
    rg, wg, k1 = weights(ctx, dtype, k, n, 1, 0x5EED0B30)
    ru, wu, k2 = weights(ctx, dtype, k, n, 1, 0x5EED0B31)
    x = synth.normal(0x5EED0B32, m * k).reshape(m, k)
    hb, ub = lh.GpuBuffer(ctx, 4 * m * n), lh.GpuBuffer(ctx, 4 * m * n)
    lh.dispatch_silu_gate_up_batch(ctx, lh.upload_f32(ctx, x), wg[0], wu[0], hb, ub, k, n, m, wg[1])
    h = hb.read_f32(m * n).reshape(m, n).astype(np.float64)
    for r in (0, 31, 32, m - 1):
        g, _ = orc.proj_quant_f64(x[r], rg, dtype, k, n)
        u, _ = orc.proj_quant_f64(x[r], ru, dtype, k, n)
        want = dfo.silu_mul(g, u)
        assert np.max(np.abs(h[r] - want)) <= 1e-4 * np.max(np.abs(want))


@pytest.mark.parametrize("m,ctx_len", [(17, 40), (24, 0), (31, 70)])
def test_draft_blocks_of_34_to_62_rows(ctx, m, ctx_len):
    print(f"draft block m={m} ctx={ctx_len}", flush=True)
    model, (W, layers, feat, tok, kc, vc) = build(ctx, SMALL, 0x5EED0B40 + m, m, ctx_len, trained_scale=True)
    y = model.forward_block(feat, tok)
    check("forward_block", y, dfo.forward_block(feat, tok, W, layers, kc, vc, ctx_len, SMALL), TOL_FWD_TRAINED)
    assert np.array_equal(y, model.forward_block(feat, tok))
