"""GPU: attention of many queries per kv head, and of head sizes 64 and 256, against the
f64 oracle.  The kernel takes blocks of 64 queries over tiles of 32 positions, in one
chunk or several, on f16 parts of its operands (1e-5 of the largest result, as the other
matrix-core attention: measured below 2e-6); a tile that those parts cannot hold goes
element by element.  And the kernels beside it: 16 queries per workgroup (a strong key,
huge values), one wavefront per query."""
import ctypes

import numpy as np
import pytest

import dflash_oracle as dfo
import laguna_hip as lh
import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def inputs(n_q, n_kv, hd, rows, S, seed):
    return (synth.normal(seed, rows * n_q * hd).reshape(rows, -1), synth.normal(seed + 1, S * n_kv * hd).reshape(S, -1),
            synth.normal(seed + 2, S * n_kv * hd).reshape(S, -1))


def run(ctx, q, K, V, n_q, n_kv, hd, q_pos, causal=1):
    qb, kb, vb = lh.upload_f32(ctx, q), lh.upload_f32(ctx, K), lh.upload_f32(ctx, V)
    ob = lh.GpuBuffer(ctx, q.nbytes)
    lh.dispatch_mha_attn_seq(ctx, qb, kb, vb, ob, n_q, n_kv, hd, K.shape[0], q_pos, rows=q.shape[0], causal=causal)
    return ob.read_f32(q.size).reshape(q.shape)


def check(y, want, tol=TOL):
    assert np.all(np.isfinite(y))
    e = float(np.max(np.abs(y - want)) / np.max(np.abs(want)))
    print(f"  |err|inf/|y|inf = {e:.2e}", flush=True)
    assert e <= tol


@pytest.mark.parametrize("n_q,n_kv,hd,rows,S,q_pos,causal", [
    (8, 2, 128, 17, 1, 0, 1),        # one position; 68 queries: a second block of four
    (8, 8, 128, 65, 65, 0, 1),       # a whole causal triangle, one past a block and two tiles
    (32, 8, 128, 32, 4095, 4063, 1),  # chunks merged, a ragged last tile
    (4, 1, 128, 64, 96, 31, 0),      # not causal
    (2, 2, 128, 130, 700, 600, 1),   # rows that see past the sequence's end
    (4, 4, 64, 1, 33, 32, 1), (8, 2, 64, 20, 515, 400, 1),
    (2, 1, 256, 1, 31, 30, 1), (8, 2, 256, 33, 300, 250, 1),
    (64, 1, 128, 2, 200, 198, 1),    # 64 heads of one kv head
])
def test_attention_rows(ctx, n_q, n_kv, hd, rows, S, q_pos, causal):
    print(f"attn n_q={n_q} n_kv={n_kv} hd={hd} rows={rows} S={S} q_pos={q_pos} causal={causal}", flush=True)
    q, K, V = inputs(n_q, n_kv, hd, rows, S, 0x5EED0700 + S)
    y = run(ctx, q, K, V, n_q, n_kv, hd, q_pos, causal)
    check(y, dfo.attention(q, K, V, q_pos + np.arange(rows), n_q, n_kv, hd, causal=bool(causal)))
    assert np.array_equal(y, run(ctx, q, K, V, n_q, n_kv, hd, q_pos, causal))


# two and three, seven and eight, and whole numbers of tiles a chunk (256 CUs): both LDS buffers,
# tiles loaded ahead, a ragged end
@pytest.mark.parametrize("n_q,n_kv,hd,rows,S", [
    (32, 8, 64, 32, 1503), (64, 32, 64, 5, 2000), (16, 16, 64, 3, 1024),
    (32, 8, 256, 32, 1503), (64, 32, 256, 5, 2000), (16, 16, 256, 3, 1024),
    (32, 8, 128, 32, 1503), (64, 32, 128, 33, 1984),
])
def test_attention_rows_tiles(ctx, n_q, n_kv, hd, rows, S):
    print(f"attn rows tiles n_q={n_q} n_kv={n_kv} hd={hd} rows={rows} S={S}", flush=True)
    q, K, V = inputs(n_q, n_kv, hd, rows, S, 0x5EED0710 + S)
    y = run(ctx, q, K, V, n_q, n_kv, hd, S - rows)
    check(y, dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd))
    assert np.array_equal(y, run(ctx, q, K, V, n_q, n_kv, hd, S - rows))


# positions in the first, second and third tile of a chunk of three (256 CUs: tiles 2, 3, 4)
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("at", [70, 100, 150])
@pytest.mark.parametrize("case", ["k_wide", "k_ninf", "v_wide", "v_inf", "v_zero"])
def test_attention_rows_mixed_chunk(ctx, hd, at, case):
    """A tile for the element-wise path (or of zeros) among others of its chunk."""
    n_q, n_kv, rows, S = 32, 8, 20, 1503
    print(f"attn rows mixed chunk hd={hd} at={at}: {case}", flush=True)
    q, K, V = (a.reshape(a.shape[0], -1, hd) for a in inputs(n_q, n_kv, hd, rows, S, 0x5EED0730))
    sees = np.ones((rows, n_q, hd), bool)
    if case == "k_wide":
        q[:, :, 5] = 0.0
        K[at, 2, 5] = 7.0e30
    elif case == "k_ninf":
        q[:, :, 0] = np.abs(q[:, :, 0]) + 1.0
        K[at, :, 0] = -np.inf
    elif case == "v_wide":
        V[at, 1, 17] = 7.0e4
    elif case == "v_inf":
        V[at, 0, 3] = np.inf
        sees[:, :4, 3] = False
    else:
        V[at // 32 * 32:at // 32 * 32 + 32] = 0.0
    q, K, V = q.reshape(rows, -1), K.reshape(S, -1), V.reshape(S, -1)
    y = run(ctx, q, K, V, n_q, n_kv, hd, S - rows).reshape(sees.shape)
    ko, vo = np.where(np.isneginf(K), -1e30, K), np.where(np.isfinite(V), V, 0.0)
    with np.errstate(all="ignore"):
        want = dfo.attention(q, ko, vo, S - rows + np.arange(rows), n_q, n_kv, hd).reshape(sees.shape)
    check(y[sees], want[sees])
    if case == "v_inf":
        assert np.all(np.isposinf(y[~sees]))
    if case == "v_wide":  # the other dims are held to their own size
        check(np.delete(y, 17, axis=2), np.delete(want, 17, axis=2))


@pytest.mark.parametrize("n_q,n_kv,hd,rows,S,off", [
    (4, 2, 96, 3, 50, 0), (8, 2, 80, 17, 130, 0), (2, 2, 192, 5, 77, 0), (3, 1, 20, 2, 9, 0),
    (8, 2, 64, 20, 130, 4), (8, 2, 128, 20, 130, 4), (4, 4, 256, 3, 65, 4), (32, 8, 128, 4, 100, 8),
])
def test_attention_wavefront_per_query(ctx, n_q, n_kv, hd, rows, S, off):
    """The plain kernel: other head sizes, and operands that are not 16-byte aligned."""
    print(f"attn plain n_q={n_q} n_kv={n_kv} hd={hd} rows={rows} S={S} off={off}", flush=True)
    q, K, V = inputs(n_q, n_kv, hd, rows, S, 0x5EED0750 + S)
    bufs = []
    for a in (q, K, V, np.zeros_like(q)):
        b = lh.GpuBuffer(ctx, a.nbytes + off)
        b.fill(0xFF)
        b.upload(np.ascontiguousarray(a, np.float32), off)
        bufs.append(b)
    st = lh.lib().lg_dispatch_mha_attn(*(b.ptr + off for b in bufs), n_q, n_kv, hd, S, S - rows, rows, 1, ctx.stream)
    lh.check(st)
    y = bufs[3].read_f32(q.size + off // 4)[off // 4:].reshape(q.shape)
    check(y, dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd))


@pytest.mark.parametrize("case", ["k_wide", "k_small", "q_wide", "v_wide", "v_small", "masked_nan", "v_inf", "k_ninf"])
def test_attention_rows_range(ctx, case):
    n_q, n_kv, hd, rows, S, q_pos = 32, 8, 128, 20, 300, 275
    print(f"attn rows range: {case}", flush=True)
    q, K, V = (a.reshape(a.shape[0], -1, hd) for a in inputs(n_q, n_kv, hd, rows, S, 0x5EED0720))
    sees = np.ones((rows, n_q, hd), bool)
    if case == "k_wide":  # a key far above f16's range against zero query elements
        q[:, :, 5] = 0.0
        K[37, 2, 5] = 7.0e30
    elif case == "k_small":  # keys far below f16's, queries as far above
        K *= np.float32(2.0 ** -60)
        q *= np.float32(2.0 ** 60)
    elif case == "q_wide":
        K[:, :, 9] = 0.0
        q[3, 9, 9] = 7.0e30
    elif case == "v_wide":
        V[100, 1, 17] = 7.0e30
    elif case == "v_small":
        V *= np.float32(2.0 ** -30)
    elif case == "masked_nan":  # rows 0 .. 4 do not see position 280, no row sees 296 ..
        V[280, 3, 7] = np.nan
        K[296:], V[296:] = np.nan, np.inf
        sees[5:, 12:16] = False  # the rows whose kv head 3 meets the NaN
    elif case == "v_inf":
        V[50, 0, 3] = np.inf
        sees[:, :4, 3] = False
    else:  # a key of -inf against positive queries: weight 0
        q[:, :, 0] = np.abs(q[:, :, 0]) + 1.0
        K[60, :, 0] = -np.inf
    q, K, V = q.reshape(rows, -1), K.reshape(S, -1), V.reshape(S, -1)
    y = run(ctx, q, K, V, n_q, n_kv, hd, q_pos).reshape(sees.shape)
    ko, vo = K.copy(), V.copy()
    ko[296:], vo[296:] = (0.0, 0.0) if case == "masked_nan" else (ko[296:], vo[296:])
    with np.errstate(all="ignore"):
        ko = np.where(np.isneginf(ko), -1e30, ko)
        vo = np.where(np.isfinite(vo), vo, 0.0)
        want = dfo.attention(q, ko, vo, q_pos + np.arange(rows), n_q, n_kv, hd).reshape(sees.shape)
    check(y[sees], want[sees])
    if case == "v_inf":
        assert np.all(np.isposinf(y[~sees]))
    if case == "masked_nan":  # element by element: only the NaN's own dim, in the rows that see it
        assert np.all(np.isnan(y[5:, 12:16, 7])) and np.all(np.isfinite(np.delete(y, 7, axis=2)))


# several tiles a chunk (16 / 8 / 9 on 256 CUs), so that weights meet a running maximum
SINK_SHAPES = [(64, 64, 64, 3, 2048), (64, 16, 128, 20, 2048), (32, 32, 256, 2, 2304)]

# An exponent below 32 (base 2) is rounded at most three times on its way to a weight, 2^-20
# each: 3 * 2^-20 * ln 2 of the weight; what the parts of weights and values add lies below.
WEIGHT_TOL = 2.5e-6


def sink_inputs(n_q, n_kv, hd, rows, S, nats, at):
    """One key far above the others whose value row is zero: the result is made of the
    small weights alone."""
    q, K, V = (a.reshape(a.shape[0], -1, hd) for a in inputs(n_q, n_kv, hd, rows, S, 0x5EED0760 + hd))
    q[:, :, 0], K[:, :, 0] = 2.0, 0.0
    K[at], V[at] = 0.0, 0.0
    K[at, :, 0] = (nats + 3.5) * np.sqrt(hd) / 2.0  # the others reach about 3.5
    return q.reshape(rows, -1), K.reshape(S, -1), V.reshape(S, -1)


@pytest.mark.parametrize("n_q,n_kv,hd,rows,S", SINK_SHAPES)
@pytest.mark.parametrize("nats", [9, 12, 16])
def test_attention_rows_sink(ctx, n_q, n_kv, hd, rows, S, nats):
    q, K, V = sink_inputs(n_q, n_kv, hd, rows, S, nats, 5)
    print(f"attn rows sink hd={hd} {nats} nats", flush=True)
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd)
    check(run(ctx, q, K, V, n_q, n_kv, hd, S - rows), want, WEIGHT_TOL)


@pytest.mark.parametrize("n_q,n_kv,hd,rows,S", SINK_SHAPES)
@pytest.mark.parametrize("top", [0, 12])
def test_attention_rows_unequal_dims(ctx, n_q, n_kv, hd, rows, S, top):
    """Value dimensions of very different magnitude, each held to its own largest result."""
    q, K, V = inputs(n_q, n_kv, hd, rows, S, 0x5EED0780 + hd)
    scale = np.exp2(top - np.arange(hd) * 37 % 29).astype(np.float32)  # over 28 binary orders
    V = (V.reshape(S, n_kv, hd) * scale).reshape(S, -1)
    print(f"attn rows unequal dims hd={hd} from 2^{top}", flush=True)
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd).reshape(-1, hd)
    y = run(ctx, q, K, V, n_q, n_kv, hd, S - rows).reshape(-1, hd)
    check(y / scale, want / scale, WEIGHT_TOL)


def test_attention_rows_first_call_captured(ctx):
    """A capture on a stream that has no workspace yet: the sequence is taken whole, and
    the graph's result is the eager one's within rounding."""
    n_q, n_kv, hd, rows, S = 32, 8, 128, 32, 1000
    print("attn rows captured before any call on the stream", flush=True)
    q, K, V = inputs(n_q, n_kv, hd, rows, S, 0x5EED0740)
    hip = ctypes.CDLL("libamdhip64.so")
    vp = ctypes.c_void_p
    hip.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    hip.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]
    hip.hipGraphLaunch.argtypes, hip.hipGraphExecDestroy.argtypes, hip.hipGraphDestroy.argtypes = [vp, vp], [vp], [vp]
    qb, kb, vb = lh.upload_f32(ctx, q), lh.upload_f32(ctx, K), lh.upload_f32(ctx, V)
    ob = lh.GpuBuffer(ctx, q.nbytes)
    run(ctx, q, K, V, n_q, n_kv, hd, S - rows)  # the kernel is loaded (on the null stream)
    s, g, ge = lh.Stream(), vp(), vp()
    assert hip.hipStreamBeginCapture(s.ptr, 1) == 0
    st = lh.lib().lg_dispatch_mha_attn(qb.ptr, kb.ptr, vb.ptr, ob.ptr, n_q, n_kv, hd, S, S - rows, rows, 1, s.ptr)
    assert hip.hipStreamEndCapture(s.ptr, ctypes.byref(g)) == 0
    lh.check(st)
    assert hip.hipGraphInstantiate(ctypes.byref(ge), g, None, None, 0) == 0
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd)
    for rep in range(3):
        ob.fill(0xFF)
        ctx.sync()
        assert hip.hipGraphLaunch(ge, s.ptr) == 0
        s.sync()
        check(ob.read_f32(q.size).reshape(q.shape), want)
        check(run(ctx, q, K, V, n_q, n_kv, hd, S - rows), want)
    hip.hipGraphExecDestroy(ge)
    hip.hipGraphDestroy(g)
    s.destroy()


@pytest.mark.parametrize("hd,rows,S", [(64, 3, 40), (64, 40, 700), (256, 3, 40), (256, 40, 700),
                                       (128, 70, 2000)])
def test_attention_rows_large_close_scores(ctx, hd, rows, S):
    """Scores of several thousand, exact in f32, half apart: only their differences count."""
    n_q, n_kv = 4, 4
    q, K, V = (a.reshape(a.shape[0], -1, hd) for a in inputs(n_q, n_kv, hd, rows, S, 0x5EED07C0))
    q[:], K[:] = 0.0, 0.0
    q[:, :, 0] = 64.0
    # of q . k: 64 times a multiple of 2^-8 (heads of 128: their scores lie 0.35 apart)
    K[:, :, 0] = (12000.0 + 4.0 * (np.arange(S) % 7)[:, None]) * 2.0 ** (np.log2(hd) // 2) / 512.0
    q, K, V = q.reshape(rows, -1), K.reshape(S, -1), V.reshape(S, -1)
    print(f"attn rows large close scores hd={hd} S={S}", flush=True)
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd)
    check(run(ctx, q, K, V, n_q, n_kv, hd, S - rows), want, WEIGHT_TOL)


# 9 to 64 queries per kv head of 128: 16 to a workgroup, the sequence over its wavefronts
@pytest.mark.parametrize("n_q,n_kv,rows,S", [(32, 8, 16, 2048), (64, 64, 9, 700)])
@pytest.mark.parametrize("nats", [9, 12, 16])
@pytest.mark.parametrize("at", [0, 5, 300])
def test_attention_groups_sink(ctx, n_q, n_kv, rows, S, nats, at):
    q, K, V = sink_inputs(n_q, n_kv, 128, rows, S, nats, at)
    print(f"attn groups sink n_kv={n_kv} {nats} nats at {at}", flush=True)
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, 128)
    # a weight is held to 2^-39 of the key's where both meet in one wavefront, a tenth of the
    # positions at most
    tol = WEIGHT_TOL + 0.1 * 2.0 ** -39 * np.exp(nats + 3.5)
    check(run(ctx, q, K, V, n_q, n_kv, 128, S - rows), want, tol)


def test_attention_groups_huge_value(ctx):
    """A value of 3e37 beside ordinary ones: no unit of the weights may overflow it."""
    n_q, n_kv, rows, S = 32, 8, 16, 500
    q, K, V = inputs(n_q, n_kv, 128, rows, S, 0x5EED07A0)
    V = V.reshape(S, n_kv, 128)
    V[100, 3, 17] = 3.0e37
    V = V.reshape(S, -1)
    print("attn groups huge value", flush=True)
    want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, 128)
    y = run(ctx, q, K, V, n_q, n_kv, 128, S - rows)
    check(y, want)
    big = np.abs(want) > 1e30
    check(y[~big], want[~big])
