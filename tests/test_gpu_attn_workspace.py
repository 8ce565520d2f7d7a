"""GPU: attention calls of different head counts in turn on one stream.  They share a
workspace whose arrival counters have to read zero whatever the previous call wrote behind
them; a group whose counter does not is never written."""
import ctypes

import numpy as np
import pytest

import dflash_oracle as dfo
import laguna_hip as lh
import synth
import target_oracle as tgo

pytestmark = pytest.mark.gpu

TOL = 1e-5


class Call:
    """One attention shape, its inputs and its oracle."""

    def __init__(self, ctx, n_q, n_kv, hd, rows, S, seed):
        self.shape, self.rows = (n_q, n_kv, hd, S), rows
        q = synth.normal(seed, rows * n_q * hd).reshape(rows, -1)
        K, V = (synth.normal(seed + i, S * n_kv * hd).reshape(S, -1) for i in (1, 2))
        self.bufs = [lh.upload_f32(ctx, a) for a in (q, K, V)] + [lh.GpuBuffer(ctx, q.nbytes)]
        self.want = dfo.attention(q, K, V, S - rows + np.arange(rows), n_q, n_kv, hd)
        self.ctx = ctx

    def run(self, stream):
        n_q, n_kv, hd, S = self.shape
        self.bufs[3].fill(0xFF)  # NaN: what the call does not write shows
        self.ctx.sync()
        lh.check(lh.lib().lg_dispatch_mha_attn(*(b.ptr for b in self.bufs), n_q, n_kv, hd, S, S - self.rows, self.rows, 1,
                                               stream.ptr))
        stream.sync()
        y = self.bufs[3].read_f32(self.want.size).reshape(self.want.shape)
        bad = int(np.sum(~np.isfinite(y)))
        e = float(np.max(np.abs(y - self.want)) / np.max(np.abs(self.want))) if not bad else np.inf
        print(f"  {self.shape} rows={self.rows}: {bad} of {y.size} unwritten, |err|inf/|y|inf = {e:.2e}", flush=True)
        assert bad == 0 and e <= TOL


# before: a call whose partials lie right behind few counters, over a workspace no smaller
# than the second call's; after: one with more counters than that
@pytest.mark.parametrize("before", [
    (32, 8, 128, 32, 4096),  # 64-query blocks
    (8, 2, 64, 9, 700), (8, 2, 256, 9, 700),
    (16, 8, 128, 2, 9000),   # a few queries: dots from memory
    (32, 8, 128, 16, 4096),  # 16-query groups, fewer of them
])
def test_counters_survive_other_head_counts(ctx, before):
    after = (32, 32, 128, 49, 256)  # 128 groups of 16 queries
    print(f"attention workspace: {before} between two calls of {after}", flush=True)
    a, b, s = Call(ctx, *after, 0x5EED0C00), Call(ctx, *before, 0x5EED0C10), lh.Stream()
    for c in (b, a, b, a, a):
        c.run(s)
    s.destroy()


def test_more_groups_than_counters(ctx):
    """4100 kv heads of 9 queries each: more groups than the counters' region is sized for."""
    print("attention workspace: 4100 kv heads", flush=True)
    c, s = Call(ctx, 4100, 4100, 128, 9, 12, 0x5EED0C40), lh.Stream()
    c.run(s)
    c.run(s)
    s.destroy()


def test_counters_survive_other_models(ctx):
    """Two targets of different widths, 16 query heads on one kv head, in turn on one stream."""
    models = []
    for i, (E, FF) in enumerate([(512, 512), (1024, 4096)]):
        args = dict(n_embd=E, n_heads=16, n_kv=1, head_dim=128, n_ff=FF, n_layers=2, n_vocab=300, rope_dim=128)
        cfg, hp = lh.TargetConfig(**args), tgo.Hparams(**args)
        layers, ex = synth.target_model(0x5EED0C20 + i, cfg)
        m = lh.TargetModel(ctx, cfg, layers, output_norm=ex["output_norm"], output=ex["output"],
                           output_dtype=ex["output_dtype"])
        models.append((m, hp, layers, ex))
    for step, i in enumerate((0, 1, 0, 1, 0)):
        m, hp, layers, ex = models[i]
        x = synth.normal(0x5EED0C30 + step, hp.n_embd)
        print(f"target {i} (n_embd {hp.n_embd}), step {step}", flush=True)
        lg, _ = m.forward_token(x, [])
        want, _ = tgo.forward_token(x, layers, hp, ex["output_norm"], ex["output"], ex["output_dtype"], [])
        e = float(np.max(np.abs(lg - want)) / np.max(np.abs(want)))
        print(f"  |err|inf/|y|inf = {e:.2e}", flush=True)
        assert e <= 2e-5  # test_gpu_target's bound
    for m, *_ in models:
        m.free()


@pytest.mark.parametrize("n_q,n_kv,hd,rows,S", [(32, 32, 64, 1, 65536), (64, 16, 256, 2, 20000), (8, 1, 128, 9, 200000)])
def test_workspace_of_long_sequences(ctx, n_q, n_kv, hd, rows, S):
    """A long sequence takes no more than its partials: a workgroup of 64 queries per CU."""
    print(f"attention workspace: {n_q}/{n_kv} heads of {hd}, {rows} rows, {S} positions", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    q, o = lh.GpuBuffer(ctx, 4 * rows * n_q * hd), lh.GpuBuffer(ctx, 4 * rows * n_q * hd)
    kv = [lh.GpuBuffer(ctx, 4 * S * n_kv * hd) for _ in range(2)]
    for b in (q, *kv):
        b.fill(0)
    o.fill(0xFF)
    ctx.sync()
    s = lh.Stream()
    before = free()
    lh.check(lh.lib().lg_dispatch_mha_attn(q.ptr, kv[0].ptr, kv[1].ptr, o.ptr, n_q, n_kv, hd, S, S - rows, rows, 1, s.ptr))
    s.sync()
    used = before - free()
    print(f"  {used / 1e6:.1f} MB", flush=True)
    assert not np.any(o.read_f32(rows * n_q * hd))  # weights of equal keys over zero values
    assert used <= 4 * (256 * 64 * (hd + 2) + 16384) + (4 << 20)  # allocation granularity
    s.destroy()
