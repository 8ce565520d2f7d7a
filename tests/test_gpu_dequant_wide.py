"""GPU: lg_dequant_to_f32 at the edges of its workgroups (4096 values, four a thread),
bit for bit against the oracle: remainders, unaligned inputs and outputs, truncated data."""
import numpy as np
import pytest

import laguna_hip as lh
import oracle as orc
import synth

pytestmark = pytest.mark.gpu


def want(raw, dtype, n):
    return orc.dequant_q4k(raw, n) if dtype == lh.Q4_K else orc.dequant_to_f32(raw, dtype, n)


@pytest.mark.parametrize("dtype", [lh.Q4_K, lh.Q8_0, lh.F16, lh.BF16, lh.F32])
@pytest.mark.parametrize("n,off_in,off_out,cut", [(4096, 0, 0, 0), (4097, 0, 0, 0), (8191, 0, 4, 0), (12291, 0, 0, 0),
                                                  (5120, 1, 0, 0), (5122, 2, 8, 0), (9000, 0, 0, 1500), (3, 0, 0, 0)])
def test_edges(ctx, dtype, n, off_in, off_out, cut):
    print(f"dequant dtype={dtype} n={n} in+{off_in} out+{off_out} cut={cut}", flush=True)
    if dtype == lh.Q4_K:
        raw = synth.q4k_weight(0x5EED0900 + n, 256, -(-n // 256))
    elif dtype == lh.Q8_0:
        raw = synth.q8_0_weight(0x5EED0901 + n, 32, -(-n // 32))
    elif dtype == lh.F32:
        raw = synth.normal(0x5EED0902 + n, n).view(np.uint8)
    else:  # every kind of half code, NaNs and subnormals among them
        raw = (np.arange(n, dtype=np.uint64) * 40503 % 65536).astype(np.uint16).view(np.uint8)
    raw = np.ascontiguousarray(raw).ravel()
    raw = raw[:raw.size - cut]
    src, dst = lh.GpuBuffer(ctx, raw.size + 32), lh.GpuBuffer(ctx, 4 * n + 32)
    src.fill(0x5A)
    dst.fill(0xFF)
    src.upload(raw, offset=off_in)
    lh.dequant_to_f32_device(ctx, src.ptr + off_in, raw.size, dtype, n, dst.ptr + off_out)
    got = dst.download().view(np.uint32)
    lo = off_out // 4
    assert np.array_equal(got[lo:lo + n], want(raw, dtype, n).view(np.uint32))
    assert np.all(got[:lo] == 0xFFFFFFFF) and np.all(got[lo + n:] == 0xFFFFFFFF)  # nothing beside the output
