// Q8_0, M = 1, rows of whole blocks in any number (k a multiple of 32; plain calls of k a
// multiple of 256 up to 4096 go to the integer-dot kernel), plain or with the fused
// silu(gate) * up input: proj_q80_rows.
#include <mutex>

#include "lg_common.hpp"

namespace {

using namespace lg;

// The workgroup holds the activations (FUSE: silu(x) * up, computed once) in LDS; each
// wavefront takes R rows at a time, lane u the half blocks u, u + 64, ...: 16 quants in one
// load (2-byte aligned, as the blocks are) and the block's scale, the next half block's in
// flight.  Every weight is q d and every product x (q d), as the reference's loop
// (kernels/proj_q8_0.comp:47-66), so non-finite values meet the same products.
//
// Against the element-wise path (one element per lane and step, each decoded from bytes):
// 14336 -> 4096 fused 196 -> 22.3 us, 6688 -> 1326 54 -> 6.0; against rows staged through
// each wavefront's LDS with the activations in registers, plain 14336 -> 4096 38.0 -> 20.5
// (62 MB, 3.0 TB/s).  At k <= 4096 the integer-dot kernel stays ahead (2816 -> 2880 4.3 us,
// here 5.1 at k = 2880).
constexpr int QR_WAVES = 8;
constexpr uint32_t QR_STRIDE = 20;  // floats per 16 staged activations: 16-byte reads of 16 lanes on distinct banks
constexpr uint32_t QR_K_MAX = 32768;  // 160 KiB of LDS

typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));

template <int R, bool FUSE>
__global__ __launch_bounds__(QR_WAVES * 64) void k_q80_rows(const float *__restrict__ x, const float *__restrict__ up,
                                                            const uint8_t *__restrict__ w, float *__restrict__ y,
                                                            uint32_t k, uint32_t n) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t units = k / 16, last = units - 1;
    const uint64_t row_bytes = (uint64_t)k / QK8_0 * Q80_BYTES;
    uint32_t row = (blockIdx.x * QR_WAVES + wave) * R;
    u32x4a2 q[2][R];
    uint32_t d[2][R];
    auto load = [&](int b, uint32_t row0, uint32_t u) __attribute__((always_inline)) {
        const uint32_t uc = u < units ? u : last;  // past the row: dropped
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t rr = row0 + r < n ? row0 + r : n - 1;  // past n: not stored
            const uint8_t *blk = w + rr * row_bytes + (uint64_t)(uc >> 1) * Q80_BYTES;
            d[b][r] = *reinterpret_cast<const uint16_t *>(blk);
            q[b][r] = *reinterpret_cast<const u32x4a2 *>(blk + 2 + 16 * (uc & 1u));
        }
    };
    if (row < n) load(0, row, lane);  // in flight while the activations are staged
    for (uint32_t e = threadIdx.x; e < k / 4; e += QR_WAVES * 64) {
        float4 v = reinterpret_cast<const float4 *>(x)[e];
        if constexpr (FUSE) {
            const float4 u = reinterpret_cast<const float4 *>(up)[e];
            v = make_float4(silu_mul(v.x, u.x), silu_mul(v.y, u.y), silu_mul(v.z, u.z), silu_mul(v.w, u.w));
        }
        *reinterpret_cast<float4 *>(xs + QR_STRIDE * (e >> 2) + 4 * (e & 3u)) = v;
    }
    __syncthreads();
    for (; row < n; row += gridDim.x * QR_WAVES * R) {  // uniform over the wavefront
        float acc[R][2];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = 0.0f;
        auto use = [&](int b, uint32_t u) __attribute__((always_inline)) {
            if (u >= units) return;
            float xv[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 t = *reinterpret_cast<const float4 *>(xs + QR_STRIDE * u + 4 * i);
                xv[4 * i] = t.x, xv[4 * i + 1] = t.y, xv[4 * i + 2] = t.z, xv[4 * i + 3] = t.w;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float df = ref_half(d[b][r]);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float wv = __fmul_rn((float)(int8_t)(q[b][r][i >> 2] >> (8 * (i & 3))), df);
                    acc[r][i & 1] = __builtin_fmaf(xv[i], wv, acc[r][i & 1]);
                }
            }
        };
        for (uint32_t u0 = 0; u0 < units; u0 += 128) {
            load(1, row, u0 + 64 + lane);
            use(0, u0 + lane);
            if (u0 + 128 < units) load(0, row, u0 + 128 + lane);
            else load(0, row + gridDim.x * QR_WAVES * R, lane);  // the next rows (past n: row n - 1)
            use(1, u0 + 64 + lane);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float s = wave_sum(acc[r][0] + acc[r][1]);
            if (lane == 0 && row + r < n) y[row + r] = s;
        }
    }
}

// Few rows: latency and idle CUs bound them, not bandwidth (16384 -> 275, 4.8 MB, is 16 steps of
// one wavefront a row on 35 workgroups above).  The eight wavefronts of a workgroup share R
// rows, thread t the half blocks t, t + 512, ..., its activations straight from memory (so few
// readers pay for no staging); four rows a workgroup lost to two (16384 -> 1024 6.4 against 6.3
// us, -> 512 6.0 against 4.3).
template <int R, bool FUSE>
__global__ __launch_bounds__(QR_WAVES * 64) void k_q80_split(const float *__restrict__ x, const float *__restrict__ up,
                                                             const uint8_t *__restrict__ w, float *__restrict__ y,
                                                             uint32_t k, uint32_t n) {
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t units = k / 16, row = blockIdx.x * R;
    const uint64_t row_bytes = (uint64_t)k / QK8_0 * Q80_BYTES;
    float acc[R][2];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = 0.0f;
    for (uint32_t u0 = threadIdx.x; u0 < units; u0 += 2 * QR_WAVES * 64) {
        u32x4a2 q[2][R];
        uint32_t d[2][R];
        float4 xv[2][4], uv[2][4];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t u = u0 + QR_WAVES * 64 * b < units ? u0 + QR_WAVES * 64 * b : u0;  // past the row: dropped
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t rr = row + r < n ? row + r : n - 1;  // past n: not stored
                const uint8_t *blk = w + rr * row_bytes + (uint64_t)(u >> 1) * Q80_BYTES;
                d[b][r] = *reinterpret_cast<const uint16_t *>(blk);
                q[b][r] = *reinterpret_cast<const u32x4a2 *>(blk + 2 + 16 * (u & 1u));
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                xv[b][i] = reinterpret_cast<const float4 *>(x)[4 * u + i];
                if constexpr (FUSE) uv[b][i] = reinterpret_cast<const float4 *>(up)[4 * u + i];
            }
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if (u0 + QR_WAVES * 64 * b >= units) break;
            float xe[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float4 v = xv[b][i];
                if constexpr (FUSE) {
                    const float4 u = uv[b][i];
                    v = make_float4(silu_mul(v.x, u.x), silu_mul(v.y, u.y), silu_mul(v.z, u.z), silu_mul(v.w, u.w));
                }
                xe[4 * i] = v.x, xe[4 * i + 1] = v.y, xe[4 * i + 2] = v.z, xe[4 * i + 3] = v.w;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float df = ref_half(d[b][r]);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float wv = __fmul_rn((float)(int8_t)(q[b][r][i >> 2] >> (8 * (i & 3))), df);
                    acc[r][i & 1] = __builtin_fmaf(xe[i], wv, acc[r][i & 1]);
                }
            }
        }
    }
    __shared__ float part[QR_WAVES][R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float s = wave_sum(acc[r][0] + acc[r][1]);
        if (lane == 0) part[wave][r] = s;
    }
    __syncthreads();
    if (threadIdx.x < R && row + threadIdx.x < n) {
        float s = part[0][threadIdx.x];
#pragma unroll
        for (int v = 1; v < QR_WAVES; v++) s += part[v][threadIdx.x];
        y[row + threadIdx.x] = s;
    }
}

std::mutex g_mu;
bool g_attr[64][2][2] = {};

template <int R, bool FUSE>
int launch(const float *x, const float *up, const uint8_t *w, float *y, uint32_t k, uint32_t n, hipStream_t s) {
    int dev = 0;
    LG_HIP_TRY(hipGetDevice(&dev));
    LG_REQUIRE(dev >= 0 && dev < 64, "proj_q8_0_rows: device %d", dev);
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (!g_attr[dev][R - 1][FUSE]) {
            LG_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_q80_rows<R, FUSE>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)(QR_K_MAX / 16 * QR_STRIDE * 4)));
            g_attr[dev][R - 1][FUSE] = true;
        }
    }
    const uint32_t per = QR_WAVES * R, cap = 2 * (uint32_t)device_cus(), want = (n + per - 1) / per;
    hipLaunchKernelGGL((k_q80_rows<R, FUSE>), dim3(want < cap ? want : cap), dim3(QR_WAVES * 64), k / 16 * QR_STRIDE * 4, s,
                       x, up, w, y, k, n);
    return after_launch("proj_q8_0_rows", s);
}

}  // namespace

namespace lg {

bool proj_q80_rows_ok(uint32_t k, uint32_t n, const float *x, const float *up, const void *w) {
    auto mis = [](const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; };
    return k && k % QK8_0 == 0 && k <= QR_K_MAX && n <= 0x7FFFFFFFu && !mis(x, 16) && !mis(up, 16) && !mis(w, 2);
}

int proj_q80_rows(const float *x, const float *up, const void *w, float *y, uint32_t k, uint32_t n, hipStream_t s) {
    const uint8_t *wb = static_cast<const uint8_t *>(w);
    // fewer rows than keep the chip busy at one wavefront each: a workgroup per row (a CU's
    // worth of rows or less) or two.  Plain, 16384 -> 256 10.1 -> 3.9 us, -> 3072 18.3 -> 16.3,
    // 5120 -> 3072 6.9 -> 6.1, -> 16000 21.7 against 24.7 here; fused, 14336 -> 1024 11.3 -> 10.4,
    // -> 2048 11.5 against 20.8: each row repeats the SiLU
    const uint32_t cus = (uint32_t)device_cus();
    if (n < (up ? 4u * cus + 1 : 16u * cus)) {
        const dim3 b(QR_WAVES * 64);
        if (n <= cus) {
            if (up) hipLaunchKernelGGL((k_q80_split<1, true>), dim3(n), b, 0, s, x, up, wb, y, k, n);
            else hipLaunchKernelGGL((k_q80_split<1, false>), dim3(n), b, 0, s, x, up, wb, y, k, n);
        } else {
            if (up) hipLaunchKernelGGL((k_q80_split<2, true>), dim3((n + 1) / 2), b, 0, s, x, up, wb, y, k, n);
            else hipLaunchKernelGGL((k_q80_split<2, false>), dim3((n + 1) / 2), b, 0, s, x, up, wb, y, k, n);
        }
        return after_launch("proj_q8_0_split", s);
    }
    // two rows a wavefront share the reads of x once every CU has its eight wavefronts
    if (!up) return launch<2, false>(x, up, wb, y, k, n, s);
    return n >= 16u * cus ? launch<2, true>(x, up, wb, y, k, n, s) : launch<1, true>(x, up, wb, y, k, n, s);
}

}  // namespace lg
