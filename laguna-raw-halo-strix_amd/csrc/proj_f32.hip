// f32 weights, small M (1 < m <= 64): proj_f32_mm.
#include "lg_common.hpp"

namespace {

using namespace lg;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Exact f32 products (v_mfma_f32_16x16x4f32) straight from memory: k a multiple of 4,
// 16-byte aligned operands.  A workgroup owns RT 16-row tiles and all of k; its four
// wavefronts take 64-element blocks of k in turn, so that no element of W or x is read
// twice by a workgroup and nothing leaves it (no workspace): the wavefronts' sums meet in
// LDS in wavefront order.  Lane (l16, kg) loads elements 16 s + 4 kg .. + 3 of weight row
// l16 (and of token row l16) as one float4, component c supplying k step c of both
// operands; the next block is in flight.  Each block is summed by itself, in eight chains of
// two matrix instructions that meet pairwise, before it joins the wavefront's sum: rows of 512
// are then 8.7e-8 off (2-norm), of 4096 1.1e-7, no more than one element a lane and step
// (8.6e-8, 1.6e-7).  Two chains of eight a block: 1.17e-7 and 1.37e-7, in the same time; one
// chain over all blocks 3.6 times the error of that.
//
// Memory bound, and slower with more requests in flight: 4096 -> 4096 at m = 16 20.0 us
// (67 MB, 3.4 TB/s; the element-wise path 381, a plain read 10.7), with a third block held
// 20.8, a fourth 21.5, with eight wavefronts 20.1 (and 61.5 against 56.1 at k = 14336),
// with 16 22.9, nontemporal weight loads 25.1, the weights staged through LDS in whole rows
// 20.7; taking the matrix products out changes nothing.
constexpr int FM_WAVES = 4;

template <int TT, int RT, bool XB>
__global__ __launch_bounds__(FM_WAVES * 64) void k_f32_mm(const void *__restrict__ x, const float *__restrict__ w,
                                                          float *c, const float *res, uint32_t m, uint32_t k,
                                                          uint32_t n) {
    __shared__ f32x4 part[FM_WAVES][RT * TT][64];
    const uint32_t lane = threadIdx.x & 63u, l16 = lane & 15u, kg = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t row0 = blockIdx.x * 16 * RT, nb = (k + 63) / 64;
    const float *wr[RT];  // rows past n read row n - 1, tokens past m token m - 1 (never stored)
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const uint32_t row = row0 + 16 * i + l16;
        wr[i] = w + (uint64_t)(row < n ? row : n - 1) * k;
    }
    uint64_t xr[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) xr[t] = (uint64_t)(16 * t + l16 < m ? 16 * t + l16 : m - 1) * k;
    typedef uint32_t xraw __attribute__((ext_vector_type(XB ? 2 : 4)));
    f32x4 W[2][RT][4];
    xraw X[2][TT][4];
    auto load = [&](int b, uint32_t blk) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint32_t e0 = 64 * blk + 16 * s + 4 * kg, e = e0 < k ? e0 : 0;  // past k: masked when used
#pragma unroll
            for (int i = 0; i < RT; i++) W[b][i][s] = *reinterpret_cast<const f32x4 *>(wr[i] + e);
#pragma unroll
            for (int t = 0; t < TT; t++)
                X[b][t][s] = *reinterpret_cast<const xraw *>(static_cast<const uint8_t *>(x) + (XB ? 2 : 4) * (xr[t] + e));
        }
    };
    f32x4 acc[RT][TT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // this wavefront's blocks wave, wave + FM_WAVES, ...; past the last the loads repeat it
    const uint32_t mine = nb > wave ? (nb - wave + FM_WAVES - 1) / FM_WAVES : 0;
    auto blk = [&](uint32_t i) { i = i < mine ? i : mine - 1; return wave + FM_WAVES * i; };
    if (mine) {
        load(0, blk(0));
        for (uint32_t i0 = 0; i0 < mine; i0 += 2) {
#pragma unroll
            for (int b = 0; b < 2; b++) {
                if (i0 + b >= mine) break;  // uniform over the wavefront
                load(b ^ 1, blk(i0 + b + 1));
                __builtin_amdgcn_sched_barrier(0);
                const uint32_t cur = blk(i0 + b);
                if (64 * cur + 64 > k) {  // uniform: a partial last block, both operands 0 past k
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        const bool ok = 64 * cur + 16 * s + 4 * kg < k;
#pragma unroll
                        for (int i = 0; i < RT; i++) W[b][i][s] = ok ? W[b][i][s] : (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int t = 0; t < TT; t++) X[b][t][s] = ok ? X[b][t][s] : (xraw)(0u);
                    }
                }
                f32x4 sum[RT][TT][2];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    f32x4 ch[RT][TT][2];
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int t = 0; t < TT; t++) {
                            float xv;
                            if constexpr (XB) xv = __uint_as_float(j & 1 ? X[b][t][s][j / 2] & 0xFFFF0000u : X[b][t][s][j / 2] << 16);
                            else xv = __uint_as_float(X[b][t][s][j]);
#pragma unroll
                            for (int i = 0; i < RT; i++)
                                ch[i][t][j % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                    xv, W[b][i][s][j], j < 2 ? (f32x4){0.f, 0.f, 0.f, 0.f} : ch[i][t][j % 2], 0, 0, 0);
                        }
#pragma unroll
                    for (int i = 0; i < RT; i++)
#pragma unroll
                        for (int t = 0; t < TT; t++) {
                            const f32x4 c = ch[i][t][0] + ch[i][t][1];
                            sum[i][t][s >> 1] = s & 1 ? sum[i][t][s >> 1] + c : c;
                        }
                }
#pragma unroll
                for (int i = 0; i < RT; i++)
#pragma unroll
                    for (int t = 0; t < TT; t++) acc[i][t] += sum[i][t][0] + sum[i][t][1];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int t = 0; t < TT; t++) part[wave][i * TT + t][lane] = acc[i][t];
    __syncthreads();
    // tile (i, t) of wavefront w: lane (l16, kg) holds tokens 16 t + 4 kg + r of row l16
    for (int it = wave; it < RT * TT; it += FM_WAVES) {
        f32x4 v = part[0][it][lane];
#pragma unroll
        for (int q = 1; q < FM_WAVES; q++) v += part[q][it][lane];
        const uint32_t row = row0 + 16 * (it / TT) + l16, t0 = 16 * (it % TT) + 4 * kg;
        if (row < n)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (t0 + r < m) {
                    const uint64_t o = (uint64_t)(t0 + r) * n + row;
                    c[o] = res ? res[o] + v[r] : v[r];
                }
    }
}

template <int TT, int RT>
void launch_f32(const void *x, bool bf16, const float *w, float *c, const float *res, uint32_t m, uint32_t k, uint32_t n,
                hipStream_t s) {
    const dim3 grid((n + 16 * RT - 1) / (16 * RT)), block(FM_WAVES * 64);
    if (bf16) hipLaunchKernelGGL((k_f32_mm<TT, RT, true>), grid, block, 0, s, x, w, c, res, m, k, n);
    else hipLaunchKernelGGL((k_f32_mm<TT, RT, false>), grid, block, 0, s, x, w, c, res, m, k, n);
}

template <int TT>
void launch_f32_tt(const void *x, bool bf16, const float *w, float *c, const float *res, uint32_t m, uint32_t k,
                   uint32_t n, hipStream_t s) {
    // two row tiles (half the reads of x) when that still gives a workgroup per CU: 4096 ->
    // 14336 at m = 16 63.3 against 72.8 us; from 33 tokens the registers hold one
    if constexpr (TT <= 2)
        if ((n + 31) / 32 >= (uint32_t)device_cus()) {
            launch_f32<TT, 2>(x, bf16, w, c, res, m, k, n, s);
            return;
        }
    launch_f32<TT, 1>(x, bf16, w, c, res, m, k, n, s);
}

}  // namespace

namespace lg {

int proj_f32_mm(const void *x, bool bf16, const float *w, float *c, const float *res, uint32_t m, uint32_t k, uint32_t n,
                  hipStream_t s) {
    if (m <= 16) launch_f32_tt<1>(x, bf16, w, c, res, m, k, n, s);
    else if (m <= 32) launch_f32_tt<2>(x, bf16, w, c, res, m, k, n, s);
    else if (m <= 48) launch_f32_tt<3>(x, bf16, w, c, res, m, k, n, s);
    else launch_f32_tt<4>(x, bf16, w, c, res, m, k, n, s);
    return after_launch("proj_f32_mm", s);
}

}  // namespace lg
