// Whole-tensor dequantization on the device: lg_dequant_to_f32.
//
// Reference: dequant_to_f32 (src/dflash.rs:331-465), a serial CPU loop run at
// model load.  Q8_0 follows its branch (:379-397); Q4_K follows the ggml decode
// of kernels/proj_q4k.comp:28-87 (the Rust Q4_K branch is a different format).
// Both products are exact in f32 (f16 d has 11 significant bits, sc <= 63,
// q <= 15, |int8| <= 128), so `(d*sc)*q - dmin*m` rounds once, at the
// subtraction, and the result is bit-identical to the reference for every
// non-NaN input; __fmul_rn/__fsub_rn keep the compiler from reassociating.
#include "lg_common.hpp"

namespace {

using namespace lg;

// Four consecutive values per thread, DQ_UNITS times: a wavefront's store is 1 KiB of
// contiguous f32 (and, Q4_K, one super-block), whatever the format.  The stores are most
// of the traffic (4 bytes against 0.56 to 2 read), so their layout sets the rate: with a
// block of 32 or a 16-byte quant chunk per thread, its stores 64 or 128 bytes apart, 58.7 M
// values took Q8_0 95 us and Q4_K 76.6, now 42.7 (7.0 TB/s) and 38.7; with ordinary instead
// of nontemporal stores 65.2 and 51.5.
constexpr uint32_t DQ_UNITS = 4, DQ_WG = DQ_UNITS * 1024;  // values per workgroup

// Values e .. e + 3 (those below n) of out.
__device__ __forceinline__ void dq_store(float *out, uint64_t e, uint64_t n, const float (&v)[4], int vec_out) {
    if (vec_out && e + 4 <= n) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store((f32x4){v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4 *>(out + e));
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (e + i < n) out[e + i] = v[i];
    }
}

__global__ __launch_bounds__(256) void k_dequant_q4k(const uint8_t *__restrict__ data,
                                                     uint64_t blocks_avail, uint64_t n,
                                                     float *__restrict__ out, int vec_out) {
    const uint64_t e0 = (uint64_t)blockIdx.x * DQ_WG + 4u * threadIdx.x;
    const uint32_t w = 4u * (threadIdx.x & 63u), g = w >> 6, hi = (w >> 5) & 1u;  // this thread's place in its super-block
    uint4 hd[DQ_UNITS];
    uint32_t qs[DQ_UNITS];
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t b = (e0 + 1024u * u) / QK_K;
        if (b < blocks_avail) {
            const uint8_t *blk = data + b * Q4K_BYTES;
            hd[u] = *reinterpret_cast<const uint4 *>(blk);
            qs[u] = *reinterpret_cast<const uint32_t *>(blk + 16 + 32 * g + (w & 31u));
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t e = e0 + 1024u * u, b = e / QK_K;
        if (e >= n) break;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (b < blocks_avail) {
            uint32_t sc, mn;
            scale_min_k4(2 * g + hi, hd[u].y, hd[u].z, hd[u].w, sc, mn);
            const float a = __fmul_rn(ref_half(hd[u].x & 0xFFFFu), (float)sc);
            const float c = __fmul_rn(ref_half(hd[u].x >> 16), (float)mn);
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[i] = __fsub_rn(__fmul_rn(a, (float)((qs[u] >> (8 * i + 4 * hi)) & 15u)), c);
        }
        dq_store(out, e, n, v, vec_out);
    }
}

// Byte-addressed variant for a tensor base that is not 16-byte aligned.
__global__ __launch_bounds__(256) void k_dequant_q4k_bytes(const uint8_t *__restrict__ data,
                                                           uint64_t blocks_avail, uint64_t n,
                                                           float *__restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t b = i / QK_K;
    if (b >= blocks_avail) {
        out[i] = 0.0f;
        return;
    }
    const uint8_t *blk = data + b * Q4K_BYTES;
    const uint32_t e = i % QK_K, j = e / 32, g = e / 64, w = e % 64;
    uint32_t s[3];
    for (int t = 0; t < 3; t++)
        s[t] = blk[4 + 4 * t] | (blk[5 + 4 * t] << 8) | (blk[6 + 4 * t] << 16) | ((uint32_t)blk[7 + 4 * t] << 24);
    uint32_t sc, mn;
    scale_min_k4(j, s[0], s[1], s[2], sc, mn);
    const float d = ref_half(blk[0] | (blk[1] << 8)), dmin = ref_half(blk[2] | (blk[3] << 8));
    const uint32_t byte = blk[16 + 32 * g + (w % 32)];
    const float q = (float)(w < 32 ? (byte & 15u) : (byte >> 4));
    out[i] = __fsub_rn(__fmul_rn(__fmul_rn(d, (float)sc), q), __fmul_rn(dmin, (float)mn));
}

// value = float(q) * d (src/dflash.rs:389-394).  A2: the tensor's base is 2-byte aligned
// (blocks of 34 bytes keep that).
template <bool A2>
__device__ __forceinline__ uint32_t dq_u16(const uint8_t *p) {
    if constexpr (A2) return *reinterpret_cast<const uint16_t *>(p);
    else return p[0] | (p[1] << 8);
}

template <bool A2>
__global__ __launch_bounds__(256) void k_dequant_q8_0(const uint8_t *__restrict__ data,
                                                      uint64_t blocks_avail, uint64_t n,
                                                      float *__restrict__ out, int vec_out) {
    const uint64_t e0 = (uint64_t)blockIdx.x * DQ_WG + 4u * threadIdx.x;
    uint32_t d[DQ_UNITS], q[DQ_UNITS];
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t e = e0 + 1024u * u, b = e / QK8_0;
        d[u] = q[u] = 0u;
        if (b < blocks_avail) {
            const uint8_t *blk = data + b * Q80_BYTES, *p = blk + 2 + e % QK8_0;
            d[u] = dq_u16<A2>(blk);
            q[u] = dq_u16<A2>(p) | (dq_u16<A2>(p + 2) << 16);
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t e = e0 + 1024u * u;
        if (e >= n) break;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (e / QK8_0 < blocks_avail) {
            const float df = ref_half(d[u]);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = __fmul_rn((float)(int8_t)(q[u] >> (8 * i)), df);
        }
        dq_store(out, e, n, v, vec_out);
    }
}

// F32 / F16 / "BF16" branches (src/dflash.rs:333-378, :437-462), with the reference's
// per-element length check.
__device__ __forceinline__ float dq_half(uint32_t h, bool bf16) {
    if (bf16) return ref_half(h);
    // LG_F16: IEEE subnormals, canonical NaN
    const uint32_t e = (h >> 10) & 31u, m = h & 0x3FFu;
    const float sign = (h & 0x8000u) ? -1.0f : 1.0f;
    if (e == 0) return __fmul_rn(__fmul_rn(sign, 6.103515625e-05f), __fdiv_rn((float)m, 1024.0f));
    if (e == 31) return m == 0 ? sign * __builtin_inff() : __uint_as_float(0x7FC00000u);
    return __fmul_rn(__fmul_rn(sign, ldexpf(1.0f, (int)e - 15)), __fadd_rn(1.0f, __fdiv_rn((float)m, 1024.0f)));
}

__global__ __launch_bounds__(256) void k_dequant_elem(const uint8_t *__restrict__ data, uint64_t len,
                                                      int dtype, uint64_t n, float *__restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float r = 0.0f;
    if (dtype == LG_F32) {
        if (i * 4 + 4 <= len)
            r = __uint_as_float(data[4 * i] | (data[4 * i + 1] << 8) | (data[4 * i + 2] << 16) |
                                ((uint32_t)data[4 * i + 3] << 24));
    } else if (i * 2 + 2 <= len) {
        r = dq_half(data[2 * i] | (data[2 * i + 1] << 8), dtype == LG_BF16);
    }
    out[i] = r;
}

// The same over a whole, 16-byte aligned tensor (len covers all n elements), four values a
// load.  F16 codes other than NaNs decode as the hardware conversion does (exact).
__global__ __launch_bounds__(256) void k_dequant_elem4(const uint8_t *__restrict__ data, int dtype, uint64_t n,
                                                       float *__restrict__ out, int vec_out) {
    const uint64_t e0 = (uint64_t)blockIdx.x * DQ_WG + 4u * threadIdx.x;
    uint4 w[DQ_UNITS];
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t e = e0 + 1024u * u;
        if (e + 4 <= n) {
            if (dtype == LG_F32) {
                w[u] = *reinterpret_cast<const uint4 *>(data + 4 * e);
            } else {
                const uint2 h = *reinterpret_cast<const uint2 *>(data + 2 * e);
                w[u] = make_uint4(h.x & 0xFFFFu, h.x >> 16, h.y & 0xFFFFu, h.y >> 16);
            }
        } else {  // the last one to three values
            uint32_t t[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (e + i < n)
                    t[i] = dtype == LG_F32 ? reinterpret_cast<const uint32_t *>(data)[e + i]
                                           : reinterpret_cast<const uint16_t *>(data)[e + i];
            w[u] = make_uint4(t[0], t[1], t[2], t[3]);
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < DQ_UNITS; u++) {
        const uint64_t e = e0 + 1024u * u;
        if (e >= n) break;
        const uint32_t t[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (dtype == LG_F32) v[i] = __uint_as_float(t[i]);
            else if (dtype == LG_BF16) v[i] = ref_half(t[i]);
            else
                v[i] = (t[i] & 0x7FFFu) > 0x7C00u ? __uint_as_float(0x7FC00000u)
                                                  : (float)__builtin_bit_cast(_Float16, (uint16_t)t[i]);
        }
        dq_store(out, e, n, v, vec_out);
    }
}

inline unsigned grid_for(uint64_t threads) { return (unsigned)((threads + 255) / 256); }
inline unsigned dq_grid(uint64_t n) { return (unsigned)((n + DQ_WG - 1) / DQ_WG); }

}  // namespace

extern "C" int lg_dequant_to_f32(const void *data, uint64_t data_len, int dtype, uint64_t n,
                                 float *out, void *stream) {
    clear_error();
    if (n == 0) return LG_OK;
    LG_REQUIRE(out, "lg_dequant_to_f32: null out");
    LG_REQUIRE(data || data_len == 0, "lg_dequant_to_f32: null data with data_len %llu",
               (unsigned long long)data_len);
    LG_REQUIRE(n <= (1ull << 40), "lg_dequant_to_f32: n_elements %llu too large", (unsigned long long)n);
    LG_EXTENT(out, n * 4, "lg_dequant_to_f32 out");
    if (data_len) LG_EXTENT(data, data_len, "lg_dequant_to_f32 data");
    hipStream_t s = (hipStream_t)stream;
    const auto *d = static_cast<const uint8_t *>(data);
    const int vec_out = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    switch (dtype) {
    case LG_Q4_K: {
        const uint64_t need = (n + QK_K - 1) / QK_K, have = data_len / Q4K_BYTES;
        const uint64_t avail = have < need ? have : need;
        if ((reinterpret_cast<uintptr_t>(d) & 15u) == 0)
            hipLaunchKernelGGL(k_dequant_q4k, dim3(dq_grid(n)), dim3(256), 0, s, d, avail, n, out, vec_out);
        else
            hipLaunchKernelGGL(k_dequant_q4k_bytes, dim3(grid_for(n)), dim3(256), 0, s, d, avail, n, out);
        return after_launch("dequant_q4k", s);
    }
    case LG_Q8_0: {
        const uint64_t need = (n + QK8_0 - 1) / QK8_0, have = data_len / Q80_BYTES;
        const uint64_t avail = have < need ? have : need;
        if ((reinterpret_cast<uintptr_t>(d) & 1u) == 0)
            hipLaunchKernelGGL(k_dequant_q8_0<true>, dim3(dq_grid(n)), dim3(256), 0, s, d, avail, n, out, vec_out);
        else
            hipLaunchKernelGGL(k_dequant_q8_0<false>, dim3(dq_grid(n)), dim3(256), 0, s, d, avail, n, out, vec_out);
        return after_launch("dequant_q8_0", s);
    }
    case LG_F32:
    case LG_F16:
    case LG_BF16:
        if ((reinterpret_cast<uintptr_t>(d) & 15u) == 0 && data_len / (dtype == LG_F32 ? 4 : 2) >= n) {
            hipLaunchKernelGGL(k_dequant_elem4, dim3(dq_grid(n)), dim3(256), 0, s, d, dtype, n, out, vec_out);
            return after_launch("dequant_elem", s);
        }
        hipLaunchKernelGGL(k_dequant_elem, dim3(grid_for(n)), dim3(256), 0, s, d, data_len, dtype, n, out);
        return after_launch("dequant_elem", s);
    default:  // src/dflash.rs:463: unsupported types decode to zeros
        LG_HIP_TRY(hipMemsetAsync(out, 0, n * 4, s));
        return after_launch("dequant_zeros", s);
    }
}
