// Device helpers shared by the NSN kernels (gfx950 / CDNA4, wave64).
//
// Arithmetic that must reproduce the reference bit-for-bit (the codec) uses
// only IEEE-exact building blocks: explicit fmaf where torch fuses, unfused
// multiply/add elsewhere (the library is built with -ffp-contract=off),
// correctly rounded division and square root, round-half-even, and RNE
// conversions to fp16/bf16.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "../../include/nsn_hip.h"

namespace nsn {

constexpr int kDim = 128;       // channels per token row (head_dim)
constexpr int kBlockTok = 64;   // tokens per packed block
constexpr float kEps = 1e-12f;  // clamp_min of the norms

__host__ __device__ constexpr int packed_block_bytes(int bits) { return kBlockTok * kDim * bits / 8; }

// ------------------------------------------------------------ conversions

// Materialise an fp32 value in a VGPR.  Without it the backend may fold
// "fp32 multiply, then convert to fp16" into one v_fma_mixlo_f16, which rounds
// the exact product straight to fp16 and skips the fp32 rounding the
// reference performs -- a different result at fp16 ties.
__device__ __forceinline__ float keep_f32(float x) {
    asm volatile("" : "+v"(x));
    return x;
}

__device__ __forceinline__ float f16_bits_to_f32(uint16_t h) {
    return __half2float(__ushort_as_half(h));
}
__device__ __forceinline__ uint16_t f32_to_f16_bits(float f) {
    return __half_as_ushort(__float2half_rn(keep_f32(f)));   // v_cvt_f16_f32, round to nearest even
}
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
    return __uint_as_float(static_cast<uint32_t>(b) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
    return static_cast<uint16_t>((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

template <int DT> struct Elem;
template <> struct Elem<NSN_DTYPE_F16> {
    using T = uint16_t;
    static __device__ __forceinline__ float load(T v) { return f16_bits_to_f32(v); }
    static __device__ __forceinline__ T store(float f) { return f32_to_f16_bits(f); }
};
template <> struct Elem<NSN_DTYPE_BF16> {
    using T = uint16_t;
    static __device__ __forceinline__ float load(T v) { return bf16_bits_to_f32(v); }
    static __device__ __forceinline__ T store(float f) { return f32_to_bf16_bits(f); }
};
template <> struct Elem<NSN_DTYPE_F32> {
    using T = float;
    static __device__ __forceinline__ float load(T v) { return v; }
    static __device__ __forceinline__ T store(float f) { return f; }
};

// ------------------------------------------------------ exact arithmetic

// Correctly rounded fp32 square root: the double square root is correctly
// rounded, and rounding a correctly rounded 53-bit square root to 24 bits is
// again correctly rounded (53 >= 2*24 + 2).
__device__ __forceinline__ float sqrt_rn(float x) {
    return static_cast<float>(__dsqrt_rn(static_cast<double>(x)));
}

// a / b for fp32 a, b given rb = 1.0 / (double)b (correctly rounded double).
// The fp64 product is within 2^-52 (relative) of a/b, while a quotient of two
// 24-bit significands is never closer than 2^-49 (relative) to a rounding
// midpoint of fp32 unless it is exact; so the final rounding to fp32 equals
// IEEE division.  Costs one fp64 multiply per element instead of the ~10
// instruction fp32 division sequence.
__device__ __forceinline__ float div_by_recip(float a, double rb) {
    return static_cast<float>(static_cast<double>(a) * rb);
}

__device__ __forceinline__ double recip_rn(float b) { return __ddiv_rn(1.0, static_cast<double>(b)); }

// torch's clamp_min(1e-12): NaN propagates.
__device__ __forceinline__ float clamp_eps(float n) { return (n > kEps || n != n) ? n : kEps; }

__device__ __forceinline__ bool finite(float x) { return __builtin_isfinite(x); }

// Lane-ordered accumulation of squares that reproduces torch-CPU's
// vector_norm over a contiguous row of 128 fp32 values: lane j (0..7) holds
// fma-chained squares of elements j, j+8, ..., then the lanes are summed in
// order 0..7.
__device__ __forceinline__ float lane8_sum(const float (&acc)[8]) {
    float s = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) s = s + acc[j];
    return s;
}

template <int BITS>
__device__ __forceinline__ void unpack32(const uint32_t (&w)[BITS], uint32_t (&c)[32]) {
    constexpr uint32_t mask = (1u << BITS) - 1u;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int pos = i * BITS, d = pos >> 5, sh = pos & 31;
        uint32_t v = w[d] >> sh;
        if (sh + BITS > 32) v |= w[d + 1] << (32 - sh);
        c[i] = v & mask;
    }
}

// ------------------------------------------------- packed blocks in LDS
//
// The exact restore of a packed block by 256 threads, shared by the restore,
// factor and exact-order attention kernels.  Thread tid unpacks codes 32*tid ..
// (row tid / 4) to bytes in LDS, rows kCodePitch apart: at the rows' own 128
// bytes the 16 rows that a wave sums at once started on one bank, and every
// byte was read by itself.  Both passes now read 2 and 8 codes at a time
// without conflicts (16256 blocks to bf16: 110.5 -> 77.0 us).

constexpr int kCodePitch = kDim + 8;

template <int BITS>
__device__ __forceinline__ void unpack_bytes(const uint32_t (&w)[BITS], uint32_t (&c4)[8]) {
    uint32_t c[32];
    unpack32<BITS>(w, c);
#pragma unroll
    for (int k = 0; k < 8; ++k) c4[k] = c[4 * k] | (c[4 * k + 1] << 8) | (c[4 * k + 2] << 16) | (c[4 * k + 3] << 24);
}
template <int BITS>
__device__ __forceinline__ void unpack_bytes(const uint8_t *block, int tid, uint32_t (&c4)[8]) {
    const uint32_t *src = reinterpret_cast<const uint32_t *>(block) + tid * BITS;
    uint32_t w[BITS];
#pragma unroll
    for (int k = 0; k < BITS; ++k) w[k] = src[k];
    unpack_bytes<BITS>(w, c4);
}
__device__ __forceinline__ void put_codes(uint8_t *codes_s, int tid, const uint32_t (&c4)[8]) {
    uint2 *dst = reinterpret_cast<uint2 *>(codes_s + (tid >> 2) * kCodePitch + 32 * (tid & 3));
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = make_uint2(c4[2 * k], c4[2 * k + 1]);
}

// Norm of row tid / 4 of d = m + s*q (sm: scale, min per channel) in torch's
// 8-lane order, on the row's first thread: its 4 threads sum channels 8k + 2j
// and 8k + 2j + 1.
__device__ __forceinline__ float block_row_norm(const uint8_t *codes_s, const float2 *sm_s) {
    const int tid = threadIdx.x;
    const int jp = (tid & 3) * 2;
    const uint8_t *cr = codes_s + (tid >> 2) * kCodePitch + jp;
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint32_t q = *reinterpret_cast<const uint16_t *>(cr + 8 * k);
        const float4 sm = *reinterpret_cast<const float4 *>(sm_s + 8 * k + jp);
        const float p0 = sm.x * static_cast<float>(q & 0xffu);
        const float p1 = sm.z * static_cast<float>(q >> 8);
        const float d0 = sm.y + p0, d1 = sm.w + p1;
        a0 = __builtin_fmaf(d0, d0, a0);
        a1 = __builtin_fmaf(d1, d1, a1);
    }
    const float b0 = __shfl_down(a0, 1), b1 = __shfl_down(a1, 1);
    const float c0 = __shfl_down(a0, 2), c1 = __shfl_down(a1, 2);
    const float d0 = __shfl_down(a0, 3), d1 = __shfl_down(a1, 3);
    const float acc[8] = {a0, a1, b0, b1, c0, c1, d0, d1};
    return sqrt_rn(lane8_sum(acc));
}
// Scale and min of channels 8*cg .. 8*cg + 7.
__device__ __forceinline__ void load_channels(const float2 *sm_s, int cg, float (&sc)[8], float (&mn)[8]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float4 v = *reinterpret_cast<const float4 *>(sm_s + 8 * cg + 2 * k);
        sc[2 * k] = v.x;
        mn[2 * k] = v.y;
        sc[2 * k + 1] = v.z;
        mn[2 * k + 1] = v.w;
    }
}
// n * (d / |d|) of byte e of c4, nsn_decode's arithmetic (rd = 1 / |d|).
__device__ __forceinline__ float restore_value(uint32_t c4, int e, float s, float m, float n, double rd) {
    const float prod = s * static_cast<float>((c4 >> (8 * e)) & 0xffu);
    const float d = m + prod;
    const float val = n * div_by_recip(d, rd);
    return (n == 0.f) ? 0.f : val;
}

// Two fp32 values to a packed pair of the 16-bit type DT, round to nearest even.
typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
template <int DT>
__device__ __forceinline__ uint32_t pack16(float a, float b) {
    if constexpr (DT == NSN_DTYPE_BF16) {
        const bf16_pair h = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
        return __builtin_bit_cast(uint32_t, h);
    } else {
        return static_cast<uint32_t>(Elem<DT>::store(a)) | (static_cast<uint32_t>(Elem<DT>::store(b)) << 16);
    }
}
// Nonzero iff one of the pair is Inf or NaN: its exponent plus one carries into the sign bit.
template <int DT>
__device__ __forceinline__ uint32_t nonfinite16(uint32_t w) {
    constexpr uint32_t m = DT == NSN_DTYPE_BF16 ? 0x7F807F80u : 0x7C007C00u;
    constexpr uint32_t one = DT == NSN_DTYPE_BF16 ? 0x00800080u : 0x04000400u;
    return ((w & m) + one) & 0x80008000u;
}

// Fast (MFMA) decode attention launcher, defined in nsn_fast.hip.
int launch_attn_fast(const nsn_attn_args *a, hipStream_t st);

// ------------------------------------------------------------ status word

__device__ __forceinline__ void raise_status(int32_t* status, int bits) {
    if (status && bits) atomicOr(status, bits);
}

}  // namespace nsn
