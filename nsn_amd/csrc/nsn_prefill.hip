// Chunked-prefill attention over a packed K/V context (gfx950).
//
// One chunk of n_q queries per (sequence, q-head) attends the sequence's
// context -- packed 64-token blocks, then an fp16/bf16 tail -- and the chunk's
// own dense K/V, causally (chunk query i sees chunk tokens 0..i).  The
// products run in the chunk's dtype: v_mfma_f32_32x32x16_f16 for fp16 data,
// v_mfma_f32_32x32x16_bf16 for bf16 data (no value is squeezed into the
// fp16 range); a tail of the other dtype is converted as it is staged.  The
// reference path materialises the whole K/V (restore of every packed block
// plus the tail, loop_kv_pk01_cache.py:87-106) and runs dense attention on it;
// here the packed blocks are dequantised tile by tile into LDS and never reach
// HBM in dense form.
//
// Workgroup = 8 waves = 256 rows of one (sequence, kv-head), a row being one
// chunk query of one of the group's q-heads; each wave owns 32 rows (one MFMA
// column tile).  Tiles run over head ends: with short chunks a block is
// dequantised for several heads at once (77 queries x 7 heads: 3 tiles a kv-head
// instead of 7).  Per 64-token
// block:
//   1. the raw block (K/V codes, K/V min and scale, K/V decode factors; for
//      a tail or chunk block its dense K/V rows) is staged into LDS by DMA
//      two blocks ahead;
//   2. the 512 threads dequantise it once for the workgroup (threads 0-255
//      K', 256-511 V'^T) into K' [64 tok][128 ch] and V'^T [128 ch][64 tok]
//      (the reconstructed values f_t * (m + s*z), rounded to the compute
//      dtype), double-buffered;
//   3. each wave computes S^T = K' Q^T and O^T += V'^T P^T on MFMA -- the
//      transposed products keep P in registers: the C layout of S^T is
//      already the B layout of P^T for the token order vpos.
// Softmax runs in the log2 domain: fp16 queries are pre-scaled by
// scale*log2(e); bf16 queries enter the product exactly and the scores are
// scaled after it.
//
// What bounds it: per wave and block 32 MFMA (1024 cycles), ~130 VALU of fill
// and ~85 VALU + 32 exp of softmax, on SIMDs that hold two waves each.  While
// one wave's MFMA runs, the other issues VALU at 58 % of its rate and exp at
// its full rate (measured), so a SIMD's block takes at least ~3600 cycles
// with everything overlapped and ~5200 one after the other.  The two waves of
// a SIMD therefore run half a block out of step (see the block loop).  A late
// 512-query chunk of a batch (32 sequences, 16 heads, 7680 tokens of context)
// took 1260 us with 16x16x32 tiles and both waves in step, 1160 us so (in turn
// on one box, 1146-1213 us over boxes, at 1.8 GHz under the full load); one sequence of 32K tokens, 32 query heads, which
// loads a quarter of the CUs at 2.3 GHz, 1206 -> 873 us.
#include <type_traits>

#include "nsn_common.hpp"

namespace nsn {
namespace prefill {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;                // waves per workgroup
constexpr int kQTile = 32 * kWaves;      // chunk queries per workgroup
// LDS banking on gfx950 (measured on the exact patterns): a ds_read_b128 takes
// 16 lanes a cycle over 16 slots of 16 bytes; lanes 0-3, 12-15, 20-27 share a
// cycle, the other 16 of lanes 0-31 the next, lanes 32-63 likewise.
constexpr int kKP = 136;      // K' row pitch (halves): 272 B rows (17 slots), so that the S^T operand
                              // reads (32 rows, one chunk per pass) take 32 different slots
constexpr int kVP = 64;       // V'^T row pitch (halves): 128 B rows, slots kept apart by vchunk
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 8.f;  // running-maximum slack (log2 units): weights < 2^8

// D = A B + C on the compute dtype CT (NSN_DTYPE_F16 or NSN_DTYPE_BF16), 32 x
// 32 x 16.  Lane l (h = l / 32) holds row (column) l % 32 of A (B) at k = 8h ..
// 8h + 7, and rows 8 (i / 4) + 4h + i % 4 of column l % 32 of C in register i.
template <int CT>
__device__ __forceinline__ f32x16 mfma(const u32x4 &a, const u32x4 &b, const f32x16 &c) {
    if constexpr (CT == NSN_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                       0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                      0);
}
// Instruction order of a product loop: N LDS operand reads, each feeding M
// MFMA, with kAhead reads in flight before the first one (measured: 3 874 us,
// 4 881 us, 6 887 us, 8 932 us on the single 32K-token sequence; left to the
// compiler every MFMA waits for its own read).
constexpr int kAhead = 3;
template <int N, int M>
__device__ __forceinline__ void mfma_order() {
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);   // (0x100: LDS reads, 8: MFMA)
#pragma unroll
    for (int i = 0; i < N - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, M, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, M * kAhead, 0);
}
// acc + the sum of a packed pair of the compute dtype.
template <int CT>
__device__ __forceinline__ float add_pair(uint32_t x, float acc) {
    if constexpr (CT == NSN_DTYPE_BF16)
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x), __builtin_bit_cast(bf16x2, 0x3F803F80u), acc,
                                               false);
    else
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, x), __builtin_bit_cast(half2v, 0x3C003C00u), acc, false);
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}
// fp32 pair -> packed pair of the compute dtype (round to nearest even)
template <int CT>
__device__ __forceinline__ uint32_t pk(float a, float b) {
    if constexpr (CT == NSN_DTYPE_BF16) {
        const bf16x2 h = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
        return __builtin_bit_cast(uint32_t, h);
    } else {
        const half2v h = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
        return __builtin_bit_cast(uint32_t, h);
    }
}
// Maxima of scores.  The NaN-propagating maximum is one v_maximum3_f32 with
// no operand quieted first (fmaxf on MFMA results costs a self-maximum per
// operand); a NaN score makes its query's output NaN either way.  Not inline
// asm: the compiler must see that these read MFMA results, which take wait
// states that the hardware does not insert.
__device__ __forceinline__ float max2f(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float max3f(float a, float b, float c) { return max2f(max2f(a, b), c); }
// The two halves of the wave (lanes l and l ^ 32) combined, on every lane,
// without LDS: v_permlane32_swap gives (lo, lo) and (hi, hi).
__device__ __forceinline__ float halves_max(float x) {
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return max2f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// fp32 pair -> bf16 hi (round to nearest even) + bf16 lo = rn(x - hi): the
// pair to ~2^-17 relative.
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t &hi, uint32_t &lo) {
    hi = pk<NSN_DTYPE_BF16>(a, b);
    lo = pk<NSN_DTYPE_BF16>(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u));
}
__device__ __forceinline__ float h16(uint32_t w, int hi) {
    return static_cast<float>(__builtin_bit_cast(half2v, w)[hi]);
}

// Channel order inside each group of 8 (the K' columns and the Q
// fragments share it): element p holds channel chE[p], whose 3-bit code the
// unpack leaves at bit kE[p] of an fp16 half (a subnormal z * 2^(kE-24)).
template <int BITS> struct Order;
template <> struct Order<3> {
    static constexpr int chE[8] = {0, 3, 1, 4, 2, 5, 6, 7};
    static constexpr int kE[8] = {0, 1, 3, 4, 6, 7, 2, 5};
};
template <> struct Order<5> {
    static constexpr int chE[8] = {0, 1, 2, 3, 4, 5, 6, 7};
    static constexpr int kE[8] = {0, 0, 0, 0, 0, 0, 0, 0};
};

// The 8 codes of one token's 8-channel group: bytes BITS*cg .. of its row, in
// the row's dwords w0 = (BITS*cg)/4 and w1 (the next), from bit sh = 8 *
// ((BITS*cg) % 4) of w0 -> 4 dwords, element p (dword p/2, half p%2) = code of
// channel chE[p] at bit kE[p].
template <int BITS>
__device__ __forceinline__ void codes8(uint32_t w0, uint32_t w1, uint32_t sh, uint32_t (&B)[4]) {
    const uint32_t x = __builtin_amdgcn_alignbit(w1, w0, sh);
    if constexpr (BITS == 3) {
        const uint32_t P = perm(x, x, 0x02010100u), Q = perm(x, x, 0x0C020C02u);
        B[0] = P & 0x000E0007u;
        B[1] = P & 0x00700038u;
        B[2] = P & 0x038001C0u;
        B[3] = Q & 0x00E0001Cu;
    } else {
        const uint32_t y = w1 >> sh;   // code bits 32..39
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t z[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = 2 * i + h;
                z[h] = (e < 6) ? __builtin_amdgcn_ubfe(x, 5 * e, 5)
                     : (e == 6) ? (__builtin_amdgcn_alignbit(y, x, 30) & 31u)
                                : ((y >> 3) & 31u);
            }
            B[i] = z[0] | (z[1] << 16);
        }
    }
}

struct Side {
    const uint8_t *codes;
    const uint16_t *mins, *scales;
    const float *factors;
    const int32_t *blocks;
    int64_t block_cap;
    const uint16_t *tail;   // TDT
    int64_t tail_cap;
};

struct PrefillParams {
    const uint16_t *q;     // [B, Hq, n_q, 128] DT
    int64_t batch, heads_q, heads_kv, n_q;
    int group;
    int run_heads;         // q-heads whose rows a run of tiles covers: the group (tiles over head ends) or 1
    float qscale;          // scale * log2(e)
    const int32_t *ctx_len;
    Side k, v;
    const uint16_t *kc, *vc;   // chunk K/V [B, Hkv, n_q, 128] DT
    uint16_t *out;             // [B, Hq, n_q, 128] DT
    int32_t *status;
    uint16_t *ka, *va;         // append: the K / V tails written (TDT), else null
    int splits;                // workgroups that share a tile's blocks (context splits)
    float *part;               // splits > 1: their partials, see Parts
};

// Context splits.  A grid of few tiles (one long sequence, a short chunk)
// leaves most CUs idle, so a tile's blocks are then shared by up to kMaxSplits
// workgroups and a second kernel merges their softmax states.  A split takes
// at least kSplitBlocks blocks; the workgroups past nblk / kSplitBlocks leave
// at once, and a tile with one split left writes its output itself.
// Workspace: per (tile, split) 256 pairs (running maximum, weight sum), then
// per (tile, split) the unnormalised O^T in register order, [8 waves][16][64
// lanes] float4.  A weight sum of kDone marks a slot without partials: every
// slot of a tile whose output is written, and the splits that left at once.
// (The maximum cannot mark them: it is also -inf where all of a split's scores
// are NaN, or its tokens masked, and its NaN must reach the output.)
constexpr int kMaxSplits = 16, kSplitBlocks = 8;
constexpr float kDone = -1.f;
struct Parts {
    float2 *ml;
    float4 *acc;
    __device__ Parts(float *part, int64_t tiles, int splits, int64_t tile, int split) {
        const int64_t slot = tile * splits + split;
        ml = reinterpret_cast<float2 *>(part) + slot * kQTile;
        acc = reinterpret_cast<float4 *>(part + 2 * tiles * splits * kQTile) + slot * (kQTile * kDim / 4);
    }
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from global memory straight into LDS at M0 + 16*lane,
// with the non-temporal hint: a workgroup streams each block of its context
// once (C4 last chunk 1241-1242 -> 1222-1228 us).  The s_nop is the wait state
// that a load to LDS needs after a scalar write of M0.
__device__ __forceinline__ void dma16(const void *src, void *dst) {
    const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst));
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(src), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// Staged block layout (bytes): [K codes NB | V codes NB | K min 256 | K scale 256 |
// V min 256 | V scale 256 | K factor 256 | V factor 256 | (512 not read)].  K code rows are in
// token order.  The 16-byte chunk x of V code row t sits at chunk 64x + 16 (t % 4) +
// t / 4 of its part: the V'^T fill's lanes read rows 4 apart, which in row
// order fall on two banks.
template <int BITS> struct Stage {
    static constexpr int NB = packed_block_bytes(BITS);
    static constexpr int META = 2 * NB;
    static constexpr int BYTES = 2 * NB + 2048;
    static constexpr int NI = 2 * NB / 1024 + 2;   // 1 KiB DMA instructions per block
    static constexpr int PER_WAVE = (NI + kWaves - 1) / kWaves;
};

// One wave's share of the DMA of a packed block: instruction i = wave + 8n of
// the block.  A lane's source moves by a fixed step per block, so a block's
// request is one 64-bit multiply-add per instruction.
struct PackedDma {
    const uint8_t *src;   // the lane's 16 bytes of block 0 of the stream
    uint32_t step;        // bytes between two blocks
    uint32_t dst;         // offset in the stage
};
template <int BITS>
__device__ __forceinline__ PackedDma packed_dma(const PrefillParams &p, int64_t rk, int64_t rv, int i, int l) {
    using S = Stage<BITS>;
    constexpr int NK = S::NB / 1024;
    const int q = l & 15;
    if (i < NK) return {p.k.codes + rk * S::NB + 1024 * i + 16 * l, S::NB, 1024u * i};
    if (i < 2 * NK) {
        const int x = i - NK, t = 4 * q + (l >> 4);
        return {p.v.codes + rv * S::NB + (S::NB / kBlockTok) * t + 16 * x, S::NB, 1024u * i};
    }
    if (i == 2 * NK) {
        const uint16_t *m = (l < 16) ? p.k.mins + rk * kDim : (l < 32) ? p.k.scales + rk * kDim
                          : (l < 48) ? p.v.mins + rv * kDim : p.v.scales + rv * kDim;
        return {reinterpret_cast<const uint8_t *>(m + 8 * q), 2 * kDim, S::META};
    }
    const float *f = (l & 16) ? p.v.factors + rv * kBlockTok : p.k.factors + rk * kBlockTok;   // (lanes 32-63: again)
    return {reinterpret_cast<const uint8_t *>(f + 4 * q), 4 * kBlockTok, S::META + 1024};
}

// A dense block (tail or chunk tokens, 2-byte elements) is staged by DMA
// like a packed one: K rows then V rows, 256 B each.  The 16-byte chunk c of
// row t sits at chunk position c ^ ((t >> 2) & 15) of the row, so that the
// 16 lanes of either fill role's reads (one row, 16 chunks; or 16 rows 4
// apart, one chunk) fall on 16 different bank groups.
constexpr int kDenseStage = 2 * kBlockTok * kDim * 2;   // 32 KiB
__device__ __forceinline__ int dswz(int t, int c) { return c ^ ((t >> 2) & 15); }

// DMA of the first `valid` rows of a dense block (K rows from xk, V rows
// from xv, 128-element row pitch) into a stage: instruction i writes rows
// 4*(i%16) .. +3 of side i/16 and is issued by wave i % kWaves; lane l
// writes chunk position l%16 of row l/16 and so reads chunk dswz(row, l%16).
// Rows past `valid` are neither read nor written.
__device__ __forceinline__ void stage_dense(const uint16_t *xk, const uint16_t *xv, int valid, int wave, int l,
                                            uint8_t *st) {
    const int r = l >> 4, cp = l & 15;
    for (int i = wave; i < 32; i += kWaves) {
        if (4 * (i & 15) >= valid) continue;   // (wave-uniform)
        const int t = 4 * (i & 15) + r;
        if (t < valid) dma16(((i < 16) ? xk : xv) + t * kDim + 8 * dswz(t, cp), st + 1024 * i);
    }
}

// V'^T keeps each channel's 64 tokens in the k order of the PV product:
// token t = 16c + 8a + 4h + i sits at position 16c + 8h + 4a + i, so the 8
// tokens that half h of the wave contracts in 16-token step c (the rows of
// S^T that its registers hold) are one 16-byte read.  Groups of 4 stay together.
__device__ __forceinline__ int vpos(int t) { return (t & 51) | ((t & 4) << 1) | ((t & 8) >> 1); }

// V'^T row `r` keeps its 16-byte chunk c at position c ^ ((r >> 1) & 7).  Rows
// are 128 B, half a pass of the banks: of the rows that one pass of a PV
// operand read takes (0-3, 12-15, 20-27 or the other 16 of 32), the eight of
// each parity get eight different slots (the measured cycles of the exact
// pattern equal a linear read's; r >> 2 is 2-way).  A fill write pass (16
// token groups of one row) writes a whole row.
__device__ __forceinline__ int vchunk(int r, int c) { return c ^ ((r >> 1) & 7); }
__device__ __forceinline__ int vcol_at(int r, int t) { return 8 * vchunk(r, vpos(t) >> 3) + (vpos(t) & 7); }

// The block buffer compute reads: K' [64 tok][kKP], V'^T [128 ch][kVP].
// A fill thread's place in it: K' rows 4*rg .. +3 from kt (channels 8*cg ..);
// V'^T rows 8*cg + c (c = 0 .. 7), tokens 4*rg .. +3, at vt + vx[c / 2] + c * kVP
// (the chunk XOR of row 8*cg + c is that of row 8*cg with c / 2 on top).
struct KV {
    uint16_t *kt, *vt;
    uint32_t vx[4];
};
__device__ __forceinline__ void store_vcol(const KV &kv, int c, const uint32_t (&w)[2]) {
    *reinterpret_cast<u32x2 *>(kv.vt + kv.vx[c >> 1] + c * kVP) = u32x2{w[0], w[1]};
}

// Fill one side of a KV buffer from a staged dense block of dtype DT
// (`valid` rows; rows past it are zero), rounded to CT.  Thread: tokens
// 4*rg .. 4*rg+3, channels 8*cg .. 8*cg+7; side 0 writes K' rows, side 1
// V'^T columns.  `app` (nullable): the block's rows also go to app + t*128,
// rounded to ADT (the chunk's append to the tail).
template <int BITS, int DT, int CT, int side, int ADT>
__device__ __forceinline__ void fill_dense(const uint8_t *st, int valid, int rg, int cg, const KV &kv,
                                           uint16_t *app) {
    using O = Order<BITS>;
    uint32_t vcol[8][2];   // V'^T: per channel, tokens 4rg..4rg+3 as 2 fp16 pairs
    float vprev[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = 4 * rg + i;
        float f[8];
        if (t < valid) {
            const uint4 a = *reinterpret_cast<const uint4 *>(st + kDenseStage / 2 * side + 256 * t + 16 * dswz(t, cg));
            const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = Elem<DT>::load(static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1))));
            if (app) {
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = static_cast<uint32_t>(Elem<ADT>::store(f[2 * e])) |
                           (static_cast<uint32_t>(Elem<ADT>::store(f[2 * e + 1])) << 16);
                *reinterpret_cast<uint4 *>(app + t * kDim + 8 * cg) = uint4{o[0], o[1], o[2], o[3]};
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = 0.f;
        }
        if constexpr (side == 0) {
            *reinterpret_cast<uint4 *>(kv.kt + t * kKP + 8 * cg) =
                uint4{pk<CT>(f[O::chE[0]], f[O::chE[1]]), pk<CT>(f[O::chE[2]], f[O::chE[3]]),
                      pk<CT>(f[O::chE[4]], f[O::chE[5]]), pk<CT>(f[O::chE[6]], f[O::chE[7]])};
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (i & 1) vcol[e][i >> 1] = pk<CT>(vprev[e], f[e]);
                else vprev[e] = f[e];
            }
        }
    }
    if constexpr (side == 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            store_vcol(kv, e, vcol[e]);
    }
}

// Fill one side of a KV buffer from a staged packed block: direction m + s*z
// per element (one fma with the code as an exact fp16 subnormal, scaled back
// by 2^(24-k)) times the token's decode factor -- the reconstructed value
// itself (|x| <= its fp16 norm, so within fp16 range by construction),
// rounded to CT.
template <int BITS, int CT, int side>
__device__ __forceinline__ void fill_packed(const uint8_t *st, int rg, int cg, const KV &kv) {
    using S = Stage<BITS>;
    using O = Order<BITS>;
    constexpr int ROWB = BITS * 16;   // code bytes per token row
    const uint4 m4 = *reinterpret_cast<const uint4 *>(st + S::META + 512 * side + 16 * cg);
    const uint4 s4 = *reinterpret_cast<const uint4 *>(st + S::META + 512 * side + 256 + 16 * cg);
    const float4 f4 = *reinterpret_cast<const float4 *>(st + S::META + 1024 + 256 * side + 16 * rg);
    const float fac[4] = {f4.x, f4.y, f4.z, f4.w};
    const uint32_t M[4] = {m4.x, m4.y, m4.z, m4.w}, SC[4] = {s4.x, s4.y, s4.z, s4.w};
    float mE[8], sE[8];   // per element p (channel chE[p])
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int c = O::chE[p];
        mE[p] = h16(M[c >> 1], c & 1);
        sE[p] = __builtin_fmaf(h16(SC[c >> 1], c & 1), static_cast<float>(1u << (24 - O::kE[p])), 0.f);   // (one fma_mix)
    }
    const int byte = BITS * cg, d0 = byte >> 2;
    const uint32_t sh = 8u * static_cast<uint32_t>(byte & 3);
    // token 4*rg + i's dwords d0 and d0 + 1 (past the last group's row: the
    // next row or part, whose bits are shifted out)
    auto vdw = [&](int d) { return S::NB + 1024 * (d >> 2) + 16 * rg + 4 * (d & 3); };
    const uint8_t *c0 = st + (side ? vdw(d0) : ROWB * 4 * rg + 4 * d0);
    const uint8_t *c1 = st + (side ? vdw(d0 + 1) : ROWB * 4 * rg + 4 * d0 + 4);
    constexpr int PITCH = side ? 256 : ROWB;
    uint32_t vcol[8][2];
    float vprev[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = 4 * rg + i;
        uint32_t b[4];
        codes8<BITS>(*reinterpret_cast<const uint32_t *>(c0 + PITCH * i), *reinterpret_cast<const uint32_t *>(c1 + PITCH * i),
                     sh, b);
        float d[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) d[p] = __builtin_fmaf(h16(b[p >> 1], p & 1), sE[p], mE[p]) * fac[i];
        if constexpr (side == 0) {
            *reinterpret_cast<uint4 *>(kv.kt + t * kKP + 8 * cg) =
                uint4{pk<CT>(d[0], d[1]), pk<CT>(d[2], d[3]), pk<CT>(d[4], d[5]), pk<CT>(d[6], d[7])};
        } else {
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                if (i & 1) vcol[p][i >> 1] = pk<CT>(vprev[p], d[p]);
                else vprev[p] = d[p];
            }
        }
    }
    if constexpr (side == 1) {
#pragma unroll
        for (int p = 0; p < 8; ++p)
            store_vcol(kv, O::chE[p], vcol[p]);
    }
}

// DT: dtype of the queries, the chunk K/V, the output and the products; TDT:
// dtype of the context tail.  LO (bf16 only): the softmax weights enter the
// PV product and the row sums as bf16 hi + lo (~2^-17 relative) instead of
// one bf16 rounding (2^-9) -- for chunks with little or no context, whose
// first queries attend a handful of tokens, where one weight's bf16 rounding
// moves the output by up to 2^-9 of |v|.  It costs 16 more MFMA and the split
// of 32 weights per wave and block (a late chunk 1160 -> 1640 us, the first
// chunk 119 -> 138 us), so the caller asks for it.
template <int BITS, int DT, int TDT, bool LO>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void prefill_kernel(PrefillParams p) {
    using S = Stage<BITS>;
    using O = Order<BITS>;
    constexpr bool QPRE = DT == NSN_DTYPE_F16;   // fp16 queries carry scale*log2(e); bf16 ones stay exact
    static_assert(!LO || DT == NSN_DTYPE_BF16, "hi + lo weights are a bf16 form");
    __shared__ __align__(16) uint16_t kt[2][kBlockTok * kKP];
    __shared__ __align__(16) uint16_t vt[2][kDim * kVP];
    __shared__ __align__(16) uint8_t stg[2][S::BYTES > kDenseStage ? S::BYTES : kDenseStage];

    const int tid = threadIdx.x, l = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // (uniform: the DMA targets are scalar)
    const int col = l & 31, h = l >> 5;
    // fill role: threads 0..255 fill K' (lanes over channel groups: each pass
    // writes whole K' rows), 256..511 V'^T (lanes over token groups: each pass
    // writes one contiguous V'^T row)
    const int side = __builtin_amdgcn_readfirstlane(tid >> 8);   // (wave-uniform)
    const int rg = side ? (tid & 15) : ((tid >> 4) & 15);
    const int cg = side ? ((tid >> 4) & 15) : (tid & 15);
    // The rows of a kv-head are its group's queries, (q-head, query) in memory
    // order; a tile is 256 of them, whatever heads they belong to (or, a run of
    // tiles per q-head, 256 of one head's: grid z).  Grid (tile, split, sequence,
    // kv-head), tiles slowest and in reverse: the last tile holds the latest
    // queries, which see the most causal chunk blocks.
    const int nq = static_cast<int>(p.n_q);              // (< 2^24, checked by the host)
    const int nrows = p.run_heads * nq;                  // (rows of 256 bytes: fewer than 2^31 fit the memory)
    const uint32_t hkv = static_cast<uint32_t>(p.heads_kv);
    const uint32_t per_tile = gridDim.y > 1 ? hkv : static_cast<uint32_t>(p.batch) * hkv;   // (y: sequences, in a huge grid)
    const uint32_t zs = blockIdx.x / per_tile, rem = blockIdx.x - zs * per_tile;
    const uint32_t z = zs / static_cast<uint32_t>(p.splits);
    const int split = static_cast<int>(zs - z * static_cast<uint32_t>(p.splits));
    const int b = static_cast<int>(rem / hkv + blockIdx.y);
    const int kvh = static_cast<int>(rem % hkv);
    const int tiles = (nrows + kQTile - 1) / kQTile;
    const int q0 = (tiles - 1 - static_cast<int>(z)) * kQTile;
    const int rw = q0 + 32 * wave;                       // this wave's first row
    const int r = rw + col;                              // this lane's row,
    const int qi = r % nq;                               // and its query
    const int64_t seqrow = static_cast<int64_t>(b) * p.heads_kv + kvh;
    const int64_t row0 = (seqrow * p.group + blockIdx.z) * p.n_q;   // row 0 of the run in q and out

    // ---- Q fragments (B operand of S^T = K' Q^T): row rw + l % 32, channels
    // 16*ks + 8*h + chE[e] (fp16: times scale*log2(e)).  All eight loads go out
    // at once, before the context lengths are needed, from the last row where
    // the lane's is past it (behind a test each, they were eight round trips a
    // workgroup: the ragged 77-query chunks 45.6 -> 44.6 us).
    u32x4 qf[8];
    const uint16_t *qrow = p.q + (row0 + (r < nrows ? r : nrows - 1)) * kDim + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const u32x4 *>(qrow + 16 * ks);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            x[e] = Elem<DT>::load(static_cast<uint16_t>(qf[ks][e >> 1] >> (16 * (e & 1))));
            if (QPRE) x[e] *= p.qscale;
        }
        qf[ks] = u32x4{pk<DT>(x[O::chE[0]], x[O::chE[1]]), pk<DT>(x[O::chE[2]], x[O::chE[3]]),
                       pk<DT>(x[O::chE[4]], x[O::chE[5]]), pk<DT>(x[O::chE[6]], x[O::chE[7]])};
    }

    auto parts = [&]() {
        return Parts(p.part, static_cast<int64_t>(tiles) * p.batch * p.heads_kv, p.splits,
                     (static_cast<int64_t>(q0 / kQTile) * p.batch + b) * p.heads_kv + kvh, split);
    };
    const int64_t T = p.ctx_len[b];
    const int64_t nbk = p.k.blocks ? p.k.blocks[b] : 0;
    const int64_t nbv = p.v.blocks ? p.v.blocks[b] : 0;
    if (nbk != nbv || nbk < 0 || (nbk > 0 && (nbk > p.k.block_cap || nbk > p.v.block_cap)) || T - nbk * kBlockTok < 0 ||
        T - nbk * kBlockTok > p.k.tail_cap || T - nbk * kBlockTok > p.v.tail_cap) {
        if (tid == 0) raise_status(p.status, NSN_ST_CAPACITY);   // inconsistent cache (host checks first)
        if (p.splits > 1 && tid < kQTile) parts().ml[tid] = float2{-INFINITY, kDone};
        return;
    }
    const int nb = static_cast<int>(nbk), ntail = static_cast<int>(T - nbk * kBlockTok);
    // chunk tokens this workgroup sees: up to its last row's query, all of
    // them where its rows run over the end of a head
    const int rl = (q0 + kQTile < nrows ? q0 + kQTile : nrows) - 1;
    const int qend = (rl / nq == q0 / nq) ? rl % nq + 1 : nq;
    const int nt_blk = static_cast<int>((static_cast<int64_t>(ntail) + kBlockTok - 1) / kBlockTok);
    const int nblk = nb + nt_blk + (qend + kBlockTok - 1) / kBlockTok;
    // this workgroup's blocks [j0, j1)
    int splits = nblk / kSplitBlocks;
    splits = splits < 1 ? 1 : (splits < p.splits ? splits : p.splits);
    if (split >= splits) {
        if (tid < kQTile) parts().ml[tid] = float2{-INFINITY, kDone};
        return;
    }
    const int j0 = static_cast<int>(static_cast<int64_t>(nblk) * split / splits);
    const int j1 = static_cast<int>(static_cast<int64_t>(nblk) * (split + 1) / splits);
    // append: the workgroups of a kv-head's last tile (they stage every chunk
    // block) write the chunk's K/V to tail rows ntail .. ntail + n_q - 1 as
    // they fill them; no room: flag, no append
    const bool app_wg = p.ka && z == 0 && blockIdx.z == 0;
    const bool app_ok = app_wg && ntail + p.n_q <= p.k.tail_cap && ntail + p.n_q <= p.v.tail_cap;
    if (app_wg && !app_ok && tid == 0) raise_status(p.status, NSN_ST_CAPACITY);

    f32x16 acc[4];   // O^T tiles: channels 32*ct + 8*(i/4) + 4*h + i%4 of query qi
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[ct][i] = 0.f;
    float m_run = -INFINITY;
    float lsum = 0.f;   // sum of the rounded weights of this lane's tokens (half of the query's)
    bool bad = false;
    const bool live = rw < nrows;   // (a wave past the last row only helps stage and fill)

    // Block j: packed (j < nb), tail (nb <= j < nb + nt_blk), or chunk; its rows
    // in use and (chunk blocks) the chunk position of its first token.
    auto block_rows = [&](int j, int &valid, int &cpos) __attribute__((always_inline)) {
        cpos = -1;
        if (j < nb) {
            valid = kBlockTok;
        } else if (j < nb + nt_blk) {
            const int t0 = (j - nb) * kBlockTok;
            valid = (ntail - t0 < kBlockTok) ? ntail - t0 : kBlockTok;
        } else {
            cpos = (j - nb - nt_blk) * kBlockTok;
            valid = (qend - cpos < kBlockTok) ? qend - cpos : kBlockTok;
        }
    };
    uint32_t vx[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) vx[x] = 8 * cg * kVP + vcol_at(8 * cg + 2 * x, 4 * rg);
    // Fill side SIDE of block j (K' or V'^T) into buffer j & 1 from its raw stage j & 1.
    auto fill = [&](auto side_c, auto packed_c, int j) __attribute__((always_inline)) {
        constexpr int SIDE = decltype(side_c)::value;
        constexpr bool PACKED = decltype(packed_c)::value;
        const KV kv{kt[j & 1], vt[j & 1], {vx[0], vx[1], vx[2], vx[3]}};
        if (PACKED || j < nb) {
            fill_packed<BITS, DT, SIDE>(stg[j & 1], rg, cg, kv);
            if (!PACKED) asm volatile("; packed block filled");   // (keeps the two paths' stores apart: merged, they cost address moves)
        } else {
            int valid;
            int cpos;
            block_rows(j, valid, cpos);
            if (cpos < 0) {
                fill_dense<BITS, TDT, DT, SIDE, TDT>(stg[j & 1], valid, rg, cg, kv, nullptr);
            } else {
                uint16_t *app = nullptr;
                if (app_ok)
                    app = SIDE ? p.va + (seqrow * p.v.tail_cap + ntail + cpos) * kDim
                               : p.ka + (seqrow * p.k.tail_cap + ntail + cpos) * kDim;
                fill_dense<BITS, DT, DT, SIDE, TDT>(stg[j & 1], valid, rg, cg, kv, app);
            }
        }
    };
    PackedDma pdma[S::PER_WAVE];
#pragma unroll
    for (int n = 0; n < S::PER_WAVE; ++n)
        pdma[n] = packed_dma<BITS>(p, seqrow * p.k.block_cap, seqrow * p.v.block_cap, wave + kWaves * n, l);
    // Stage the raw data of block j into stage j & 1: packed codes and
    // metadata, or the valid rows of its tail / chunk tokens.
    auto stage = [&](auto packed_c, int j) __attribute__((always_inline)) {
        if (decltype(packed_c)::value || j < nb) {
#pragma unroll
            for (int n = 0; n < S::PER_WAVE; ++n)
                if (wave + kWaves * n < S::NI)
                    dma16(pdma[n].src + static_cast<uint64_t>(static_cast<uint32_t>(j)) * pdma[n].step,
                          stg[j & 1] + pdma[n].dst);
        } else {
            int valid;
            int cpos;
            block_rows(j, valid, cpos);
            if (cpos < 0) {
                const int64_t t0 = (j - nb) * kBlockTok;
                stage_dense(p.k.tail + (seqrow * p.k.tail_cap + t0) * kDim,
                            p.v.tail + (seqrow * p.v.tail_cap + t0) * kDim, valid, wave, l, stg[j & 1]);
            } else {
                stage_dense(p.kc + (seqrow * p.n_q + cpos) * kDim, p.vc + (seqrow * p.n_q + cpos) * kDim, valid,
                            wave, l, stg[j & 1]);
            }
        }
    };

    // ---- S^T[token][query] = K' Q^T: register i of s[tt] holds token
    // 32*tt + 8*(i/4) + 4*h + i%4
    f32x16 s[2];
    auto scores = [&](int j) __attribute__((always_inline)) {
        const uint16_t *ktj = kt[j & 1] + col * kKP + 8 * h;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 16; ++i) s[tt][i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const u32x4 a = *reinterpret_cast<const u32x4 *>(ktj + 32 * tt * kKP + 16 * ks);
                s[tt] = mfma<DT>(a, qf[ks], s[tt]);
            }
        mfma_order<16, 1>();
    };
    // ---- online softmax of the lane's query.  The running maximum (and the
    // state's rescale) only moves when some lane's block maximum passes it by
    // more than kLazy (log2 units): weights then stay below 2^kLazy, which
    // every weight form holds exactly as well as weights below 1.
    u32x4 pb[4];              // P''^T B operands of the 16-token steps (LO: the bf16 hi parts)
    u32x4 pl[LO ? 4 : 1];     // LO: the bf16 lo parts
    auto softmax = [&](auto packed_c, int j) __attribute__((always_inline)) {
        int valid = kBlockTok;
        int cpos = -1;
        if (!decltype(packed_c)::value) block_rows(j, valid, cpos);
        if (valid < kBlockTok || cpos >= 0) {   // (uniform) partial or causal block
            // allowed tokens of this block: tok < valid and (chunk blocks) tok <= query - cpos
            const int rel = (cpos >= 0) ? qi - cpos : kBlockTok;
            const int lim = (rel < valid - 1) ? rel : valid - 1;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (32 * tt + 8 * (i >> 2) + 4 * h + (i & 3) > lim) s[tt][i] = -INFINITY;
        }
        float mx = max2f(s[0][15], s[1][15]);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const float a0 = max3f(s[tt][0], s[tt][1], s[tt][2]), a1 = max3f(s[tt][3], s[tt][4], s[tt][5]);
            const float a2 = max3f(s[tt][6], s[tt][7], s[tt][8]), a3 = max3f(s[tt][9], s[tt][10], s[tt][11]);
            const float a4 = max3f(s[tt][12], s[tt][13], s[tt][14]);
            mx = max3f(mx, max3f(a0, a1, a2), max2f(a3, a4));
        }
        mx = halves_max(mx);
        if (!QPRE) mx *= p.qscale;   // (bf16: the scores scale inside the exponent below)
        if (__builtin_amdgcn_ballot_w64(mx > m_run + kLazy)) {
            const float mnew = fmaxf(m_run, mx);
            const float alpha = (m_run == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_run - mnew);
            lsum *= alpha;
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) acc[ct] *= alpha;
            m_run = mnew;
        }
        const float msafe = (m_run == -INFINITY) ? 0.f : m_run;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float w[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const float v = s[c >> 1][8 * (c & 1) + 2 * e + x];
                    w[x] = __builtin_amdgcn_exp2f(QPRE ? v - msafe : __builtin_fmaf(v, p.qscale, -msafe));
                }
                if constexpr (LO) split_bf16(w[0], w[1], hi[e], lo[e]);
                else hi[e] = pk<DT>(w[0], w[1]);
                // the row sum takes the rounded weights that the PV product uses
                lsum = add_pair<DT>(hi[e], lsum);
                if constexpr (LO) lsum = add_pair<DT>(lo[e], lsum);
            }
            pb[c] = u32x4{hi[0], hi[1], hi[2], hi[3]};
            if constexpr (LO) pl[c] = u32x4{lo[0], lo[1], lo[2], lo[3]};
        }
    };
    // ---- O^T[channel][query] += V'^T P''^T over the block's four 16-token steps
    auto output = [&](int j) __attribute__((always_inline)) {
        const uint16_t *vtj = vt[j & 1] + col * kVP;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {   // (row 32*ct + col: the same XOR for every ct)
                const u32x4 a = *reinterpret_cast<const u32x4 *>(vtj + 32 * ct * kVP + 8 * vchunk(col, 2 * c + h));
                acc[ct] = mfma<DT>(a, pb[c], acc[ct]);
                if constexpr (LO) acc[ct] = mfma<DT>(a, pl[c], acc[ct]);
            }
        mfma_order<16, LO ? 2 : 1>();
    };
    auto barrier = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    using F_ = std::false_type;
    using T_ = std::true_type;
    using K_ = std::integral_constant<int, 0>;
    using V_ = std::integral_constant<int, 1>;

    // ---- prologue: the first two raw blocks staged together (one round trip), K' of the first filled
    stage(F_{}, j0);
    if (j0 + 1 < j1) stage(F_{}, j0 + 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (side == 0) fill(K_{}, F_{}, j0);
    barrier();

    // ---- The two waves of a SIMD (w and w + 4) run half a block out of step,
    // so that one's MFMA work meets the other's VALU work.  Per block j:
    //   first half    waves 0-3: S^T(j), softmax(j)    waves 4-7: fill V'^T(j), O^T(j-1)
    //   second half   waves 0-3: fill K'(j+1), O^T(j)  waves 4-7: S^T(j), softmax(j)
    // K'(j+1) goes into the buffer whose last readers (S^T(j-1)) are a half
    // block back, V'^T(j) into the one that O^T(j-2) left; raw block j + 2 is
    // requested when V'^T(j) has been read and waited for before K'(j+2).
    // Priorities: a fill goes before the other wave's softmax (and its own
    // products come right behind it), so that the products overlap the rest of
    // that softmax; without priorities the older waves win every conflict and
    // the late chunk takes 6 % longer.  The packed stretch (blocks
    // j .. j + 2 packed) has a loop of its own: its body has no branch on the
    // block kind.
    auto attend = [&](auto packed_c, int j) __attribute__((always_inline)) {
        if (!live) return;
        __builtin_amdgcn_s_setprio(2);
        scores(j);
        __builtin_amdgcn_s_setprio(0);
        softmax(packed_c, j);
    };
    auto step_k = [&](auto packed_c, int j) __attribute__((always_inline)) {
        constexpr bool PACKED = decltype(packed_c)::value;
        attend(packed_c, j);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // raw block j + 1
        barrier();
        if (PACKED || j + 2 < j1) stage(packed_c, j + 2);
        __builtin_amdgcn_s_setprio(3);
        if (PACKED || j + 1 < j1) fill(K_{}, packed_c, j + 1);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(3);
        if (live) output(j);
        barrier();
    };
    auto step_v = [&](auto packed_c, int j) __attribute__((always_inline)) {
        constexpr bool PACKED = decltype(packed_c)::value;
        __builtin_amdgcn_s_setprio(3);
        fill(V_{}, packed_c, j);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(3);
        if (live && j > j0) output(j - 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        barrier();
        if (PACKED || j + 2 < j1) stage(packed_c, j + 2);
        attend(packed_c, j);
        barrier();
    };
    const int jp = nb < j1 ? nb : j1;
    int j = j0;
    if (side == 0) {
        for (; j + 2 < jp; ++j) step_k(T_{}, j);
        for (; j < j1; ++j) step_k(F_{}, j);
    } else {
        for (; j + 2 < jp; ++j) step_v(T_{}, j);
        for (; j < j1; ++j) step_v(F_{}, j);
        if (live) output(j1 - 1);
    }

    // ---- output: O[q][c] = O^T / l
    const float lt = halves_sum(lsum);
    if (splits > 1) {   // the split's state instead
        const Parts pt = parts();
        if (h == 0) pt.ml[32 * wave + col] = float2{m_run, lt};
        if (!live) return;
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                pt.acc[(wave * 16 + 4 * ct + c) * 64 + l] =
                    float4{acc[ct][4 * c], acc[ct][4 * c + 1], acc[ct][4 * c + 2], acc[ct][4 * c + 3]};
        return;
    }
    if (p.splits > 1 && tid < kQTile) parts().ml[tid] = float2{-INFINITY, kDone};
    if (r < nrows) {
        const float rl = 1.f / lt;
        uint16_t *dst = p.out + (row0 + r) * kDim + 4 * h;
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[i] = acc[ct][4 * c + i] * rl;
                    bad |= !finite(o[i]);
                }
                const uint32_t w0 = static_cast<uint32_t>(Elem<DT>::store(o[0])) | (static_cast<uint32_t>(Elem<DT>::store(o[1])) << 16);
                const uint32_t w1 = static_cast<uint32_t>(Elem<DT>::store(o[2])) | (static_cast<uint32_t>(Elem<DT>::store(o[3])) << 16);
                *reinterpret_cast<u32x2 *>(dst + 32 * ct + 8 * c) = u32x2{w0, w1};
            }
    }
    if (bad) raise_status(p.status, NSN_ST_NONFINITE_OUTPUT);
}

// Merge of the context splits: O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s.
// One workgroup per 32 rows (a wave's tile) of a tile, one wave per 32 channels:
// lane l holds row l % 32's channels 32*ct + 8*c + 4*(l/32) .. +3 as the
// attention kernel left them, so every read is 1 KB in a row.
template <int DT>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillParams p) {
    const int l = threadIdx.x & 63, ct = threadIdx.x >> 6;
    const int64_t tile = blockIdx.x >> 3;
    const int wave = blockIdx.x & 7;
    const int nrows = p.group * static_cast<int>(p.n_q);
    const int64_t per_tile = p.batch * p.heads_kv;
    const int64_t seqrow = tile % per_tile;
    const int r = static_cast<int>(tile / per_tile) * kQTile + 32 * wave + (l & 31);
    const int64_t tiles = (nrows + kQTile - 1) / kQTile * per_tile;
    float m[kMaxSplits], w[kMaxSplits];
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s) {
        m[s] = -INFINITY;
        w[s] = kDone;
        if (s < p.splits) {
            const float2 v = Parts(p.part, tiles, p.splits, tile, s).ml[32 * wave + (l & 31)];
            m[s] = v.x;
            w[s] = v.y;
            M = fmaxf(M, v.x);
        }
    }
    if (w[0] == kDone || r >= nrows) return;
    float L = 0.f;
    float o[4][4] = {};
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s) {
        if (w[s] != kDone) {   // (true for NaN)
            const float a = (m[s] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[s] - M);   // (0 * NaN stays NaN)
            L = __builtin_fmaf(a, w[s], L);
            const float4 *src = Parts(p.part, tiles, p.splits, tile, s).acc + (wave * 16 + 4 * ct) * 64 + l;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float4 v = src[64 * c];
                o[c][0] = __builtin_fmaf(a, v.x, o[c][0]);
                o[c][1] = __builtin_fmaf(a, v.y, o[c][1]);
                o[c][2] = __builtin_fmaf(a, v.z, o[c][2]);
                o[c][3] = __builtin_fmaf(a, v.w, o[c][3]);
            }
        }
    }
    const float rl = 1.f / L;
    bool bad = false;
    uint16_t *dst = p.out + (seqrow * nrows + r) * kDim + 32 * ct + 4 * (l >> 5);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        uint16_t e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = o[c][i] * rl;
            bad |= !finite(x);
            e[i] = Elem<DT>::store(x);
        }
        *reinterpret_cast<u32x2 *>(dst + 8 * c) =
            u32x2{static_cast<uint32_t>(e[0]) | (static_cast<uint32_t>(e[1]) << 16),
                  static_cast<uint32_t>(e[2]) | (static_cast<uint32_t>(e[3]) << 16)};
    }
    if (bad) raise_status(p.status, NSN_ST_NONFINITE_OUTPUT);
}

// Workgroups' worth of tiles of a call (256 rows of a kv-head each).
inline int64_t tile_count(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t n_q) {
    return (heads_q / heads_kv * n_q + kQTile - 1) / kQTile * batch * heads_kv;
}

inline int cu_count() {
    static const int cus = [] {      // every device is a gfx950
        int dev = 0, n = 0;
        return hipGetDevice(&dev) == hipSuccess &&
                       hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0
                   ? n
                   : 256;
    }();
    return cus;
}

}  // namespace prefill
}  // namespace nsn

using namespace nsn;

extern "C" int64_t nsn_prefill_workspace_floats(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t n_q,
                                                int n_splits) {
    using namespace nsn::prefill;
    if (batch <= 0 || heads_kv <= 0 || heads_q <= 0 || heads_q % heads_kv || n_q <= 0 || n_splits <= 1) return 0;
    return tile_count(batch, heads_q, heads_kv, n_q) * n_splits * kQTile * (kDim + 2);
}

// Context splits that pay.  Times in blocks of one workgroup (1.8 us): a
// workgroup costs 6 before its first block and after its last, a merge 4 plus
// its partials' traffic (130 KB per tile and split, written and read).
// Measured without and with the picked count: 1 sequence x 32 heads x 512
// queries over 32K tokens 892 -> 305 us (4 splits), over 4000 146 -> 74 (4);
// 7 x 32 x 128 over 16K 447 -> 292 (2); 6 ragged 5-bit sequences x 28 x 77
// over 190-3100 88 -> 48 (3); 1 x 16 x 100 over 1000 40 -> 31 (2).  From one
// tile per CU on a split only pays where it fills a half-empty last round
// (192 tiles: 281 -> 274 with 4), and below 24 blocks of capacity the merge
// costs what it saves (1 x 16 x 300 over 600: 41 -> 43 us).
extern "C" int nsn_prefill_splits(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t n_q, int64_t max_blocks) {
    using namespace nsn::prefill;
    if (batch <= 0 || heads_kv <= 0 || heads_q <= 0 || heads_q % heads_kv || n_q <= 0) return 1;
    const int64_t tiles = tile_count(batch, heads_q, heads_kv, n_q);
    if (max_blocks < 24) return 1;   // (the shortest context that is split)
    const int cus = cu_count();
    if (tiles >= cus) return 1;
    const double one = 6.0 + static_cast<double>(max_blocks);
    double best = 0.9 * one;
    int splits = 1;
    for (int s = 2; s <= kMaxSplits && 12 * s <= max_blocks; ++s) {
        const double t = static_cast<double>((tiles * s + cus - 1) / cus) * (6.0 + static_cast<double>(max_blocks) / s) +
                         4.0 + 0.036 * static_cast<double>(tiles * s);
        if (t < best) {
            best = t;
            splits = s;
        }
    }
    return splits;
}

extern "C" int nsn_prefill_attention(const nsn_prefill_args *a, nsn_stream_t stream) {
    return nsn_prefill_attention_split(a, 1, nullptr, stream);
}

extern "C" int nsn_prefill_attention_split(const nsn_prefill_args *a, int n_splits, float *workspace,
                                           nsn_stream_t stream) {
    using namespace nsn::prefill;
    if (!a || !a->q || !a->ctx_len || !a->k_chunk || !a->v_chunk || !a->out) return NSN_EINVAL;
    if (a->batch <= 0 || a->heads_kv <= 0 || a->heads_q % a->heads_kv || a->n_q < 0) return NSN_EINVAL;
    if (a->n_q == 0) return NSN_OK;
    if (a->bits != 3 && a->bits != 5) return NSN_EINVAL;
    if (a->dtype != NSN_DTYPE_F16 && a->dtype != NSN_DTYPE_BF16) return NSN_EINVAL;
    auto side_ok = [](const nsn_kv_side &s) {
        if (s.blocks && (!s.codes || !s.mins || !s.scales || !s.factors || s.block_cap <= 0)) return false;
        if (s.codes && (reinterpret_cast<uintptr_t>(s.codes) & 15u)) return false;
        if (s.mins && (reinterpret_cast<uintptr_t>(s.mins) & 15u)) return false;
        if (s.scales && (reinterpret_cast<uintptr_t>(s.scales) & 15u)) return false;
        if (s.factors && (reinterpret_cast<uintptr_t>(s.factors) & 15u)) return false;
        if (s.tail && (reinterpret_cast<uintptr_t>(s.tail) & 15u)) return false;
        if (s.tail_cap > 0 && !s.tail) return false;
        return true;
    };
    if (!side_ok(a->k) || !side_ok(a->v)) return NSN_EINVAL;
    if (!a->k.blocks != !a->v.blocks) return NSN_EINVAL;
    if (a->append && (!a->k.tail || !a->v.tail || a->k.tail_cap <= 0 || a->v.tail_cap <= 0)) return NSN_EINVAL;
    auto tail_ok = [](const nsn_kv_side &s) {
        return !s.tail || s.tail_dtype == NSN_DTYPE_F16 || s.tail_dtype == NSN_DTYPE_BF16;
    };
    if (!tail_ok(a->k) || !tail_ok(a->v)) return NSN_EINVAL;
    if (a->k.tail && a->v.tail && a->k.tail_dtype != a->v.tail_dtype) return NSN_EINVAL;
    const nsn_kv_side &ts = a->k.tail ? a->k : a->v;
    const bool tbf = ts.tail ? ts.tail_dtype == NSN_DTYPE_BF16 : a->dtype == NSN_DTYPE_BF16;
    for (const void *ptr : {static_cast<const void *>(a->q), a->k_chunk, a->v_chunk, static_cast<const void *>(a->out)})
        if (reinterpret_cast<uintptr_t>(ptr) & 15u) return NSN_EINVAL;
    const int64_t qt = (a->n_q + kQTile - 1) / kQTile;
    if (qt > 65535 || a->heads_q > 0x7fffffff || a->batch > 65535) return NSN_EINVAL;
    if (n_splits < 1 || n_splits > kMaxSplits) return NSN_EINVAL;
    if (n_splits > 1 && (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15u))) return NSN_EINVAL;
    PrefillParams p{};
    p.splits = n_splits;
    p.part = workspace;
    p.q = static_cast<const uint16_t *>(a->q);
    p.batch = a->batch;
    p.heads_q = a->heads_q;
    p.heads_kv = a->heads_kv;
    p.n_q = a->n_q;
    p.group = static_cast<int>(a->heads_q / a->heads_kv);
    p.qscale = a->scale * kLog2e;
    p.ctx_len = a->ctx_len;
    auto side = [](const nsn_kv_side &s) {
        return Side{s.codes, s.mins, s.scales, s.factors, s.blocks, s.block_cap,
                    static_cast<const uint16_t *>(s.tail), s.tail_cap};
    };
    p.k = side(a->k);
    p.v = side(a->v);
    p.kc = static_cast<const uint16_t *>(a->k_chunk);
    p.vc = static_cast<const uint16_t *>(a->v_chunk);
    p.out = static_cast<uint16_t *>(a->out);
    p.status = a->status;
    if (a->append) {   // the caller grants write access to the tails' rows past the context
        p.ka = static_cast<uint16_t *>(const_cast<void *>(a->k.tail));
        p.va = static_cast<uint16_t *>(const_cast<void *>(a->v.tail));
    }
    // One workgroup per 256 rows of a kv-head (rows: the queries of its group),
    // or of a q-head where all of those fit the CUs at once: dequantising for
    // each head again costs nothing on idle CUs, while a fuller tile takes
    // longer (1 x 32:8 heads, bf16, 64 queries over 256 tokens 20.6 -> 17.7 us,
    // 128 over 512 30.6 -> 26.6, 300 over 256 32.6 -> 29.1; none slower over 16
    // to 512 queries and 64 to 4096 tokens).
    const bool heads = n_splits == 1 && (a->n_q + kQTile - 1) / kQTile * a->heads_q * a->batch <= cu_count();
    p.run_heads = heads ? 1 : p.group;
    const int64_t tiles = (p.run_heads * a->n_q + kQTile - 1) / kQTile * n_splits;
    const int64_t wgs = tiles * a->batch * a->heads_kv;
    constexpr int64_t kMaxGrid = 1 << 22;     // workgroups of one grid dimension (2^31 threads)
    if (tiles * a->heads_kv > kMaxGrid) return NSN_EINVAL;   // (more rows than memory holds)
    const dim3 grid = wgs <= kMaxGrid ? dim3(static_cast<unsigned>(wgs), 1, static_cast<unsigned>(p.group / p.run_heads))
                                      : dim3(static_cast<unsigned>(tiles * a->heads_kv), static_cast<unsigned>(a->batch));
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool bf = a->dtype == NSN_DTYPE_BF16;
#define NSN_PREFILL_LAUNCH(B_, D_, L_)                                                                              \
    do {                                                                                                            \
        if (tbf) hipLaunchKernelGGL((prefill_kernel<B_, D_, NSN_DTYPE_BF16, L_>), grid, dim3(64 * kWaves), 0, st, p); \
        else hipLaunchKernelGGL((prefill_kernel<B_, D_, NSN_DTYPE_F16, L_>), grid, dim3(64 * kWaves), 0, st, p);      \
    } while (0)
    const bool lo = bf && a->precise_weights;
    if (a->bits == 3) {
        if (lo) NSN_PREFILL_LAUNCH(3, NSN_DTYPE_BF16, true);
        else if (bf) NSN_PREFILL_LAUNCH(3, NSN_DTYPE_BF16, false);
        else NSN_PREFILL_LAUNCH(3, NSN_DTYPE_F16, false);
    } else {
        if (lo) NSN_PREFILL_LAUNCH(5, NSN_DTYPE_BF16, true);
        else if (bf) NSN_PREFILL_LAUNCH(5, NSN_DTYPE_BF16, false);
        else NSN_PREFILL_LAUNCH(5, NSN_DTYPE_F16, false);
    }
#undef NSN_PREFILL_LAUNCH
    if (n_splits > 1) {
        if (hipGetLastError() != hipSuccess) return NSN_ELAUNCH;
        const dim3 mgrid(static_cast<unsigned>(8 * (wgs / n_splits)));   // (8 per tile; < 2^25: the grid's limit)
        if (bf) hipLaunchKernelGGL(prefill_merge_kernel<NSN_DTYPE_BF16>, mgrid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(prefill_merge_kernel<NSN_DTYPE_F16>, mgrid, dim3(256), 0, st, p);
    }
    return hipGetLastError() == hipSuccess ? NSN_OK : NSN_ELAUNCH;
}
