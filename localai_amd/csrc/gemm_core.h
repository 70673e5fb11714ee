// Pieces shared by the f16 MFMA GEMMs (gemm.hip, gemm_dense.hip): the kernel
// arguments, the decode of a weight slice into an MFMA operand, and the
// global-to-LDS copies and barriers whose completion the kernels count
// themselves.
#pragma once
#include "f16rows.h"
#include "gemv_core.h"
#include "internal.h"
#include "mfma_core.h"

namespace lq {

typedef _Float16 lq_h8 __attribute__((ext_vector_type(8)));

constexpr int GM_BK = 128;             // K values per step (two 64-value units)

typedef _Float16 lq_h2 __attribute__((ext_vector_type(2)));

// Bytes 0, 1 (lo) or 2, 3 (hi) of w below the exponent byte 0x64: two f16
// values 1024 + byte (one v_perm_b32; selector bytes 0..3 pick w's bytes,
// 4 picks the first byte of 0x64646464).
__device__ __forceinline__ uint32_t f16_bytes_lo(uint32_t w) {
    return __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u);
}
__device__ __forceinline__ uint32_t f16_bytes_hi(uint32_t w) {
    return __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
}

// Q8_0 weights straight to f16 pairs: byte q + 128 under the f16 exponent of
// 1024 reads as 1152 + q (exact), minus 1152 gives q exactly, and one f16
// multiply by d rounds d * q once (the same value as rounding the exact fp32
// product). Four int8 quants in `w` -> two f16 pairs.
__device__ __forceinline__ void q8_pairs(uint32_t w, lq_h2 d2, uint32_t &lo, uint32_t &hi) {
    const uint32_t b = w ^ 0x80808080u;
    const uint32_t l = f16_bytes_lo(b), h = f16_bytes_hi(b);
    const lq_h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    lo = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(lq_h2, l) - off) * d2);
    hi = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(lq_h2, h) - off) * d2);
}

enum { GM_DENSE = 0, GM_MOE_GATE_UP = 1, GM_MOE_DOWN = 2 };

// Dense: Xh [ntok, ldh]; Y[t * y_ts + r * y_rs].
// MoE: work tile blockIdx.y of the expert tile list (expert, first row of
// the expert-major Xh, valid rows); gate_up writes silu(g) * u to
// Y[p * y_ts + r] for r < inter, down writes Y[p * y_ts + r].
struct GemmArgs {
    lq_geom g;
    const uint8_t *W;          // dense: the matrix; MoE: expert 0 of the [E, rows, cols] handle
    const _Float16 *Xh;        // f16 rows, stride ldh (zero past cols)
    int ldh;
    const float *inv;          // per Xh row output scale
    int64_t ntok;
    float *Y;
    int64_t y_ts, y_rs;
    const int32_t *tile_e, *tile_p0, *tile_n, *n_tiles;
    int64_t inter;
    const uint8_t *Wt;         // tile form (mfma_core.h) or null; MoE: expert 0
    int64_t wt_bytes;          // tile-form bytes per matrix
    const int32_t *rows_map;   // null, or: token p reads Xh / inv row rows_map[p] / rows_k
    int rows_k;
    // MoE gate_up on the tile form, f16 output (Yh not null): SiLU * up of
    // token p goes to Yh row p (stride ldy) times 2^s, inv_out[p] = 2^-s, s
    // from the bound 4 |gate rows| |up rows| |h row|^2 (wnorm: the expert
    // handle's row_norm, xnorm2: sum of squares per Xh row)
    _Float16 *Yh;
    int64_t ldy;
    float *inv_out;
    const float *wnorm, *xnorm2;
};

// Xh / inv row of token position p
__device__ __forceinline__ int64_t gemm_xrow(const GemmArgs &a, int64_t p) {
    return a.rows_map ? (int64_t)(a.rows_map[p] / a.rows_k) : p;
}

// Workgroup barrier without the fence of __syncthreads, whose wait for every
// outstanding LDS read would stall on the next step's operand prefetch. What
// crosses it is ordered by hand: each wave waits (vmcnt) for its own copies
// into the ring before arriving, and every read of a ring slot has been
// consumed by an MFMA (lgkmcnt wait) before the barrier that precedes the
// slot's refill. The memory clobber keeps the compiler from moving memory
// accesses across it.
__device__ __forceinline__ void cu_barrier() { asm volatile("s_barrier" ::: "memory"); }

// 1 KB from global memory (16 bytes per lane) into LDS at the wave-uniform
// byte address lds (lane i's bytes at lds + 16 i), through M0, which it saves
// and restores
__device__ __forceinline__ void cu_dma(const void *src, uint32_t lds) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(src), "s"(lds)
                 : "memory");
}
// global loads with a wave-uniform 64-bit base in SGPRs and a 32-bit per-lane
// byte offset (fewer VGPRs than 64-bit addresses per load)
__device__ __forceinline__ void cu_load(mt_i4 &v, const void *base, uint32_t off) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void cu_load(int &v, const void *base, uint32_t off) {
    asm volatile("global_load_dword %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}

template <int T> struct GtRaw;
template <> struct GtRaw<LQ_Q4_K> { uint4 qs, hd; };
template <> struct GtRaw<LQ_Q6_K> { uint4 ql, qh, sc; uint32_t d; };
template <> struct GtRaw<LQ_Q8_0> { uint4 p0, p1, dd; };

// Q4_K sub-block scale pair {d * sc, dmin * mn} (packed f16, each rounded
// once) of row lane % 16, sub-block 4 HALF + lane / 16: the four lane groups
// of a wave cover the four sub-blocks of a half at once; gt_b fetches the
// pair of its own sub-block from the lane that computed it
template <int HALF>
__device__ __forceinline__ uint32_t gt_q4k_pair(const uint4 &hd, int q) {
    const uint32_t s0 = hd.y, s4 = hd.z, s8 = hd.w;   // scale bytes 0..3, 4..7, 8..11
    uint32_t sc, mn;
    if constexpr (HALF == 0) {
        sc = __builtin_amdgcn_ubfe(s0, 8 * q, 6);
        mn = __builtin_amdgcn_ubfe(s4, 8 * q, 6);
    } else {
        sc = __builtin_amdgcn_ubfe(s8, 8 * q, 4) | (__builtin_amdgcn_ubfe(s0, 8 * q + 6, 2) << 4);
        mn = __builtin_amdgcn_ubfe(s8, 8 * q + 4, 4) | (__builtin_amdgcn_ubfe(s4, 8 * q + 6, 2) << 4);
    }
    // packed f16: {sc, mn} exactly (0x6400 | n reads as 1024 + n), times
    // {d, dmin} rounds d * sc and dmin * mn once each
    const lq_h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const lq_h2 scmn = __builtin_bit_cast(lq_h2, sc | (mn << 16) | 0x64006400u) - k1024;
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(lq_h2, hd.x) * scmn);
}

// B operand (8 f16) of slice kk (0..3) of half HALF of the block, lane group
// q; Q4_K: pair = the slice's scale pair for the lane's row (gt_q4k_pair)
template <int T, int HALF, int KK>
__device__ __forceinline__ lq_h8 gt_b(const GtRaw<T> &r, int q, uint32_t pair_ab = 0) {
    uint4 o;
    if constexpr (T == LQ_Q4_K) {
        // group g = 4 HALF + KK: qs chunk g / 2 (bytes 8 ((g / 2) % 2) ..), nibble g % 2;
        // a value is round(a * q - b) from the exact q (one fused multiply-add)
        constexpr int g = 4 * HALF + KK, hb = (g >> 1) & 1, nib = g & 1;
        const lq_h2 ab = __builtin_bit_cast(lq_h2, pair_ab);
        const lq_h2 a2 = {ab.x, ab.x}, nb2 = {-ab.y, -ab.y};
        const uint32_t w0 = ((hb ? r.qs.z : r.qs.x) >> (4 * nib)) & 0x0F0F0F0Fu;
        const uint32_t w1 = ((hb ? r.qs.w : r.qs.y) >> (4 * nib)) & 0x0F0F0F0Fu;
        // the byte 0000qqqq read as FP8 e4m3 is exactly q 2^-9 (subnormal
        // below 8, normal from 8 on); the scaled conversion times 2^9 gives
        // two f16 q exactly in one instruction
        auto fma2 = [&](lq_h2 q) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, a2, nb2)); };
        o.x = fma2(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 512.0f, false));
        o.y = fma2(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 512.0f, true));
        o.z = fma2(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 512.0f, false));
        o.w = fma2(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 512.0f, true));
    } else if constexpr (T == LQ_Q6_K) {
        // slice g = 4 HALF + KK: values 128 HALF + 32 KK + 8q .. ; ql nibble KK / 2 of
        // bytes 8 (KK % 2) ..; qh bits 2 KK of bytes 8 HALF ..; sub-block 2g + q / 2
        constexpr int g = 4 * HALF + KK;
        const uint32_t l0 = ((KK & 1) ? r.ql.z : r.ql.x) >> (4 * (KK >> 1));
        const uint32_t l1 = ((KK & 1) ? r.ql.w : r.ql.y) >> (4 * (KK >> 1));
        const uint32_t e0 = (HALF ? r.qh.z : r.qh.x) >> (2 * KK), e1 = (HALF ? r.qh.w : r.qh.y) >> (2 * KK);
        const uint32_t w0 = (l0 & 0x0F0F0F0Fu) | ((e0 & 0x03030303u) << 4);
        const uint32_t w1 = (l1 & 0x0F0F0F0Fu) | ((e1 & 0x03030303u) << 4);
        // sub-blocks 2g and 2g + 1 share scale dword g / 2
        const uint32_t sw = (g >> 1) == 0 ? r.sc.x : (g >> 1) == 1 ? r.sc.y : (g >> 1) == 2 ? r.sc.z : r.sc.w;
        const int sbyte = ((2 * g) & 3) + (q >> 1);
        // packed f16: 1024 + q minus 1056 is q - 32 exactly; times d * sc
        // (rounded once) rounds each value once
        const _Float16 dsc = __builtin_bit_cast(_Float16, (uint16_t)(r.d & 0xFFFFu)) *
                             (_Float16)(int)__builtin_amdgcn_sbfe((int)sw, 8 * sbyte, 8);
        const lq_h2 d2 = {dsc, dsc}, k1056 = {(_Float16)1056.0f, (_Float16)1056.0f};
        auto pair = [&](uint32_t bits) {
            return __builtin_bit_cast(uint32_t, (__builtin_bit_cast(lq_h2, bits) - k1056) * d2);
        };
        o.x = pair(f16_bytes_lo(w0));
        o.y = pair(f16_bytes_hi(w0));
        o.z = pair(f16_bytes_lo(w1));
        o.w = pair(f16_bytes_hi(w1));
    } else {
        // GGML block 4 HALF + KK: piece KK / 2 of the half, bytes 8 (KK % 2) ..
        const uint4 pc = (KK >> 1) ? r.p1 : r.p0;
        const uint32_t w0 = (KK & 1) ? pc.z : pc.x, w1 = (KK & 1) ? pc.w : pc.y;
        constexpr int g = 4 * HALF + KK;
        const uint32_t dw = g < 2 ? r.dd.x : g < 4 ? r.dd.y : g < 6 ? r.dd.z : r.dd.w;
        const uint32_t dh = (dw >> (16 * (g & 1))) & 0xFFFFu;
        const lq_h2 d2 = __builtin_bit_cast(lq_h2, dh * 0x10001u);
        q8_pairs(w0, d2, o.x, o.y);
        q8_pairs(w1, d2, o.z, o.w);
    }
    return __builtin_bit_cast(lq_h8, o);
}

// Dense product (gemm_dense.hip), a.Wt (Q4_K, Q6_K, Q8_0) or the row planes a.W
// (Q5_K, Q4_0), a.Xh / a.inv filled in;
// split_ws: up to split_bytes of scratch for K splits (none: one split)
int launch_gemm_dense(const GemmArgs &a, void *split_ws, int64_t split_bytes, hipStream_t s);
double gemm_dense_us(const lq_geom &g, int64_t ntok, int64_t *split_bytes);

}  // namespace lq
