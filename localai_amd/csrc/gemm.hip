// Prefill matmul on MFMA: Y[t, r] = sum_c W[r, c] * X[t, c] for many tokens.
//
// Counterpart of decoded_matmul_row / localai_*_matmul
// (engine/native_quant.cpp:444-531, :744-768): the reference decodes each row
// exactly to fp32 and runs fp32 FMAs over the tokens. Here weights are decoded
// exactly (the per-type formulas of the dequant kernels), rounded once to f16
// and multiplied with v_mfma_f32_16x16x32_f16 in fp32 accumulation.
//
// Activations are converted once per call (x_to_f16): each token row is scaled
// by a power of two so that its largest magnitude lies in [2^14, 2^15)
// (exact), rounded to f16, and the output is scaled back by the inverse power.
// f16 (11 significant bits) rather than bf16 (8) keeps the normwise error near
// 2^-12.
//
// Three kernels:
//   gemm_dense_kernel (gemm_dense.hip) dense products of handles in their
//                     type's usual form (tile form for Q4_K / Q6_K / Q8_0, row
//                     planes for Q5_K / Q4_0);
//   gemm_tile_kernel  the MoE expert tiles and the dense products of short K
//                     (gemm_takes_tile_kernel) on the tile form: each wave
//                     decodes its own two 16-row tiles into B operands in
//                     registers, x is staged in LDS (global_load_lds);
//   gemm_kernel       from the row planes of any type: the MoE expert tiles of
//                     handles without a tile form (Q4_0, Q5_K, or every type
//                     with LOCALAI_HIP_MFMA_MATVEC=0), and the dense products of
//                     Q4_K / Q6_K / Q8_0 handles made with that switch. A
//                     workgroup decodes a 128-row weight tile into LDS per
//                     128-value step and 4 waves multiply it with 128 tokens
//                     (expert tiles: 64).
#include <type_traits>

#include "gemm_core.h"

namespace lq {

constexpr int GM_BM = 128;             // weight rows per workgroup
constexpr int GM_BN = 128;             // tokens per workgroup (dense)
constexpr int GM_MOE_BN = 64;          // tokens per workgroup (MoE expert tiles)
constexpr int GM_LD = GM_BK + 8;       // LDS row stride in halves (272 B: 16 lanes of a
                                       // 16-byte read hit 16 distinct bank groups)

// ---------------------------------------------------------------- activations

// One wave per token row, four rows per workgroup (x_to_f16_row, f16rows.h).
template <int NG>
__global__ __launch_bounds__(256) void x_to_f16_kernel(const float *__restrict__ X, int64_t ldx, int cols,
                                                       const int32_t *__restrict__ rows_map, int k, int64_t ntok,
                                                       _Float16 *__restrict__ Xh, int ldh,
                                                       float *__restrict__ inv, int vec, float *__restrict__ nrm2) {
    const int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + wave_id();
    x_to_f16_row<NG>(t, X, ldx, cols, rows_map, k, ntok, Xh, ldh, inv, vec, nrm2);
}

// Rows of more than 2048 values: one workgroup per token row, its 256 threads
// holding the row's 8-value groups (NG each, at most 16384 values) between the
// maximum and the conversion; the same scale and values as x_to_f16_row. 333
// rows of 14336 values: 6.9 us; one wave per row, reading it twice, 19.8 us. A
// wave per row holds 4096 values too, but its eight loads a lane are latency: the
// 77-token product of 4096 x 4096 23.3 -> 22.7 us, 1000 tokens 36.9 -> 36.5; at
// 1024 values the wave per row is ahead (26.4 us against 26.5).
template <int NG>
__global__ __launch_bounds__(256) void x_to_f16_wide_kernel(const float *__restrict__ X, int64_t ldx, int cols,
                                                            const int32_t *__restrict__ rows_map, int k,
                                                            _Float16 *__restrict__ Xh, int ldh,
                                                            float *__restrict__ inv, int vec) {
    __shared__ uint32_t wmax[4];
    const int64_t t = blockIdx.x;
    const float *x = X + (rows_map ? (int64_t)(rows_map[t] / k) : t) * ldx;
    const int ngx = cols >> 3, ng = ldh >> 3;
    lq_f4 lo[NG], hi[NG];
    uint32_t mb = 0;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int gi = threadIdx.x + 256 * i;
        lo[i] = hi[i] = lq_f4{0.f, 0.f, 0.f, 0.f};
        if (gi < ngx) {
            if (vec) {
                lo[i] = *reinterpret_cast<const lq_f4 *>(x + 8 * gi);
                hi[i] = *reinterpret_cast<const lq_f4 *>(x + 8 * gi + 4);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lo[i][c] = x[8 * gi + c];
                    hi[i][c] = x[8 * gi + 4 + c];
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) mb = max(mb, max(f16_mag(lo[i]), f16_mag(hi[i])));
    mb = wave_max_u32(mb);
    if (lane_id() == 0) wmax[wave_id()] = mb;
    __syncthreads();
    const int s = f16_row_shift(max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
    const float sc = ldexpf(1.0f, s);
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int gi = threadIdx.x + 256 * i;
        if (gi >= ng) continue;
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        h8 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            o[c] = (_Float16)(lo[i][c] * sc);
            o[4 + c] = (_Float16)(hi[i][c] * sc);
        }
        *reinterpret_cast<h8 *>(Xh + t * ldh + 8 * gi) = o;
    }
    if (threadIdx.x == 0) inv[t] = ldexpf(1.0f, -s);
}

// ---------------------------------------------------------------- weights

// Exact fp32 values of unit u in unit order (the order of gemv_core.h's x
// windows); the same formulas as engine/dequant.py:62-165. Q8_0 has its own
// conversion (q8_pairs).
template <int T>
__device__ __forceinline__ void dequant_unit(const UnitW &w, int u, float *out) {
    if constexpr (T == LQ_Q4_K || T == LQ_Q5_K) {
        const int p = u & 3;
        uint32_t sc0, sc1, mn0, mn1;
        kq_pair(w.h0, p, sc0, sc1, mn0, mn1);
        const float d = f16_to_f32(w.h0.x), dmin = f16_to_f32(w.h0.x >> 16);
        const float a0 = d * (float)sc0, a1 = d * (float)sc1;
        const float b0 = dmin * (float)mn0, b1 = dmin * (float)mn1;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint32_t byte = (u4_get(j < 16 ? w.q0 : w.q1, (j & 15) >> 2) >> (8 * (j & 3))) & 0xFFu;
            uint32_t lo = byte & 15u, hi = byte >> 4;
            if constexpr (T == LQ_Q5_K) {
                const uint32_t qh = (u4_get(j < 16 ? w.h1 : w.q2, (j & 15) >> 2) >> (8 * (j & 3))) & 0xFFu;
                lo |= ((qh >> (2 * p)) & 1u) << 4;
                hi |= ((qh >> (2 * p + 1)) & 1u) << 4;
            }
            out[j] = __builtin_fmaf(a0, (float)lo, -b0);
            out[32 + j] = __builtin_fmaf(a1, (float)hi, -b1);
        }
    } else if constexpr (T == LQ_Q6_K) {
        const float d = f16_to_f32(w.d);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float dc = d * (float)(int8_t)(w.sc >> (8 * c));
            const uint4 ql = (c & 1) ? w.q1 : w.q0;
            const uint32_t sh = (c >> 1) * 4, hs = 2 * c;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t qb = (u4_get(ql, e >> 2) >> (8 * (e & 3) + sh)) & 15u;
                const uint32_t hb = (u4_get(w.h0, e >> 2) >> (8 * (e & 3) + hs)) & 3u;
                out[16 * c + e] = dc * (float)((int)(qb | (hb << 4)) - 32);
            }
        }
    } else {   // Q4_0
        const float d0 = f16_to_f32(w.sc), d1 = f16_to_f32(w.sc >> 16);
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint4 q = j < 16 ? w.q0 : w.q1;
            const uint32_t byte = (u4_get(q, (j & 15) >> 2) >> (8 * (j & 3))) & 0xFFu;
            const float d = j < 16 ? d0 : d1;
            out[2 * (j & ~15) + (j & 15)] = d * (float)((int)(byte & 15u) - 8);
            out[2 * (j & ~15) + 16 + (j & 15)] = d * (float)((int)(byte >> 4) - 8);
        }
    }
}

// Position inside the 128-value step window of value j (unit order) of unit u.
template <int T>
__device__ __forceinline__ int window_pos(int u, int j) {
    if constexpr (T == LQ_Q6_K) return 32 * (j >> 4) + 16 * (u & 1) + (j & 15);
    else return 64 * (u & 1) + j;
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    const _Float16 ha = (_Float16)a, hb = (_Float16)b;
    return (uint32_t)__builtin_bit_cast(uint16_t, ha) | ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
}

// ---------------------------------------------------------------- GEMM

template <int T, int BN, int MODE>
__global__ __launch_bounds__(256, 2) void gemm_kernel(GemmArgs a) {
    constexpr int NI = BN / 32;            // 16-token MFMA tiles per wave (waves split tokens in 2)
    __shared__ __attribute__((aligned(16))) _Float16 Ws[GM_BM * GM_LD];
    __shared__ __attribute__((aligned(16))) _Float16 Xs[BN * GM_LD];
    const lq_geom &g = a.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    // token tile
    const uint8_t *W = a.W;
    int64_t p0;
    int tn;
    int64_t rtile;
    if constexpr (MODE == GM_DENSE) {
        // 1-D grid, padded to a multiple of 8. Workgroups are dispatched to the
        // 8 XCDs round-robin (id % 8); workgroup id -> logical index
        // xcd * per + id / 8 walks the row tiles of one token tile per XCD, so
        // each XCD's L2 holds one activation tile while the weights stream.
        const int id = blockIdx.x, per = gridDim.x / 8;
        const int L = (id % 8) * per + id / 8;
        const int nrt = (int)((g.rows + GM_BM - 1) / GM_BM);
        const int64_t ntt = (a.ntok + BN - 1) / BN;
        if (L >= nrt * ntt) return;
        rtile = L % nrt;
        p0 = (int64_t)(L / nrt) * BN;
        tn = (int)(a.ntok - p0 < BN ? a.ntok - p0 : BN);
    } else {
        rtile = blockIdx.x;
        const int tile = blockIdx.y;
        if (tile >= a.n_tiles[0]) return;
        W += (int64_t)a.tile_e[tile] * g.matrix_bytes;
        p0 = a.tile_p0[tile];
        tn = a.tile_n[tile];
    }
    // weight rows of this tile: q -> matrix row (or -1 when past the end)
    const int64_t r0 = rtile * (MODE == GM_MOE_GATE_UP ? GM_BM / 2 : GM_BM);
    auto row_of = [&](int q) -> int64_t {
        if constexpr (MODE == GM_MOE_GATE_UP) {
            // wave row block rb = q / 64, MFMA tile j = (q % 64) / 16: j < 2 gate, j >= 2 up,
            // so a lane holds the gate and up sums of the same row in tiles j and j + 2
            const int rb = q >> 6, j = (q >> 4) & 3, rr = q & 15;
            const int64_t r = r0 + 32 * rb + 16 * (j & 1) + rr;
            return r < a.inter ? r + (j >> 1) * a.inter : -1;
        } else {
            return r0 + q < g.rows ? r0 + q : -1;
        }
    };
    const int U = (int)g.nu, steps = (U + 1) / 2;
    const int lr = tid >> 1, lh = tid & 1;
    int64_t wrow = row_of(lr);
    wrow = wrow < 0 ? 0 : wrow;
    // activation loader: BN rows x 128 values, 256 threads
    constexpr int XT = 256 / BN;              // threads per token row (2 or 4 or 8)
    constexpr int XV = 128 / XT;              // halves per thread
    const int xr = tid / XT, xp = tid % XT;
    const int64_t xrow = gemm_xrow(a, p0 + (xr < tn ? xr : 0));
    const _Float16 *xsrc = a.Xh + xrow * a.ldh + XV * xp;

    UnitW wreg;
    uint4 xreg[XV / 8];
    auto load = [&](int step) {
        const int u = 2 * step + lh;
        const int uc = u < U ? u : U - 1;
        const int c0 = uc & ~63;
        const int C = U - c0 < 64 ? U - c0 : 64;
        wreg = load_unit_w<T>(W, g, wrow, uc, C);
        const uint4 *xp4 = reinterpret_cast<const uint4 *>(xsrc + (int64_t)step * GM_BK);
#pragma unroll
        for (int i = 0; i < XV / 8; ++i) xreg[i] = xp4[i];
    };
    auto store = [&](int step) {
        const int u = 2 * step + lh;
        const bool valid = u < U;
        _Float16 *wd = Ws + lr * GM_LD;
        if constexpr (T == LQ_Q8_0) {
            const uint32_t dm = valid ? 0xFFFFFFFFu : 0u;
            const lq_h2 d0 = __builtin_bit_cast(lq_h2, ((wreg.sc & 0xFFFFu) * 0x10001u) & dm);
            const lq_h2 d1 = __builtin_bit_cast(lq_h2, ((wreg.sc >> 16) * 0x10001u) & dm);
            const uint4 qs[4] = {wreg.q0, wreg.q1, wreg.q2, wreg.q3};
#pragma unroll
            for (int c = 0; c < 8; ++c) {      // 8 values per 16-byte LDS write
                const uint4 q = qs[c >> 1];
                const lq_h2 d2 = c < 4 ? d0 : d1;
                uint4 p;
                q8_pairs(u4_get(q, 2 * (c & 1)), d2, p.x, p.y);
                q8_pairs(u4_get(q, 2 * (c & 1) + 1), d2, p.z, p.w);
                *reinterpret_cast<uint4 *>(wd + 64 * (u & 1) + 8 * c) = p;
            }
        } else {
            float v[64];
            dequant_unit<T>(wreg, u < U ? u : U - 1, v);
#pragma unroll
            for (int j = 0; j < 64; j += 8) {
                uint4 p;
                p.x = valid ? pack_h2(v[j + 0], v[j + 1]) : 0u;
                p.y = valid ? pack_h2(v[j + 2], v[j + 3]) : 0u;
                p.z = valid ? pack_h2(v[j + 4], v[j + 5]) : 0u;
                p.w = valid ? pack_h2(v[j + 6], v[j + 7]) : 0u;
                *reinterpret_cast<uint4 *>(wd + window_pos<T>(u, j)) = p;
            }
        }
        uint4 *xd = reinterpret_cast<uint4 *>(Xs + xr * GM_LD + XV * xp);
#pragma unroll
        for (int i = 0; i < XV / 8; ++i) xd[i] = xreg[i];
    };

    lq_f4 acc[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = lq_f4{0.0f, 0.0f, 0.0f, 0.0f};

    const int tb = wave >> 1, rb = wave & 1;
    const int fr = lane & 15, fk = 8 * (lane >> 4);
    load(0);
    for (int s = 0; s < steps; ++s) {
        store(s);
        __syncthreads();
        if (s + 1 < steps) load(s + 1);
#pragma unroll
        for (int kk = 0; kk < GM_BK / 32; ++kk) {
            lq_h8 av[NI], bv[4];
#pragma unroll
            for (int i = 0; i < NI; ++i)
                av[i] = *reinterpret_cast<const lq_h8 *>(Xs + ((BN / 2) * tb + 16 * i + fr) * GM_LD + 32 * kk + fk);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bv[j] = *reinterpret_cast<const lq_h8 *>(Ws + (64 * rb + 16 * j + fr) * GM_LD + 32 * kk + fk);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // D[m][n]: lane holds tokens 4 * (lane / 16) + v of token tile i, row lane % 16 of row tile j
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int lt = (BN / 2) * tb + 16 * i + 4 * (lane >> 4) + v;
            if (lt >= tn) continue;
            const int64_t p = p0 + lt;
            const float sc = a.inv[gemm_xrow(a, p)];
            if constexpr (MODE == GM_MOE_GATE_UP) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int64_t r = r0 + 32 * rb + 16 * j + fr;
                    if (r < a.inter) {
                        const float gv = acc[i][j][v] * sc, uv = acc[i][j + 2][v] * sc;
                        a.Y[p * a.y_ts + r] = silu(gv) * uv;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int64_t r = r0 + 64 * rb + 16 * j + fr;
                    if (r < g.rows) a.Y[p * a.y_ts + r * a.y_rs] = acc[i][j][v] * sc;
                }
            }
        }
    }
}

// --------------------------------------------------- GEMM on the tile form
// Q4_K / Q6_K / Q8_0 handles carry the tile form (mfma_core.h). For a 32-value
// slice of a 256-value block, the 8 quants that lane l (weight row l % 16,
// k = 8 (l / 16) .. + 7) holds in its 16-byte slice are exactly that lane's
// part of the B operand of v_mfma_f32_16x16x32_f16. So a wave decodes its own
// weight rows straight into B registers -- each weight value once per
// workgroup, exactly in fp32 (or, for Q8_0, exactly as 1152 + q in f16 times
// d), rounded once to f16 -- and only the f16 activations (A operands) go
// through LDS, double-buffered and shared by the waves.
//
// Workgroup: 8 waves x 2 row tiles (256 weight rows; for gate_up 128 gate rows
// and the 128 matching up rows) x 64 tokens; dense: 4 waves x 2 row tiles x 128
// tokens; 128 K values per step.

constexpr int GM_MOE_NW = 8;           // waves per workgroup of the expert tile GEMMs

// weights of half `half` (values 128 half .. + 127) of one 256-value block
template <int T>
__device__ __forceinline__ GtRaw<T> gt_load(const uint8_t *blk, int half, int lane) {
    GtRaw<T> r;
    const int n = lane & 15;
    if constexpr (T == LQ_Q4_K) {
        r.qs = ld16(blk + half * 1024 + 16 * lane);
        // the scales once per block, with half 0 (the loop derives half 1's
        // scale pairs from them too)
        if (half == 0) r.hd = ld16(blk + 2048 + 16 * n);
    } else if constexpr (T == LQ_Q6_K) {
        r.ql = ld16(blk + half * 1024 + 16 * lane);
        r.qh = ld16(blk + 2048 + 16 * lane);
        r.sc = ld16(blk + 3072 + 16 * n);
        r.d = *reinterpret_cast<const uint16_t *>(blk + 3328 + 2 * n);
    } else {
        r.p0 = ld16(blk + 2 * half * 1024 + 16 * lane);
        r.p1 = ld16(blk + (2 * half + 1) * 1024 + 16 * lane);
        r.dd = ld16(blk + 4096 + 16 * n);
    }
    return r;
}

// MFMAs of the four 32-value slices of half HALF of a block: B operands
// decoded from the wave's two row tiles, A operands from the LDS x tile
// x tile in LDS: [token][16 chunks of 8 halves], chunk c of token t stored at
// position c ^ (t % 16), so the 16 tokens of an A read hit 16 bank groups.
// The wave raises its priority while it issues a slice's MFMAs, so the wave
// that holds ready MFMAs keeps the matrix core of its SIMD (the waves of a
// SIMD come from different workgroups); the expert GEMMs gain about 1 %.
// Q4_K: pr0 / pr1 are the scale pairs of this half (gt_q4k_pair), computed
// by the caller while half 0's scale registers are live
template <int T, int HALF, int NI>
__device__ __forceinline__ void gt_half(const GtRaw<T> &w0, const GtRaw<T> &w1, const _Float16 *xs, int lane,
                                        lq_f4 (&acc)[NI][2], uint32_t pr0 = 0, uint32_t pr1 = 0) {
    const int fr = lane & 15, q = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        // all A reads of the slice in flight while the B operands are decoded
        lq_h8 av[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i)
            av[i] = *reinterpret_cast<const lq_h8 *>(xs + (16 * i + fr) * GM_BK + 8 * ((4 * kk + q) ^ fr));
        uint32_t p0 = 0, p1 = 0;
        if constexpr (T == LQ_Q4_K) {
            // the pair of sub-block 4 HALF + kk of the lane's row: lane fr + 16 kk
            const int src = 4 * (fr + 16 * kk);
            p0 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)pr0);
            p1 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)pr1);
        }
        lq_h8 b0, b1;
        if (kk == 0) { b0 = gt_b<T, HALF, 0>(w0, q, p0); b1 = gt_b<T, HALF, 0>(w1, q, p1); }
        else if (kk == 1) { b0 = gt_b<T, HALF, 1>(w0, q, p0); b1 = gt_b<T, HALF, 1>(w1, q, p1); }
        else if (kk == 2) { b0 = gt_b<T, HALF, 2>(w0, q, p0); b1 = gt_b<T, HALF, 2>(w1, q, p1); }
        else { b0 = gt_b<T, HALF, 3>(w0, q, p0); b1 = gt_b<T, HALF, 3>(w1, q, p1); }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], b0, acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], b1, acc[i][1], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
    }
}

// Waits for the loads of gt_load<T>(.., HALF, ..) into r (the compiler places
// the wait before these empty asm statements, which read and rewrite the
// loaded registers)
__device__ __forceinline__ void gt_touch(uint4 &v) {
    typedef unsigned u4v __attribute__((ext_vector_type(4)));
    u4v t = __builtin_bit_cast(u4v, v);
    asm volatile("" : "+v"(t));
    v = __builtin_bit_cast(uint4, t);
}
template <int T, int HALF>
__device__ __forceinline__ void gt_ready(GtRaw<T> &r) {
    if constexpr (T == LQ_Q4_K) {
        gt_touch(r.qs);
        if constexpr (HALF == 0) gt_touch(r.hd);
    } else if constexpr (T == LQ_Q6_K) {
        gt_touch(r.ql);
        gt_touch(r.qh);
        gt_touch(r.sc);
        asm volatile("" : "+v"(r.d));
    } else {
        gt_touch(r.p0);
        gt_touch(r.p1);
        gt_touch(r.dd);
    }
}

// Global loads gt_load<T> issues for one row tile's half HALF
template <int T, int HALF>
constexpr int gt_loads() {
    return T == LQ_Q4_K ? (HALF == 0 ? 2 : 1) : T == LQ_Q6_K ? 4 : 3;
}

// The K loop and epilogue of one workgroup with NV 16-token MFMA tiles of
// the BN holding tokens: expert tiles end partway, and each NV is its own
// copy of the loop (no per-MFMA branches, which made the compiler copy the
// accumulators around every conditional MFMA).
template <int T, int BN, int MODE, int NW, int NV>
__device__ __forceinline__ void gt_main(const GemmArgs &a, _Float16 (*Xs)[BN * GM_BK], float *tsc, float *asc,
                                        const float *wn, const uint8_t *w0p, const uint8_t *w1p, int64_t p0, int tn,
                                        int64_t t0, int64_t t1, int64_t tiles, int64_t nsb) {
    constexpr int XN = BN * 16 / (64 * NW);   // 16-byte x chunks per thread and step
    constexpr int BB = mt_block_bytes(T);
    const lq_geom &g = a.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();

    // x loader: instruction i of wave w fills tile chunks (NW i + w) * 64 + lane,
    // i.e. token row (NW i + w) * 4 + lane / 16, position lane % 16, from the
    // row's chunk (lane % 16) ^ (row % 16); straight from global memory into
    // LDS (no registers), waited for with vmcnt before the step's barrier.
    // Rows of the MFMA tiles past NV are not read.
    const _Float16 *xsrc[XN];
#pragma unroll
    for (int i = 0; i < XN; ++i) {
        const int row = (NW * i + wave) * 4 + (lane >> 4), c = (lane & 15) ^ (row & 15);
        xsrc[i] = a.Xh + gemm_xrow(a, p0 + (row < tn ? row : 0)) * a.ldh + 8 * c;
    }
    // The copies are asm (cu_dma): the compiler, which sees a builtin copy as
    // an LDS write it cannot place, waited for every load (vmcnt(0)) before
    // the first LDS read after one, the weight loads just issued included.
    // Their completion before the LDS reads is the kernel's own wait before
    // each barrier.
    const uint32_t xs0 = (uint32_t)(uintptr_t)&Xs[0][0];
    auto load_x = [&](int buf, int64_t step) {
#pragma unroll
        for (int i = 0; i < XN; ++i)
            if ((NW * i + wave) * 4 < 16 * NV)   // uniform per wave
                cu_dma(xsrc[i] + step * GM_BK, xs0 + (uint32_t)(buf * BN * GM_BK * 2 + (NW * i + wave) * 64 * 16));
    };

    lq_f4 acc[NV][2];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        acc[i][0] = lq_f4{0.0f, 0.0f, 0.0f, 0.0f};
        acc[i][1] = lq_f4{0.0f, 0.0f, 0.0f, 0.0f};
    }

    // prologue: half 0 of block 0, and each token's output scale (one
    // lookup per token rather than one per output value)
    GtRaw<T> a0 = gt_load<T>(w0p, 0, lane), a1 = gt_load<T>(w1p, 0, lane);
    load_x(0, 0);
    if (tid < BN) {
        const int64_t xr = gemm_xrow(a, p0 + (tid < tn ? tid : 0));
        tsc[tid] = a.inv[xr];
        if constexpr (MODE == GM_MOE_GATE_UP) {
            if (a.Yh) {
                // |silu(g) u| <= |g| |u| <= |gate row| |up row| |h|^2 (Cauchy-
                // Schwarz), times 4 for the rounding of the f16 operands, the
                // sums and the fast SiLU; 2^s brings the bound into [2^14,
                // 2^15), so no output overflows f16 (s = 0 for a zero or
                // non-finite bound, x_to_f16_row's rule)
                const double b = 4.0 * (double)wn[0] * (double)wn[1] * (double)a.xnorm2[xr];
                int s = 0;
                if (b > 0.0 && b <= 1.0e300) {
                    int e;
                    frexp(b, &e);
                    s = 15 - e;
                    s = s > 120 ? 120 : s < -120 ? -120 : s;
                }
                asc[tid] = ldexpf(1.0f, s);
                if (blockIdx.x == 0 && tid < tn) a.inv_out[p0 + tid] = ldexpf(1.0f, -s);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // step loop over blocks: half 0 from Xs[0] / (a0, a1), half 1 from Xs[1] /
    // (b0, b1). Each half waits for its own weights (requested one half
    // earlier), then requests the next half's x copy and, after it, the next
    // half's weights, so the wait before the barrier (vmcnt = those weight
    // loads) retires only the copy: the weights stay in flight across it.
    for (int64_t sb = 0; sb < nsb; ++sb) {
        gt_ready<T, 0>(a0);
        gt_ready<T, 0>(a1);
        // Q4_K: both halves' scale pairs now, so the block's scale registers
        // die in half 0 and the next block's scales load straight into them
        // (kept live into half 1, the compiler copied each freshly loaded
        // scale register and waited for the load right after issuing it)
        uint32_t p00 = 0, p01 = 0, p10 = 0, p11 = 0;
        if constexpr (T == LQ_Q4_K) {
            const int q = lane >> 4;
            p00 = gt_q4k_pair<0>(a0.hd, q);
            p01 = gt_q4k_pair<0>(a1.hd, q);
            p10 = gt_q4k_pair<1>(a0.hd, q);
            p11 = gt_q4k_pair<1>(a1.hd, q);
        }
        load_x(1, 2 * sb + 1);
        GtRaw<T> b0 = gt_load<T>(w0p + sb * BB, 1, lane), b1 = gt_load<T>(w1p + sb * BB, 1, lane);
        // nothing crosses: the loads stay ahead of the MFMAs
        __builtin_amdgcn_sched_barrier(0);
        gt_half<T, 0, NV>(a0, a1, Xs[0], lane, acc, p00, p01);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * gt_loads<T, 1>()) : "memory");
        __syncthreads();
        gt_ready<T, 1>(b0);
        gt_ready<T, 1>(b1);
        // next block (the last block re-reads itself: Xs[0] is not read again)
        const int64_t nx = sb + 1 < nsb ? sb + 1 : sb;
        load_x(0, 2 * nx);
        a0 = gt_load<T>(w0p + nx * BB, 0, lane);
        a1 = gt_load<T>(w1p + nx * BB, 0, lane);
        __builtin_amdgcn_sched_barrier(0);
        gt_half<T, 1, NV>(b0, b1, Xs[1], lane, acc, p10, p11);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * gt_loads<T, 0>()) : "memory");
        __syncthreads();
    }
    // D[m][n]: lane holds tokens 4 (lane / 16) + v of token tile i, row lane % 16 of row tile j.
    // Addresses advance from one base per row; 32-bit offsets (a tile spans
    // at most BN rows of Y)
    const int fr = lane & 15;
    if constexpr (MODE == GM_MOE_GATE_UP) {
        const int64_t r = t0 * MT_ROWS + fr;
        const bool rok = r < a.inter;
        if (a.Yh) {
            // the f16 rows the down GEMM reads: the same f32 value times
            // 2^s, rounded once (as x_to_f16_row rounds it)
            _Float16 *hb = a.Yh + p0 * a.ldy + r;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int lt = 16 * i + 4 * (lane >> 4) + v;
                    if (lt >= tn || !rok) continue;
                    const float sc = tsc[lt];
                    const float y = silu_fast(acc[i][0][v] * sc) * (acc[i][1][v] * sc);
                    hb[(uint32_t)lt * (uint32_t)a.ldy] = (_Float16)(y * asc[lt]);
                }
            }
        } else {
            float *yb = a.Y + p0 * a.y_ts + r;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int lt = 16 * i + 4 * (lane >> 4) + v;
                    if (lt >= tn || !rok) continue;
                    const float sc = tsc[lt];
                    yb[(uint32_t)lt * (uint32_t)a.y_ts] = silu_fast(acc[i][0][v] * sc) * (acc[i][1][v] * sc);
                }
            }
        }
    } else {
        const int64_t r0 = t0 * MT_ROWS + fr, r1 = t1 * MT_ROWS + fr;
        const bool ok0 = t0 < tiles && r0 < g.rows, ok1 = t1 < tiles && r1 < g.rows;
        float *yb0 = a.Y + p0 * a.y_ts + r0 * a.y_rs, *yb1 = a.Y + p0 * a.y_ts + r1 * a.y_rs;
        if constexpr (MODE == GM_DENSE) {
            // tokens contiguous: a lane's four in one store of four dwords, whatever
            // their alignment (2048 x 768 Q4_K, 512 tokens: 22.4 -> 15.9 us)
            if (a.y_ts == 1) {
                typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const int lt = 16 * i + 4 * (lane >> 4);
                    if (lt >= tn) continue;
                    const lq_f4 sc = *reinterpret_cast<const lq_f4 *>(tsc + lt);
                    const lq_f4 y0 = acc[i][0] * sc, y1 = acc[i][1] * sc;
                    if (lt + 3 < tn) {
                        if (ok0) *reinterpret_cast<f4u *>(yb0 + lt) = y0;
                        if (ok1) *reinterpret_cast<f4u *>(yb1 + lt) = y1;
                    } else {
#pragma unroll
                        for (int v = 0; v < 3; ++v) {
                            if (ok0 && lt + v < tn) yb0[lt + v] = y0[v];
                            if (ok1 && lt + v < tn) yb1[lt + v] = y1[v];
                        }
                    }
                }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int lt = 16 * i + 4 * (lane >> 4) + v;
                if (lt >= tn) continue;
                const float sc = tsc[lt];
                const uint32_t o = (uint32_t)lt * (uint32_t)a.y_ts;
                if (ok0) yb0[o] = acc[i][0][v] * sc;
                if (ok1) yb1[o] = acc[i][1][v] * sc;
            }
        }
    }
}

// NW waves per workgroup (4 or 8): 32 NW weight rows (gate_up: 16 NW gate and
// 16 NW up rows) share one staged x tile; 8 waves halve the x bytes each
// weight byte brings along (the MoE expert tiles);
// dense products of short K run 4
template <int T, int BN, int MODE, int NW = 4>
__global__ __launch_bounds__(64 * NW, 8 / NW) void gemm_tile_kernel(GemmArgs a) {
    constexpr int NI = BN / 16;            // 16-token MFMA tiles per wave
    constexpr int BB = mt_block_bytes(T);
    __shared__ __attribute__((aligned(16))) _Float16 Xs[2][BN * GM_BK];
    __shared__ __attribute__((aligned(16))) float tsc[BN];   // the output scale of each token of the tile
    __shared__ float asc[MODE == GM_MOE_GATE_UP ? BN : 1];   // gate_up with f16 output: its scale per token
    const lq_geom &g = a.g;
    // wave index made wave-uniform: row-tile addresses go to scalar registers
    // (MoE Q4_K GEMMs 162 -> 128 VGPRs; gate_up 85 -> 81 us, down 55 -> 48 us)
    const int wave = wave_id();
    const uint8_t *Wt = a.Wt;
    int64_t p0;
    int tn;
    int64_t blk;
    const float *wn = nullptr;   // the expert's row norms (gate_up with f16 output)
    if constexpr (MODE == GM_DENSE) {
        // 1-D grid, padded to a multiple of 8; workgroup id -> logical index
        // xcd * per + id / 8 walks the row blocks of one token tile per XCD
        const int id = blockIdx.x, per = gridDim.x / 8;
        const int L = (id % 8) * per + id / 8;
        const int nrb = (int)((g.rows + 32 * NW - 1) / (32 * NW));
        const int64_t ntt = (a.ntok + BN - 1) / BN;
        if (L >= nrb * ntt) return;
        blk = L % nrb;
        p0 = (int64_t)(L / nrb) * BN;
        tn = (int)(a.ntok - p0 < BN ? a.ntok - p0 : BN);
    } else {
        blk = blockIdx.x;
        const int tile = blockIdx.y;
        if (tile >= a.n_tiles[0]) return;
        Wt += (int64_t)a.tile_e[tile] * a.wt_bytes;
        if (a.wnorm) wn = a.wnorm + 2 * (int64_t)a.tile_e[tile];
        p0 = a.tile_p0[tile];
        tn = a.tile_n[tile];
    }
    const int64_t tiles = (g.rows + MT_ROWS - 1) / MT_ROWS, nsb = mt_nsb(g);
    // the wave's two row tiles: dense / down 2 NW blk + 2 wave + j; gate_up
    // gate tile NW blk + wave (j = 0) and its up tile inter / 16 + NW blk + wave
    int64_t t0, t1;
    if constexpr (MODE == GM_MOE_GATE_UP) {
        t0 = NW * blk + wave;
        t1 = a.inter / MT_ROWS + NW * blk + wave;
    } else {
        t0 = 2 * NW * blk + 2 * wave;
        t1 = t0 + 1;
    }
    const uint8_t *w0p = Wt + (t0 < tiles ? t0 : tiles - 1) * nsb * BB;
    const uint8_t *w1p = Wt + (t1 < tiles ? t1 : tiles - 1) * nsb * BB;
    if constexpr (MODE == GM_DENSE) {
        gt_main<T, BN, MODE, NW, NI>(a, Xs, tsc, asc, wn, w0p, w1p, p0, tn, t0, t1, tiles, nsb);
    } else {
        // expert tiles: one copy of the loop per count of 16-token tiles
        static_assert(NI == 4, "up to four 16-token tiles");
        const int nv = __builtin_amdgcn_readfirstlane((tn + 15) >> 4);
        if (nv == 1) gt_main<T, BN, MODE, NW, 1>(a, Xs, tsc, asc, wn, w0p, w1p, p0, tn, t0, t1, tiles, nsb);
        else if (nv == 2) gt_main<T, BN, MODE, NW, 2>(a, Xs, tsc, asc, wn, w0p, w1p, p0, tn, t0, t1, tiles, nsb);
        else if (nv == 3) gt_main<T, BN, MODE, NW, 3>(a, Xs, tsc, asc, wn, w0p, w1p, p0, tn, t0, t1, tiles, nsb);
        else gt_main<T, BN, MODE, NW, 4>(a, Xs, tsc, asc, wn, w0p, w1p, p0, tn, t0, t1, tiles, nsb);
    }
}

// ---------------------------------------------------------------- host side

// f16 activation rows are padded with zeros to a multiple of 256 values (the
// tile form's block; a multiple of the row-plane kernel's 128-value step)
static int64_t gemm_ldh(const lq_geom &g) { return 256 * ((g.cols + 255) / 256); }

// f16 rows of x (padded to a multiple of 16 rows) and their scales
static int64_t gemm_x_bytes(const lq_geom &g, int64_t ntok) {
    return lq_align256((ntok + 15) / 16 * 16 * gemm_ldh(g) * 2) + ntok * 4;
}

// Whether a dense product on the tile form runs gemm_tile_kernel (128 x 128 tiles,
// two workgroups per CU) instead of gemm_dense_kernel (256 x 128, one, K divided).
// Where K is short, the dense kernel's first loads, its larger stores and the sum
// of its parts take longer than the blocks: the smaller tiles then win as long as
// their workgroups come to about one per CU. Both times from fits over whole
// calls (gemm_dense_us; the tile kernel's: 0.95 to 1.05 of the measured in 98 of
// 100 calls). 2048 x 768, 512 tokens: Q4_K 20.5 us dense, 16.5 here, Q6_K 21.5,
// 17.1; 1024 x 1024, 700 tokens Q4_K 24.1, 19.4; 11008 x 2048, 256 tokens 34.8,
// 30.7; but 4096 x 4096, 128 tokens 26.9, 50.3 and 11008 x 2048, 300 tokens 34.5,
// 39.0. Of 5160 calls up to 32000 rows the choice is within 4 % of the faster
// kernel in all but 80, at worst 13 % off (11 % where it stays with the dense one).
// Up to 32 tokens the dense kernel computes a quarter of what this one does, except
// from 256 of its tiles on, where it computes whole ones: of 882 calls of 66000 to
// 256000 rows and up to 128 tokens, 25 are more than 4 % off the faster kernel
// (128256 x 1536 Q8_0, 32 tokens 57.0 us dense, 55.5 here; 202048 x 768, 1 token
// 53.7, 45.4).
// (The tile kernel's offsets into Y have 32 bits.)
// *split_bytes: what the parts of K of the dense kernel take, 0 with the tile kernel.
static bool gemm_takes_tile_kernel(const lq_geom &g, int64_t ntok, int64_t *split_bytes) {
    const double dense = gemm_dense_us(g, ntok, split_bytes);
    const bool rounds = (g.rows + 255) / 256 * ((ntok + 127) / 128) >= 256;
    if (mt_matrix_bytes(g) == 0 || (ntok <= 32 && !rounds) || g.rows >= ((int64_t)1 << 25)) return false;
    const int64_t nwg = ((g.rows + GM_BM - 1) / GM_BM) * ((ntok + GM_BN - 1) / GM_BN), left = nwg % 512;
    // us per block: a full round of 512 workgroups, one of up to 256, of more
    const double full = g.type == LQ_Q4_K ? 3.75 : g.type == LQ_Q6_K ? 4.15 : 3.9;
    const double half = g.type == LQ_Q4_K ? 2.6 : g.type == LQ_Q6_K ? 2.7 : 2.4;
    const double most = g.type == LQ_Q4_K ? 3.55 : g.type == LQ_Q6_K ? 3.85 : 3.3;
    const double per_block = full * (double)(nwg / 512) + (left == 0 ? 0.0 : left <= 256 ? half : most);
    const double us = 6.0 + (double)(ntok < GM_BN ? ntok : GM_BN) / 64.0 + per_block * (double)mt_nsb(g) +
                      1.6e-7 * (double)(g.rows * ntok);   // Y a little slower than there
    // (a launch has fewer than 2^32 threads)
    if (nwg >= ((int64_t)1 << 24) || 1.02 * us + 0.25 >= dense) return false;
    *split_bytes = 0;
    return true;
}

int64_t gemm_workspace_bytes(const lq_geom &g, int64_t ntok) {
    const int64_t x = gemm_x_bytes(g, ntok);
    int64_t split = 0;
    if (ntok > 0) gemm_takes_tile_kernel(g, ntok, &split);
    return split ? lq_align256(x) + split : x;
}

int launch_x_to_f16(const float *X, int64_t ldx, int64_t cols, const int32_t *rows_map, int k, int64_t ntok,
                    _Float16 *Xh, int64_t ldh, float *inv, hipStream_t s, float *nrm2) {
    if (ntok <= 0) return LOCALAI_OK;
    if (cols % 8 || ldh % 8 || ldh < cols) return fail(LOCALAI_EARG, "f16 rows: cols % 8 != 0");
    const int vec = (uintptr_t)X % 16 == 0 && ldx % 4 == 0;
    const int per = (int)((ldh / 8 + 63) / 64);   // 8-value groups per lane
    // (a launch has fewer than 2^32 threads)
    if (per > 4 && per <= 32 && !nrm2 && ntok < ((int64_t)1 << 24)) {
        auto gw = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((unsigned)ntok), dim3(256), 0, s, X, ldx, (int)cols, rows_map, k, Xh,
                               (int)ldh, inv, vec);
        };
        if (per <= 8) gw(x_to_f16_wide_kernel<2>);
        else if (per <= 16) gw(x_to_f16_wide_kernel<4>);
        else if (per <= 24) gw(x_to_f16_wide_kernel<6>);
        else gw(x_to_f16_wide_kernel<8>);
        LQ_HIP(hipGetLastError());
        return LOCALAI_OK;
    }
    // one token per wave; one-wave workgroups below 1024 tokens, so that 512
    // tokens reach every CU (four-wave workgroups left half of them idle)
    const int wpg = ntok < 1024 ? 1 : 4;
    const dim3 grid((unsigned)((ntok + wpg - 1) / wpg));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(64 * wpg), 0, s, X, ldx, (int)cols, rows_map, k, ntok, Xh, (int)ldh, inv,
                           vec, nrm2);
    };
    if (per <= 1)
        go(x_to_f16_kernel<1>);
    else if (per <= 2)
        go(x_to_f16_kernel<2>);
    else if (per <= 4)
        go(x_to_f16_kernel<4>);
    else if (per <= 8)
        go(x_to_f16_kernel<8>);
    else
        go(x_to_f16_kernel<0>);
    LQ_HIP(hipGetLastError());
    return LOCALAI_OK;
}

template <int MODE, int BN>
static int launch_gemm_t(const GemmArgs &a, dim3 grid, hipStream_t s) {
    switch (a.g.type) {
#define LQ_GM(TT) case TT: hipLaunchKernelGGL((gemm_kernel<TT, BN, MODE>), grid, dim3(256), 0, s, a); break;
        LQ_GM(LQ_Q4_K) LQ_GM(LQ_Q5_K) LQ_GM(LQ_Q6_K) LQ_GM(LQ_Q8_0) LQ_GM(LQ_Q4_0)
#undef LQ_GM
        default: return fail(LOCALAI_ETYPE, "matmul: unsupported GGML type");
    }
    LQ_HIP(hipGetLastError());
    return LOCALAI_OK;
}

template <int MODE, int BN, int NW = 4>
static int launch_gemm_tile_t(const GemmArgs &a, dim3 grid, hipStream_t s) {
    switch (a.g.type) {
#define LQ_GT(TT) case TT: hipLaunchKernelGGL((gemm_tile_kernel<TT, BN, MODE, NW>), grid, dim3(64 * NW), 0, s, a); break;
        LQ_GT(LQ_Q4_K) LQ_GT(LQ_Q6_K) LQ_GT(LQ_Q8_0)
#undef LQ_GT
        default: return fail(LOCALAI_ETYPE, "matmul: no tile form for this GGML type");
    }
    LQ_HIP(hipGetLastError());
    return LOCALAI_OK;
}

int launch_gemm(const lq_geom &g, const uint8_t *W, const uint8_t *Wt, const float *X, int64_t ntok, float *Y,
                int64_t y_ts, int64_t y_rs, void *ws, int64_t ws_bytes, hipStream_t s) {
    if (ntok <= 0) return LOCALAI_OK;
    if (ws_bytes < gemm_x_bytes(g, ntok)) return fail(LOCALAI_EARG, "matmul: workspace too small");
    const int64_t ldh = gemm_ldh(g);
    _Float16 *Xh = (_Float16 *)ws;
    float *inv = (float *)((uint8_t *)ws + lq_align256((ntok + 15) / 16 * 16 * ldh * 2));
    GemmArgs a{};
    a.g = g; a.W = W; a.Xh = Xh; a.ldh = (int)ldh; a.inv = inv; a.ntok = ntok; a.Y = Y; a.y_ts = y_ts; a.y_rs = y_rs;
    a.Wt = Wt;
    // row planes of a type with a tile form (a handle made without one,
    // mfma_matvec_enabled), or with rows past the dense kernel's 32-bit offsets
    // into 16 of them
    const bool planes = !Wt && (mt_matrix_bytes(g) > 0 || g.cols >= ((int64_t)1 << 29));
    const int64_t nwg = ((g.rows + GM_BM - 1) / GM_BM) * ((ntok + GM_BN - 1) / GM_BN);
    if (!Wt && !W) return fail(LOCALAI_ESTATE, "matmul: handle without weights");
    // tokens per launch: the dense kernel's 32-bit byte offsets into a tile's x rows
    const int64_t most = planes ? ntok : (((int64_t)1 << 32) - 1) / (2 * ldh);
    if (most < 1 || (planes && nwg > ((int64_t)1 << 30))) return fail(LOCALAI_EARG, "matmul: problem too large");
    if (int st = launch_x_to_f16(X, g.cols, g.cols, nullptr, 1, ntok, Xh, ldh, inv, s)) return st;
    const dim3 grid((unsigned)((nwg + 7) / 8 * 8));
    if (planes) return launch_gemm_t<GM_DENSE, GM_BN>(a, grid, s);
    int64_t split;
    if (Wt && gemm_takes_tile_kernel(g, ntok, &split)) return launch_gemm_tile_t<GM_DENSE, GM_BN>(a, grid, s);
    const int64_t xb = lq_align256(gemm_x_bytes(g, ntok));
    for (int64_t t0 = 0; t0 < ntok;) {
        // (a tile has 128 tokens: all in one launch below 16.7 million columns)
        a.ntok = most < GM_BN && ntok - t0 > most ? most : ntok - t0;
        a.Xh = Xh + t0 * ldh;
        a.inv = inv + t0;
        a.Y = Y + t0 * y_ts;
        if (int st = launch_gemm_dense(a, (uint8_t *)ws + xb, ws_bytes > xb ? ws_bytes - xb : 0, s)) return st;
        t0 += a.ntok;
    }
    return LOCALAI_OK;
}

int moe_gemm_tile() { return GM_MOE_BN; }

int launch_moe_gemm(const lq_geom &g, const uint8_t *Wall, const uint8_t *Wt_all, int64_t wt_bytes, bool gate_up,
                    const _Float16 *Xh, int64_t ldh, const float *inv, const int32_t *rows_map, int rows_k,
                    float *Y, int64_t y_ts, int64_t inter, const int32_t *tile_e, const int32_t *tile_p0,
                    const int32_t *tile_n, const int32_t *n_tiles, int max_tiles, hipStream_t s,
                    const MoeF16Out *f16_out) {
    GemmArgs a{};
    a.g = g; a.W = Wall; a.Xh = Xh; a.ldh = (int)ldh; a.inv = inv; a.Y = Y; a.y_ts = y_ts; a.y_rs = 1;
    a.rows_map = rows_map; a.rows_k = rows_k;
    a.tile_e = tile_e; a.tile_p0 = tile_p0; a.tile_n = tile_n; a.n_tiles = n_tiles; a.inter = inter;
    a.Wt = Wt_all; a.wt_bytes = wt_bytes;
    if (max_tiles <= 0) return LOCALAI_OK;
    if (max_tiles > 65535) return fail(LOCALAI_EARG, "moe: too many token tiles");
    if (f16_out) {
        if (!gate_up || !Wt_all || inter % MT_ROWS || !f16_out->wnorm || !f16_out->xnorm2)
            return fail(LOCALAI_EARG, "moe: f16 gate_up output needs the tile form, inter % 16 == 0 and the norms");
        a.Yh = f16_out->Yh; a.ldy = f16_out->ldy; a.inv_out = f16_out->inv_out;
        a.wnorm = f16_out->wnorm; a.xnorm2 = f16_out->xnorm2;
    }
    if (Wt_all && (!gate_up || inter % MT_ROWS == 0)) {
        constexpr int NW = GM_MOE_NW;
        if (gate_up)
            return launch_gemm_tile_t<GM_MOE_GATE_UP, GM_MOE_BN, NW>(
                a, dim3((unsigned)((inter + 16 * NW - 1) / (16 * NW)), (unsigned)max_tiles), s);
        return launch_gemm_tile_t<GM_MOE_DOWN, GM_MOE_BN, NW>(
            a, dim3((unsigned)((g.rows + 32 * NW - 1) / (32 * NW)), (unsigned)max_tiles), s);
    }
    if (!Wall) return fail(LOCALAI_ESTATE, "moe: expert handle without row planes");
    if (gate_up) {
        dim3 grid((unsigned)((inter + GM_BM / 2 - 1) / (GM_BM / 2)), (unsigned)max_tiles);
        return launch_gemm_t<GM_MOE_GATE_UP, GM_MOE_BN>(a, grid, s);
    }
    dim3 grid((unsigned)((g.rows + GM_BM - 1) / GM_BM), (unsigned)max_tiles);
    return launch_gemm_t<GM_MOE_DOWN, GM_MOE_BN>(a, grid, s);
}

}  // namespace lq
