// Dense prefill product on f16 MFMA: the kernel of all dense matmuls but those of
// short K and of handles without the tile form (gemm.hip, which also has the
// contract and the arithmetic).
//
// Workgroup: 8 waves x 2 row tiles (256 weight rows) x 128 tokens (16 NV of
// them computed), over a range of 256-value blocks of K. Each wave decodes its
// own weights from global memory into MFMA operands in registers; x goes
// through an LDS ring of four 128-value steps. One workgroup per CU.
//
// What bounds such a loop is not one resource but their sum when nothing
// overlaps: a 32-value slice of a wave is 2 NV MFMAs (16 clocks each), 28 to
// 60 VALU of decode and NV LDS reads, and run one after the other they took
// 4.8 us per 256 x 128 x 256 block against 1.9 us of MFMAs. Simple VALU issues
// under a running MFMA (16 MFMAs alone 108 to 113 ns, with 32 v_and, v_perm or f32
// multiply-adds 115 to 121 ns), so
// every slice's MFMAs are interleaved with the reads and the decode of the
// next slice, across the workgroup barrier too:
//   step s (128 values), slices kk = 0 .. 3: MFMAs of slice kk, beside them
//   the LDS reads and the decode of slice kk + 1 (of step s + 1 for kk = 3);
//   before slice 3's MFMAs: wait for the own part of x(s + 1) and for the
//   weights of step s + 1, then the barrier.
// The loads are asm and the kernel counts its own waits: x is requested two to
// three steps before it is read, weights three. x(s + 3) is requested after the
// barrier of step s into the slot of x(s - 1), whose last reads every wave
// consumed before it arrived there.
#include <type_traits>

#include "gemm_core.h"

namespace lq {

constexpr int GD_NW = 8;               // waves per workgroup
constexpr int GD_BM = 32 * GD_NW;      // weight rows per workgroup
constexpr int GD_BN = 128;             // tokens per workgroup
constexpr int GD_RING = 4;             // x steps in LDS
constexpr int GD_VALU = 32;            // VALU scheduled beside a slice's MFMAs, per half
constexpr int GD_SLOT = GD_BN * GM_BK * 2;   // bytes of one x step

// Q5_K and Q4_0 handles hold row planes (qformat.h), not the tile form. Any
// order of K serves a product as long as both operands have it, so lane (row n =
// lane % 16, c = lane / 16) takes one 16-byte quant piece of its row per step as
// its K values: piece c % 2 of unit 2 HALF + c / 2 (64 values) of the block,
// 16 low nibbles and 16 high ones, the operands of slices 0, 1 and 2, 3. The
// matching 8-value chunk of x is gd_chunk. Q5_K decodes in f32 (its minimum has
// 17 bits: a packed f16 decode would round twice), about 4.5 VALU per MFMA:
// 14336 x 4096, 128 tokens 43 us against Q4_K's 33; through an LDS tile of f32
// decoded weights, 112 workgroups, it took 192.
template <int T> constexpr bool gd_planes() { return T == LQ_Q5_K || T == LQ_Q4_0; }

// 256-value blocks of a row (x rows are padded with zeros to whole blocks)
__host__ __device__ inline int64_t gd_blocks(const lq_geom &g) { return (g.cols + 255) / 256; }

// the 8-value chunk (of a step's 16) that lane group q multiplies in slice KK
template <int T, int KK>
__device__ __forceinline__ int gd_chunk(int q) {
    if constexpr (T == LQ_Q5_K) return 8 * (q >> 1) + 4 * (KK >> 1) + 2 * (q & 1) + (KK & 1);
    else if constexpr (T == LQ_Q4_0) return 8 * (q >> 1) + 4 * (q & 1) + 2 * (KK >> 1) + (KK & 1);
    else return 4 * KK + q;
}

// One row tile's weights of one step (128 values), and of one 256-value block
template <int T> struct GdStep { mt_i4 q; };
template <> struct GdStep<LQ_Q8_0> { mt_i4 q, p; };
template <> struct GdStep<LQ_Q4_0> { mt_i4 q; int d; };
template <int T> struct GdBlock { mt_i4 h; };
template <> struct GdBlock<LQ_Q6_K> { mt_i4 h, sc; int d; };
template <> struct GdBlock<LQ_Q5_K> { mt_i4 h, qh; };
template <> struct GdBlock<LQ_Q4_0> {};

// loads per wave (two row tiles): each step's, each block's
template <int T> constexpr int gd_step_loads() { return T == LQ_Q8_0 || T == LQ_Q4_0 ? 4 : 2; }
template <int T> constexpr int gd_block_loads() {
    return T == LQ_Q6_K ? 6 : T == LQ_Q5_K ? 4 : T == LQ_Q4_0 ? 0 : 2;
}

__device__ __forceinline__ void cu_load_u16(int &v, const void *base, uint32_t off) {
    asm volatile("global_load_ushort %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}

template <int T, int HALF>
__device__ __forceinline__ void gd_load_step(GdStep<T> &w, const uint8_t *blk, uint32_t l16) {
    if constexpr (T == LQ_Q8_0) {
        cu_load(w.q, blk + 2048 * HALF, l16);
        cu_load(w.p, blk + 2048 * HALF + 1024, l16);
    } else {
        cu_load(w.q, blk + 1024 * HALF, l16);
    }
}
// r16: 16 (lane % 16), the lane's row in the 16-byte-per-row parts
template <int T>
__device__ __forceinline__ void gd_load_block(GdBlock<T> &b, const uint8_t *blk, uint32_t l16, uint32_t r16) {
    if constexpr (T == LQ_Q4_K) {
        cu_load(b.h, blk + 2048, r16);
    } else if constexpr (T == LQ_Q6_K) {
        cu_load(b.h, blk + 2048, l16);
        cu_load(b.sc, blk + 3072, r16);
        cu_load_u16(b.d, blk + 3328, r16 >> 3);
    } else {
        cu_load(b.h, blk + 4096, r16);
    }
}

// vmcnt wait that names the registers whose loads it completes
template <int N, int T>
__device__ __forceinline__ void gd_wait_step(GdStep<T> (&w)[2]) {
    if constexpr (T == LQ_Q8_0)
        asm volatile("s_waitcnt vmcnt(%4)" : "+v"(w[0].q), "+v"(w[0].p), "+v"(w[1].q), "+v"(w[1].p) : "n"(N) : "memory");
    else if constexpr (T == LQ_Q4_0)
        asm volatile("s_waitcnt vmcnt(%4)" : "+v"(w[0].q), "+v"(w[0].d), "+v"(w[1].q), "+v"(w[1].d) : "n"(N) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(%2)" : "+v"(w[0].q), "+v"(w[1].q) : "n"(N) : "memory");
}
template <int N, int T>
__device__ __forceinline__ void gd_wait_block(GdBlock<T> (&b)[2]) {
    if constexpr (T == LQ_Q6_K)
        asm volatile("s_waitcnt vmcnt(%6)"
                     : "+v"(b[0].h), "+v"(b[0].sc), "+v"(b[0].d), "+v"(b[1].h), "+v"(b[1].sc), "+v"(b[1].d)
                     : "n"(N) : "memory");
    else if constexpr (T == LQ_Q5_K)
        asm volatile("s_waitcnt vmcnt(%4)" : "+v"(b[0].h), "+v"(b[0].qh), "+v"(b[1].h), "+v"(b[1].qh) : "n"(N) : "memory");
    else if constexpr (T != LQ_Q4_0)
        asm volatile("s_waitcnt vmcnt(%2)" : "+v"(b[0].h), "+v"(b[1].h) : "n"(N) : "memory");
}

// Q4_K scale pair {d * sc, dmin * mn} of sub-block 4 HALF + KK of the lane's row
// (packed f16, each rounded once: gt_q4k_pair's arithmetic, without its trip
// through another lane)
template <int HALF, int KK>
__device__ __forceinline__ uint32_t gd_q4k_pair(const uint4 &hd) {
    const uint32_t s0 = hd.y, s4 = hd.z, s8 = hd.w;
    uint32_t sm;
    if constexpr (HALF == 0) {
        sm = __builtin_amdgcn_perm(s4, s0, 0x0C000C00u | KK | ((4 + KK) << 16)) & 0x003F003Fu;
    } else {
        const uint32_t lo = KK == 0 ? s8 : s8 >> (8 * KK);
        const uint32_t up = __builtin_amdgcn_perm(s4, s0, 0x0C000C00u | KK | ((4 + KK) << 16));
        sm = (lo & 0xFu) | ((lo & 0xF0u) << 12) | ((up & 0x00C000C0u) >> 2);
    }
    const lq_h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const lq_h2 scmn = __builtin_bit_cast(lq_h2, sm | 0x64006400u) - k1024;
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(lq_h2, hd.x) * scmn);
}

__device__ __forceinline__ uint4 gd_u4(const mt_i4 &v) { return __builtin_bit_cast(uint4, v); }

template <int T>
__device__ __forceinline__ GtRaw<T> gd_raw(const GdStep<T> &w, const GdBlock<T> &b) {
    GtRaw<T> r;
    if constexpr (T == LQ_Q4_K) {
        r.qs = gd_u4(w.q);
        r.hd = gd_u4(b.h);
    } else if constexpr (T == LQ_Q6_K) {
        r.ql = gd_u4(w.q);
        r.qh = gd_u4(b.h);
        r.sc = gd_u4(b.sc);
        r.d = (uint32_t)b.d;
    } else {
        r.p0 = gd_u4(w.q);
        r.p1 = gd_u4(w.p);
        r.dd = gd_u4(b.h);
    }
    return r;
}

// Q5_K: f32 scale and minimum {d * sc, dmin * mn} (exact) of the lane's sub-block
// 4 HALF + 2 (q / 2) + NIB
template <int HALF, int NIB>
__device__ __forceinline__ void gd_q5k_scale(const mt_i4 &h, int q, float &a, float &b) {
    const int o = 16 * (q >> 1) + 8 * NIB;
    const uint32_t s0 = (uint32_t)h[1], s4 = (uint32_t)h[2], s8 = (uint32_t)h[3];
    uint32_t sc, mn;
    if constexpr (HALF == 0) {
        sc = __builtin_amdgcn_ubfe(s0, o, 6);
        mn = __builtin_amdgcn_ubfe(s4, o, 6);
    } else {
        sc = __builtin_amdgcn_ubfe(s8, o, 4) | (__builtin_amdgcn_ubfe(s0, o + 6, 2) << 4);
        mn = __builtin_amdgcn_ubfe(s8, o + 4, 4) | (__builtin_amdgcn_ubfe(s4, o + 6, 2) << 4);
    }
    a = f16_to_f32((uint32_t)h[0]) * (float)sc;
    b = f16_to_f32((uint32_t)h[0] >> 16) * (float)mn;
}
// Q5_K operand of slice KK: q = nibble | high bit << 4, a value a q - b in one
// f32 fused multiply-add (exact products, rounded as the row decoders round it),
// then rounded once to f16
template <int HALF, int KK>
__device__ __forceinline__ lq_h8 gd_q5k_b(const mt_i4 &qs, const mt_i4 &qh, int q, float a, float b) {
    constexpr int nib = KK >> 1, w0 = 2 * (KK & 1);
    const int bit = 2 * (q >> 1) + 4 * HALF + nib;
    // two f32 to f16, rounded to nearest even, the f32 values opaque: seen
    // together, the compiler fused half of the multiply-adds with their
    // conversion into v_fma_mix{lo,hi}_f16, which take twice as long and do not
    // hide under the MFMAs (14336 x 4096, 1024 tokens: 161.9 us against 156.0)
    auto pack = [](float x, float y) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        asm("" : "+v"(x), "+v"(y));
        return (int)__builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, lq_h2));
    };
    mt_i4 o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t lo = ((uint32_t)qs[w0 + i] >> (4 * nib)) & 0x0F0F0F0Fu;
        const uint32_t hi = ((uint32_t)qh[w0 + i] >> bit) & 0x01010101u;
        const uint32_t v = lo | (hi << 4);
        const float f[4] = {__builtin_fmaf(a, ubyte0(v), -b), __builtin_fmaf(a, ubyte1(v), -b),
                            __builtin_fmaf(a, ubyte2(v), -b), __builtin_fmaf(a, ubyte3(v), -b)};
        o[2 * i] = pack(f[0], f[1]);
        o[2 * i + 1] = pack(f[2], f[3]);
    }
    return __builtin_bit_cast(lq_h8, o);
}
// Q4_0 operand of slice KK: q - 8 exactly, times d rounded once
template <int KK>
__device__ __forceinline__ lq_h8 gd_q40_b(const mt_i4 &qs, lq_h2 d2) {
    constexpr int nib = KK >> 1, w0 = 2 * (KK & 1);
    const lq_h2 k8 = {(_Float16)8.0f, (_Float16)8.0f};
    uint4 o;
    auto pair = [&](lq_h2 v) { return __builtin_bit_cast(uint32_t, (v - k8) * d2); };
    const uint32_t a = ((uint32_t)qs[w0] >> (4 * nib)) & 0x0F0F0F0Fu, b = ((uint32_t)qs[w0 + 1] >> (4 * nib)) & 0x0F0F0F0Fu;
    o.x = pair(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 512.0f, false));
    o.y = pair(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 512.0f, true));
    o.z = pair(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 512.0f, false));
    o.w = pair(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 512.0f, true));
    return __builtin_bit_cast(lq_h8, o);
}

// 1 KB from base + off (per lane) into LDS at the wave-uniform byte address lds
__device__ __forceinline__ void gd_dma(const void *base, uint32_t off, uint32_t lds) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(off), "s"(base), "s"(lds)
                 : "memory");
}

// Dense arguments: GemmArgs plus the division of the work. Output tiles (256
// rows x 128 tokens, token tiles fastest) 0 .. full - 1 (a multiple of 256) are
// computed whole, one per workgroup and round; the rest .. are cut `splits` ways
// in K, part i covering blocks [i * blocks, ...). With splits > 1 the parts go to
// P, part i of rest tile k at P + (i * rest + k) * GD_PART, in Y's order (rows or
// tokens fastest) and not yet scaled, and gemm_split_sum_kernel adds them.
struct DenseArgs {
    GemmArgs a;
    int full, rest, splits, blocks;
    float *P;
};
constexpr int64_t GD_PART = GD_BM * GD_BN;

// Order of the output tiles: groups of GD_TG token tiles, in a group the token
// tiles of a row block side by side, so that the 32 tiles an XCD computes at a
// time (4 x 8) share both x and weights in its L2. All token tiles of a row block
// side by side, groups of eight, of four: 14336 x 4096 Q4_K, 2048 tokens 254, 245,
// 247 us; 28000 x 2048, 1500 tokens 211, 207, 204 us.
constexpr int GD_TG = 4;
__device__ __forceinline__ void gd_tile(int tile, int ntt, int nrb, int &rb, int &tt) {
    const int grp = tile / (GD_TG * nrb), r = tile - grp * GD_TG * nrb;
    const int gs = ntt - GD_TG * grp < GD_TG ? ntt - GD_TG * grp : GD_TG;
    rb = r / gs;
    tt = GD_TG * grp + r % gs;
}

template <int T, int NV>
struct GdMain {
    static constexpr int XN = NV / 2;            // x copies per wave and step
    static constexpr int WL = gd_step_loads<T>(), HL = gd_block_loads<T>();
    static constexpr int BB = gd_planes<T>() ? 0 : mt_block_bytes(T);

    int lane, wave, nb;
    uint8_t *ring;
    uint32_t ring0, l16, r16;
    const uint8_t *w0p, *w1p;      // the two row tiles at the split's first block
    // row planes: first row of each row tile in each plane, the lane's row in
    // the tile, units of a row, the split's first block
    const uint8_t *pl[2][3];
    int nu, first;
    uint32_t dr[2], pitch[3];
    float sa[2], sm[2];            // Q5_K: scale and minimum of the slices' sub-block
    const uint8_t *xb;             // x row p0 at the split's first value
    uint32_t xoff[XN];
    lq_f4 acc[NV][2];
    GdStep<T> w[4][2];
    GdBlock<T> hd[2][2];
    lq_h8 av[2][NV / 2], bo[2][2];

    template <int I0 = 0, int I1 = XN>
    __device__ __forceinline__ void dma(int slot, int s) {
        const int sc = __builtin_amdgcn_readfirstlane(s < 2 * nb ? s : 2 * nb - 1);
        const uint8_t *base = xb + (int64_t)sc * (GM_BK * 2);
#pragma unroll
        for (int i = I0; i < I1; ++i)
            gd_dma(base, xoff[i],
                   __builtin_amdgcn_readfirstlane(ring0 + (uint32_t)(slot * GD_SLOT + (GD_NW * i + wave) * 1024)));
    }
    template <int HALF>
    __device__ __forceinline__ void load_step(GdStep<T> (&d)[2], int b) {
        if constexpr (gd_planes<T>()) {
            // the step's first unit (its last valid one past the row's end, whose
            // weights are then multiplied by a zero scale), its 64-unit chunk
            int u = 4 * (first + (b < nb ? b : nb - 1)) + 2 * HALF;
            if (T == LQ_Q4_0) u = u < nu ? u : nu - 1;
            const int c0 = u & ~63, C = nu - c0 < 64 ? nu - c0 : 64;
            const int c = lane >> 4;
            int du = c >> 1;
            if (T == LQ_Q4_0) du = u + du < nu ? du : 0;
            const int off = 16 * (du + (c & 1) * C);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                cu_load(d[j].q, pl[j][0] + 16 * (c0 + (int64_t)u), dr[j] * pitch[0] + (uint32_t)off);
                if constexpr (T == LQ_Q4_0) cu_load(d[j].d, pl[j][1] + 4 * (int64_t)u, dr[j] * pitch[1] + (uint32_t)(4 * du));
            }
            return;
        } else {
            const int64_t o = (int64_t)(b < nb ? b : nb - 1) * BB;
            gd_load_step<T, HALF>(d[0], w0p + o, l16);
            gd_load_step<T, HALF>(d[1], w1p + o, l16);
        }
    }
    __device__ __forceinline__ void load_block(GdBlock<T> (&d)[2], int b) {
        if constexpr (T == LQ_Q4_0) return;
        else if constexpr (T == LQ_Q5_K) {
            const int sb = first + (b < nb ? b : nb - 1), s0 = sb & ~15, nsb = nu >> 2;
            const int off = 16 * ((lane >> 4) & 1) * (nsb - s0 < 16 ? nsb - s0 : 16);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                cu_load(d[j].qh, pl[j][1] + 16 * (s0 + (int64_t)sb), dr[j] * pitch[1] + (uint32_t)off);
                cu_load(d[j].h, pl[j][2] + 16 * (int64_t)sb, dr[j] * pitch[2]);
            }
        } else {
            const int64_t o = (int64_t)(b < nb ? b : nb - 1) * BB;
            gd_load_block<T>(d[0], w0p + o, l16, r16);
            gd_load_block<T>(d[1], w1p + o, l16, r16);
        }
    }
    // x operands of slice KK of a slot: token tiles PART * NV / 2 .. into av[PART]
    template <int SLOT, int KK, int PART>
    __device__ __forceinline__ void read_x() {
        const int fr = lane & 15, q = lane >> 4;
        const uint8_t *xs = ring + SLOT * GD_SLOT + PART * (NV / 2) * 16 * (GM_BK * 2);
#pragma unroll
        for (int i = 0; i < NV / 2; ++i)
            av[PART][i] = *reinterpret_cast<const lq_h8 *>(xs + (16 * i + fr) * (GM_BK * 2) + 16 * (gd_chunk<T, KK>(q) ^ fr));
    }
    // operands of slice KK of half HALF from weight set SET and block header PAR;
    // b: the slice's block
    template <int SET, int PAR, int HALF, int KK, int DST>
    __device__ __forceinline__ void decode(int b) {
        const int q = lane >> 4;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (T == LQ_Q5_K) {
                if constexpr ((KK & 1) == 0) gd_q5k_scale<HALF, (KK >> 1)>(hd[PAR][j].h, q, sa[j], sm[j]);
                bo[DST][j] = gd_q5k_b<HALF, KK>(w[SET][j].q, hd[PAR][j].qh, q, sa[j], sm[j]);
            } else if constexpr (T == LQ_Q4_0) {
                // the scale of the lane's 32-value block; zero past the row's end
                const uint32_t dd = ((uint32_t)w[SET][j].d >> (16 * (q & 1))) & 0xFFFFu;
                const uint32_t d = 4 * (first + b) + 2 * HALF + (q >> 1) < nu ? dd * 0x10001u : 0u;
                bo[DST][j] = gd_q40_b<KK>(w[SET][j].q, __builtin_bit_cast(lq_h2, d));
            } else {
                const GtRaw<T> r = gd_raw<T>(w[SET][j], hd[PAR][j]);
                uint32_t p = 0;
                if constexpr (T == LQ_Q4_K) p = gd_q4k_pair<HALF, KK>(r.hd);
                bo[DST][j] = gt_b<T, HALF, KK>(r, q, p);
            }
        }
    }
    // MFMAs of token tiles PART * NV / 2 .. with the operands bo[SRC]; beside
    // each pair one LDS read and a share of the VALU that stands before them
    template <int SRC, int PART>
    __device__ __forceinline__ void mfmas() {
#pragma unroll
        for (int i = 0; i < NV / 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                lq_f4 &c = acc[PART * (NV / 2) + i][j];
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(bo[SRC][j], av[PART][i], c, 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < NV / 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, GD_VALU / NV, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, GD_VALU / NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // slice KK of slot S (operands bo[KK % 2], first half of x in av[0]), beside
    // it the second half of its x and the next slice's operands (of block bn)
    template <int S, int KK, int SN, int KN, int PN, int HN>
    __device__ __forceinline__ void slice(int bn) {
        read_x<S, KK, 1>();
        if constexpr (SN >= 0) decode<SN, PN, HN, KN, (KK + 1) & 1>(bn);
        mfmas<KK & 1, 0>();
        if constexpr (SN >= 0) read_x<SN, KN, 0>();
        mfmas<KK & 1, 1>();
    }
    // step s = 2 b + HALF of block b (b % 2 == PAR). TAIL 1..4: the first to
    // fourth step of the last one or two blocks, which request no weights
    template <int PAR, int HALF, int TAIL>
    __device__ __forceinline__ void step(int b) {
        constexpr int S = 2 * PAR + HALF, SN = (S + 1) & 3, HN = HALF ^ 1, PN = HALF ? PAR ^ 1 : PAR;
        // requests spread over the slices, the weights' registers being those
        // that the previous step decoded: second half of x(s + 2)
        if constexpr (TAIL <= 2) dma<XN / 2, XN>((S + 2) & 3, 2 * b + HALF + 2);
        slice<S, 0, S, 1, PAR, HALF>(b);
        if constexpr (TAIL <= 1) {
            // the next block's header (half 0), the weights of step s + 3
            if constexpr (HALF == 0) load_block(hd[PAR ^ 1], b + 1);
            load_step<HN>(w[(S + 3) & 3], b + 1 + HALF);
        }
        slice<S, 1, S, 2, PAR, HALF>(b);
        slice<S, 2, S, 3, PAR, HALF>(b);
        if constexpr (TAIL < 4) {
            // requested, in order: in step s - 1 the second half of x(s + 1),
            // the next block's header (if its half is 0), the weights of step
            // s + 2, the first half of x(s + 2); in step s so far the second
            // half of x(s + 2), the header (half 0), the weights of step s + 3.
            // Complete now: x(s + 1), that step's header and its weights (a
            // step older); the tail waits for what was still requested
            constexpr int N = TAIL <= 1 ? 2 * WL + XN + (HALF == 0 ? HL : 0) : TAIL == 2 ? WL + XN : 0;
            gd_wait_step<N, T>(w[SN]);
            if constexpr (HALF == 1) gd_wait_block<N, T>(hd[PN]);
            cu_barrier();
            if constexpr (TAIL <= 1) dma<0, XN / 2>((S + 3) & 3, 2 * b + HALF + 3);
            __builtin_amdgcn_sched_barrier(0);
        }
        slice<S, 3, TAIL < 4 ? SN : -1, 0, PN, HN>(b + HALF);
    }
    // the first requests of a tile (setup done): what step 0 does not request
    __device__ __forceinline__ void issue() {
        dma(0, 0);
        load_block(hd[0], 0);
        load_step<0>(w[0], 0);
        load_step<1>(w[1], 0);
        dma(1, 1);
        load_step<0>(w[2], 1);
        dma<0, XN / 2>(2, 2);
    }
    // the lane index as a fresh value: what is derived from it is computed where
    // it is needed, not kept in registers over the loop of tiles
    __device__ __forceinline__ void fresh_lane() { asm volatile("" : "+v"(lane)); }
    __device__ __forceinline__ void run() {
        fresh_lane();
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = lq_f4{0.0f, 0.0f, 0.0f, 0.0f};
        // everything requested so far has landed before the loop: the compiler
        // may copy loop-carried registers on entry
        gd_wait_step<0, T>(w[0]);
        gd_wait_step<0, T>(w[1]);
        gd_wait_step<0, T>(w[2]);
        gd_wait_block<0, T>(hd[0]);
        __syncthreads();
        read_x<0, 0, 0>();
        decode<0, 0, 0, 0, 0>(0);
        int b = 0;
        for (; b + 2 < nb; b += 2) {
            step<0, 0, 0>(b);
            step<0, 1, 0>(b);
            step<1, 0, 0>(b + 1);
            step<1, 1, 0>(b + 1);
        }
        step<0, 0, 1>(b);
        step<0, 1, 2>(b);
        if (b + 1 < nb) {
            step<1, 0, 3>(b + 1);
            step<1, 1, 4>(b + 1);
        }
        // no copy into LDS and no load into a register the compiler counts as
        // free may outlive the loop
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    // output tile (row block rb, token tile tt), blocks sb0 .. sb0 + n - 1
    __device__ __forceinline__ void setup(const GemmArgs &a, int rb, int tt, int64_t sb0, int n) {
        const int64_t p0 = (int64_t)tt * GD_BN, t0 = 2 * GD_NW * (int64_t)rb + 2 * wave;
        const int64_t tiles = (a.g.rows + MT_ROWS - 1) / MT_ROWS, nsb = gd_blocks(a.g);
        const int tn = (int)(a.ntok - p0 < GD_BN ? a.ntok - p0 : GD_BN);
        fresh_lane();
        l16 = 16 * lane;
        r16 = 16 * (lane & 15);
        nb = n;
        if constexpr (gd_planes<T>()) {
            first = (int)sb0;
            nu = (int)a.g.nu;
#pragma unroll
            for (int p = 0; p < 3; ++p) pitch[p] = (uint32_t)a.g.pitch[p];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t r = (t0 + j < tiles ? t0 + j : tiles - 1) * MT_ROWS;
                dr[j] = (uint32_t)(r + (lane & 15) < a.g.rows ? lane & 15 : a.g.rows - 1 - r);
#pragma unroll
                for (int p = 0; p < 3; ++p) pl[j][p] = a.W + a.g.plane[p] + r * a.g.pitch[p];
            }
        } else {
            w0p = a.Wt + ((t0 < tiles ? t0 : tiles - 1) * nsb + sb0) * BB;
            w1p = a.Wt + ((t0 + 1 < tiles ? t0 + 1 : tiles - 1) * nsb + sb0) * BB;
        }
        xb = reinterpret_cast<const uint8_t *>(a.Xh + p0 * a.ldh + sb0 * 256);
        // copy i of wave w fills rows 4 (8 i + w) .. + 3 of the step: lane l row
        // + l / 16, position l % 16, from the row's 16-byte chunk
        // (l % 16) ^ (row % 16), so that the 16 tokens of an operand read hit 16
        // bank groups; rows past the last token read row 0
#pragma unroll
        for (int i = 0; i < XN; ++i) {
            const int row = (GD_NW * i + wave) * 4 + (lane >> 4), c = (lane & 15) ^ (row & 15);
            xoff[i] = (uint32_t)(row < tn ? row : 0) * (uint32_t)a.ldh * 2u + 16u * (uint32_t)c;
        }
    }
    // D: the lane holds token lane % 16 of token tile i and rows 4 (lane / 16) +
    // v of row tile j: one 16-byte store where rows are contiguous. out points
    // at the tile's first row and token; scaled: results, else a part's sums
    __device__ __forceinline__ void store(const GemmArgs &a, int rb, int tt, float *out, int64_t ts, int64_t rs,
                                          bool scaled) {
        fresh_lane();
        const int fr = lane & 15, q = lane >> 4;
        const int64_t p0 = (int64_t)tt * GD_BN, r0 = (int64_t)rb * GD_BM;
        const int tn = (int)(a.ntok - p0 < GD_BN ? a.ntok - p0 : GD_BN);
        const int rn = (int)(a.g.rows - r0 < GD_BM ? a.g.rows - r0 : GD_BM);
        const bool vec = rs == 1 && ts % 4 == 0 && (uintptr_t)out % 16 == 0;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int lt = 16 * i + fr;
            if (lt >= tn) continue;
            const float sc = scaled ? a.inv[p0 + lt] : 1.0f;
            float *yp = out + lt * ts;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int r = (2 * wave + j) * MT_ROWS + 4 * q;
                const lq_f4 v = acc[i][j] * sc;
                if (vec && r + 3 < rn) {
                    *reinterpret_cast<lq_f4 *>(yp + r) = v;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (r + k < rn) yp[(r + k) * rs] = v[k];
                }
            }
        }
    }
};

template <int T>
__global__ __launch_bounds__(64 * GD_NW, 2) void gemm_dense_kernel(DenseArgs d) {
    extern __shared__ __attribute__((aligned(16))) uint8_t gd_lds[];
    const GemmArgs &a = d.a;
    const int lane = lane_id(), wave = wave_id();
    const int ntt = (int)((a.ntok + GD_BN - 1) / GD_BN), nrb = (int)((a.g.rows + GD_BM - 1) / GD_BM);
    const int nsb = (int)gd_blocks(a.g);
    // Workgroups go to the 8 XCDs round robin (id % 8); in every round each XCD
    // takes a contiguous range of the items (gd_tile's order). The round after the
    // whole tiles holds the rest's parts, ordered (part, tile).
    const int xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
    const int parts = d.rest * d.splits, pp = (parts + 7) / 8;
    const int part = idx < pp && xcd * pp + idx < parts ? xcd * pp + idx : -1;

    auto go = [&](auto n) {
        constexpr int NV = decltype(n)::value;
        GdMain<T, NV> m;
        m.lane = lane;
        m.wave = wave;
        m.ring = gd_lds;
        m.ring0 = (uint32_t)(uintptr_t)gd_lds;
        // item: a whole tile of round base / 256, or this workgroup's part
        int base = 0, tile, sp, rb, tt;
        bool whole;
        auto item = [&]() {
            whole = base < d.full;
            tile = whole ? base + 32 * xcd + idx : d.full + part % d.rest;
            sp = whole ? 0 : part / d.rest;
            gd_tile(tile, ntt, nrb, rb, tt);
        };
        auto start = [&]() {
            const int sb0 = whole ? 0 : sp * d.blocks;
            const int nb = whole ? nsb : nsb - sb0 < d.blocks ? nsb - sb0 : d.blocks;
            m.setup(a, rb, tt, sb0, nb);
            m.issue();
        };
        item();
        start();
        for (;;) {
            m.run();
            const int tile0 = tile, sp0 = sp, rb0 = rb, tt0 = tt;
            const bool to_y = whole || d.splits == 1;
            base += 256;
            const bool more = base < d.full || (base == d.full && d.full > 0 && part >= 0);
            if (more) {
                // every wave has read its last x: the next tile's first requests
                // go out before this one's results
                cu_barrier();
                item();
                start();
            }
            if (to_y)
                m.store(a, rb0, tt0, a.Y + (int64_t)tt0 * GD_BN * a.y_ts + (int64_t)rb0 * GD_BM * a.y_rs, a.y_ts, a.y_rs,
                        true);
            else
                m.store(a, rb0, tt0, d.P + ((int64_t)sp0 * d.rest + (tile0 - d.full)) * GD_PART,
                        a.y_rs == 1 ? GD_BM : 1, a.y_rs == 1 ? 1 : GD_BN, false);
            if (!more) break;
        }
    };
    if (d.full > 0) {
        go(std::integral_constant<int, 8>{});
    } else {
        // one item per workgroup: only the MFMA tiles that hold tokens
        if (part < 0) return;
        int rb, tt;
        gd_tile(part % d.rest, ntt, nrb, rb, tt);
        const int64_t left = a.ntok - (int64_t)tt * GD_BN;
        const int nv = __builtin_amdgcn_readfirstlane((int)((left + 15) >> 4));
        if (nv <= 2) go(std::integral_constant<int, 2>{});
        else if (nv <= 4) go(std::integral_constant<int, 4>{});
        else if (nv <= 6) go(std::integral_constant<int, 6>{});
        else go(std::integral_constant<int, 8>{});
    }
}

// Y of the rest tiles = the sum of their parts, in part order, times the token's
// scale (a power of two; the parts are unscaled, in the range of f16 products:
// scaled ones could overflow where the whole does not). Workgroup: tile
// blockIdx.x, 16 of its 128 tokens or 32 of its 256 rows, whichever runs slowest
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(DenseArgs d) {
    const GemmArgs &a = d.a;
    const int ntt = (int)((a.ntok + GD_BN - 1) / GD_BN), nrb = (int)((a.g.rows + GD_BM - 1) / GD_BM);
    int rb, tt;
    gd_tile(d.full + (int)blockIdx.x, ntt, nrb, rb, tt);
    const int64_t p0 = (int64_t)tt * GD_BN, r0 = (int64_t)rb * GD_BM;
    const int tn = (int)(a.ntok - p0 < GD_BN ? a.ntok - p0 : GD_BN);
    const int rn = (int)(a.g.rows - r0 < GD_BM ? a.g.rows - r0 : GD_BM);
    // slow x fast: tokens x rows, or rows x tokens
    const bool rows_fast = a.y_rs == 1;
    const int nfast = rows_fast ? GD_BM : GD_BN, sn = rows_fast ? tn : rn, fn = rows_fast ? rn : tn;
    const int64_t ys = rows_fast ? a.y_ts : a.y_rs;
    float *Y = a.Y + p0 * a.y_ts + r0 * a.y_rs;
    const bool vec = ys % 4 == 0 && (uintptr_t)Y % 16 == 0;
    const float *P = d.P + (int64_t)blockIdx.x * GD_PART;
    const int64_t stride = (int64_t)d.rest * GD_PART;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int e = (int)blockIdx.y * 4096 + 1024 * h + 4 * (int)threadIdx.x, si = e / nfast, fi = e % nfast;
        if (si >= sn || fi >= fn) continue;
        lq_f4 sc, sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int tk = rows_fast ? si : fi + k;
            sc[k] = a.inv[p0 + (tk < tn ? tk : tn - 1)];
        }
        for (int k0 = 0; k0 < d.splits; k0 += 8) {
            lq_f4 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                v[k] = *reinterpret_cast<const lq_f4 *>(P + (k0 + k < d.splits ? k0 + k : d.splits - 1) * stride + e);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k0 + k < d.splits) sum += v[k];
        }
        sum *= sc;
        float *y = Y + si * ys + fi;
        if (vec && fi + 3 < fn) {
            *reinterpret_cast<lq_f4 *>(y) = sum;
        } else {
            for (int k = 0; k < 4; ++k)
                if (fi + k < fn) y[k] = sum[k];
        }
    }
}

// ---------------------------------------------------------------- host side

struct DensePlan {
    int64_t tiles;
    int full, rest, splits, blocks;
    // at most `most` splits, none of them empty
    void fit(int64_t nsb, int64_t most) {
        const int64_t sp = splits < most ? splits : most < 2 ? 1 : most;
        blocks = (int)((nsb + sp - 1) / sp);
        splits = (int)((nsb + blocks - 1) / blocks);
    }
    int64_t bytes() const { return splits > 1 ? (int64_t)rest * splits * GD_PART * 4 : 0; }
};

// A workgroup per CU: whole rounds of 256 tiles, then the rest split in K over
// one more round. A 256-value block costs a workgroup 0.9 us (32 tokens), 1.9 (96)
// or 3.2 (128: bound by its MFMAs and decode, the others by latency), while parts
// write and read their sums (3.5 TB/s for both ways together) and need the
// summing launch (5 us, 1.5 more for every further eight parts it adds up): the
// split with the least total. One set of constants for all types, from Q4_K and
// Q6_K calls (Q5_K's decode takes longer per block). Measured, whole calls: 4096 x 4096 Q4_K, 77 tokens:
// 1 part 49.6 us, 4 23.8, 8 (taken) 22.3, 16 25.2; 14336 x 4096, 256 tokens: 1
// 56.9, 2 (taken) 45.8; 4096 x 14336 Q6_K, 333 tokens: 1 183, 4 64.8, 5 (taken)
// 63.9, 8 98 (two rounds); 14080 x 1280, 120 tokens: 1 (taken) 25.3, 3 26.9.
static DensePlan dense_plan(const lq_geom &g, int64_t ntok) {
    DensePlan p;
    const int64_t nsb = gd_blocks(g);
    p.tiles = (g.rows + GD_BM - 1) / GD_BM * ((ntok + GD_BN - 1) / GD_BN);
    p.full = (int)(p.tiles / 256 * 256);
    p.rest = (int)(p.tiles - p.full);
    p.splits = 1;
    const int64_t nv = ntok >= GD_BN ? 8 : (ntok + 31) / 32 * 2;
    const double block_us = nv == 8 ? 3.2 : 0.4 + 0.25 * (double)nv;
    const double part_us = (double)(ntok < GD_BN ? ntok : GD_BN) * GD_BM * 4.0 / 3.5e6;
    double best = 0.0;
    for (int64_t s = 1; p.rest && s <= nsb && s * p.rest <= 256; ++s) {
        const int64_t blocks = (nsb + s - 1) / s;
        if ((nsb + blocks - 1) / blocks != s) continue;
        const double us = block_us * (double)blocks + (s > 1 ? 5.0 + 1.5 * (double)((s - 1) / 8) + (double)(s * p.rest) * part_us : 0.0);
        if (s == 1 || us < best) {
            best = us;
            p.splits = (int)s;
        }
    }
    p.fit(nsb, p.splits);
    return p;
}

// Time of a whole dense call (conversion of x included), for launch_gemm's choice
// between this kernel and gemm_tile_kernel: fitted to 5900 calls (1 to 16 blocks
// of K, 512 to 128256 rows, 1 to 2048 tokens; four in five within 5.5 %). Besides
// the blocks, a workgroup's first loads and its stores are most of a short K's
// time: 2048 x 768 Q4_K, 512 tokens, 32 workgroups: 20.5 us, of which the three
// blocks take 9. *split_bytes: the parts' bytes.
double gemm_dense_us(const lq_geom &g, int64_t ntok, int64_t *split_bytes) {
    const DensePlan p = dense_plan(g, ntok);
    *split_bytes = p.bytes();
    const double fixed[4] = {6.1, 8.3, 9.2, 10.3}, block[4] = {1.6, 1.9, 2.3, 2.9};   // by computed MFMA tiles / 2
    const int i = p.full || ntok > 96 ? 3 : (int)((ntok - 1) / 32), rounds = p.full / 256;
    const double extra = g.type == LQ_Q6_K ? 0.3 : 0.0;                                 // more decode
    double us = fixed[i];
    if (rounds) us += (3.45 + extra) * (double)(rounds * gd_blocks(g)) + 2.4 * (double)(rounds - 1);
    if (p.rest) us += (block[i] + extra) * (double)p.blocks + (rounds ? 2.6 : 0.0);
    // one token tile: every weight of the rounds comes from memory, and Q8_0 has most
    if (rounds && ntok <= GD_BN && g.type == LQ_Q8_0) us += 0.3 * (double)((rounds + (p.rest ? 1 : 0)) * gd_blocks(g));
    if (p.splits > 1)
        us += 5.05 + 3.0 * (double)((p.splits - 1) / 8) +
              (double)(p.rest * p.splits * (ntok < GD_BN ? ntok : GD_BN)) * GD_BM * 4.0 / 3.3e6;
    return us;
}

int launch_gemm_dense(const GemmArgs &a, void *split_ws, int64_t split_bytes, hipStream_t s) {
    constexpr int lds = GD_RING * GD_SLOT;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    // the kernel is chosen by type alone: its weights must be the ones it reads
    if (a.g.type == LQ_Q5_K || a.g.type == LQ_Q4_0 ? !a.W : !a.Wt)
        return fail(LOCALAI_ESTATE, "matmul: handle without the weights' form");
    DensePlan p = dense_plan(a.g, a.ntok);
    if (p.rest) p.fit(gd_blocks(a.g), split_bytes / (p.rest * GD_PART * 4));
    // 32-bit byte offsets into the x rows of a workgroup
    if ((int64_t)a.ldh * 2 * (a.ntok < GD_BN ? a.ntok : GD_BN) >= ((int64_t)1 << 32) || p.tiles > ((int64_t)1 << 30))
        return fail(LOCALAI_EARG, "matmul: problem too large");
    const DenseArgs d{a, p.full, p.rest, p.splits, p.blocks, (float *)split_ws};
    const dim3 grid(p.full ? 256 : (unsigned)((p.rest * p.splits + 7) / 8 * 8));
    switch (a.g.type) {
#define LQ_GD(TT) case TT: hipLaunchKernelGGL(gemm_dense_kernel<TT>, grid, dim3(64 * GD_NW), lds, s, d); break;
        LQ_GD(LQ_Q4_K) LQ_GD(LQ_Q6_K) LQ_GD(LQ_Q8_0) LQ_GD(LQ_Q5_K) LQ_GD(LQ_Q4_0)
#undef LQ_GD
        default: return fail(LOCALAI_ETYPE, "matmul: unsupported GGML type");
    }
    LQ_HIP(hipGetLastError());
    if (p.splits > 1) {
        hipLaunchKernelGGL(gemm_split_sum_kernel, dim3((unsigned)p.rest, 8), dim3(256), 0, s, d);
        LQ_HIP(hipGetLastError());
    }
    return LOCALAI_OK;
}

}  // namespace lq
