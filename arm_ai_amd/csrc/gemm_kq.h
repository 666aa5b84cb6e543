// gemm_kq.h -- the prefill GEMM (from gemm_min_rows rows) of the K-quant weights
// (Q4_K, Q5_K, Q6_K, Q2_K, Q3_K) on the f16 matrix cores, gfx950: its kernel
// template and parameters.  k_gemm.hip holds the launch plan; one small .hip file per
// weight type instantiates the template.
//
// Replaces the M-row loop of candle-core 0.8.4 k_quants::matmul<T> at
// prefill (native/arm_ai_nif/src/llama_candle.rs:93, forward(&x[1,L], 0)):
//   y[m][n] = sum over super-blocks b of
//     d_x[m,b] * (d_w[n,b] * S[m,n,b] - dmin_w[n,b] * Smin[m,n,b]),
//   S    = sum_j sc[n,b,j] * sum_{e in sub-block j} q[n,e] * qx[m,e]
//   Smin = sum_g bsums[m,b,g] * mn[n,b,g]      (Q4_K, Q5_K, Q2_K)
// with S and Smin exact integers, as in candle's vec_dot.
//
// Exactness.  The activation operand is the Q8_K quant (|qx| <= 128), the
// weight operand the integer sc * q, both exact in f16; products and sums are
// exact in the MFMA's f32 accumulators up to 2^24:
//   Q4_K  sc * q <= 63 * 15; half a super-block stays below 2^24
//   Q5_K  sc * q <= 63 * 31; a quarter does
//   Q2_K  sc * q <= 15 * 3;  Q3_K  |sc * (u - 4)| <= 32 * 4: whole super-blocks
//   Q6_K  |sc * (q - 32)| reaches 4096, odd values above 2048 are not f16:
//         the scale is split, sc = 16 sh + sl (sh in -8..7, sl in 0..15), into
//         the operands sh (q - 32) and sl (q - 32) / 16 (at most 9 significant
//         bits each) of one chain, which holds S / 16; one step stays exact
// The integer dump restarts the chain where it could round and adds in int32.  The
// output chains a whole super-block: S is exact below 2^24 (Q6_K: while every
// partial sum is), and rounded to 24 bits by each later step beyond, which the
// sums of real files do not reach (normal activations: 2^21 on random weights).  Error
// against 64 bits, 40 x 64 x 2048, Q4_K, Q5_K, Q6_K: normal activations 7.4e-8,
// 7.2e-8, 6.5e-8 of the result; activations of one sign on the largest weights, S
// up to 2^24.8, 2^25.8, 2^26.9: 6.9e-8, 6.4e-8, 5.0e-8.
// Smin is one more f16 MFMA per tile and super-block (bsums <= 2048, mins <=
// 63; every partial sum below 2^24).
//
// The weight operand is built from the packed bytes in place: (w & mask) |
// 0x6400 puts a field of byte 0 and of byte 2 into the mantissas of a pair of
// halves, 1024 + f * 2^s, with one v_and_or_b32; one packed f16 fma by
// (sc / 2^s, -1024 sc / 2^s) leaves the exact sc * q.  Bytes 1 and 3 follow
// from w >> 8.  The pairs come in the order (0, 2, 1, 3) of each four
// elements, the order in which the quantizers write the f16 activation plane
// (ActPlanes::q16).
//
// Tiling.  A workgroup of four wavefronts owns 32 MT rows x 128 NT columns;
// wavefront w owns 32 NT columns and all the rows, so each operand it builds
// feeds MT MFMAs.  v_mfma_f32_32x32x16_f16: lane (column l % 32, half h = l /
// 32) holds, of sub-block s and i = 0, 1, the elements 32 s + 16 h + 8 i + 0..7,
// so a lane reads whole 16-byte pieces of its own column.
//   * The activation rows (f16 quants, bsums, d) go global -> LDS by
//     buffer-to-LDS copies into two stages, one per half of a super-block,
//     issued one half ahead; the plane is in fragment order, so a copy is one
//     fragment and a fragment read one conflict-free ds_read at a constant
//     offset.
//   * The weights go straight into registers, one super-block ahead.
//   * One s_waitcnt vmcnt and one barrier start each half.  Loads past the
//     last super-block go through an empty descriptor.
// Work items (tile, K split) are dealt so that the row tiles and splits of one
// column tile run on one XCD and share its L2's copy of the weights.
#pragma once

#include "aq_internal.h"

#include <type_traits>

namespace aq {

struct KqParams {
    const uint8_t *w;    // row-block tiles
    const uint16_t *wd;  // Q6_K, Q2_K: d plane
    int64_t rb_stride;
    int ng;              // super-blocks per row
    const uint16_t *x16;  // activation quants as f16 (q16_at)
    const float *xd;      // [m][ng]
    const uint16_t *xbs;  // bsums as f16 [m][k/16]
    float *y;             // [m][n], or with splits > 1 the partials [splits][m][n]
    int m, n, k;
    int ntm, splits, kbs, items, per_xcd;
    int32_t *S, *Smin;    // integer dump [m][n][ng] or null
};

// Tile forms.
struct KqForm {
    int rows, cols;
};
// 4, 5: few rows, 4 or 8 wavefronts over K (d of their rows in LDS, 128 bytes a super-block)
constexpr KqForm KQ_FORMS[] = {{32, 128}, {64, 128}, {128, 256}, {128, 128}, {32, 32}, {32, 32}};
constexpr int KQ_FEW_MAX_NG = 256;  // super-blocks of a split
hipError_t launch_kq_q4k(const KqParams &p, int form, bool dump, hipStream_t s);
hipError_t launch_kq_q5k(const KqParams &p, int form, bool dump, hipStream_t s);
hipError_t launch_kq_q6k(const KqParams &p, int form, bool dump, hipStream_t s);
hipError_t launch_kq_q2k(const KqParams &p, int form, bool dump, hipStream_t s);
hipError_t launch_kq_q3k(const KqParams &p, int form, bool dump, hipStream_t s);
// a Q4_K weight and a Q6_K or Q5_K one (type2) in one launch, both in the 64 x 128 form
hipError_t launch_kq_pair(const KqParams &p1, const KqParams &p2, int type2, hipStream_t s);

#ifdef __HIPCC__

namespace kq {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

constexpr int NXCD = 8;

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u32(h2 v) { return __builtin_bit_cast(uint32_t, v); }
// the pair (v, v) of f16 for an integer byte b of w, exact: 1024 + v, less 1024
__device__ __forceinline__ h2 pair_of_byte(uint32_t w, int b) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)b | ((uint32_t)b << 16))) -
           (h2){(_Float16)1024.0f, (_Float16)1024.0f};
}
// v through an empty asm: what is derived from it is computed where it is
// used, in an instruction or two, instead of held in registers for the loop
__device__ __forceinline__ void opaque(uint32_t &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ h2 splat(float f) { return (h2){(_Float16)f, (_Float16)f}; }

// One lane's weight bytes of one super-block of one column.
template <int TYPE> struct W;
template <> struct W<TYPE_Q4_K> { u32x4 meta, q[4]; };
template <> struct W<TYPE_Q5_K> { u32x4 meta, qh, q[4]; };
template <> struct W<TYPE_Q6_K> { u32x4 q[4], qh[2], sc; uint32_t d; };
template <> struct W<TYPE_Q2_K> { u32x4 sc, q[2]; uint32_t d; };
template <> struct W<TYPE_Q3_K> { u32x4 meta, hm, q[2]; };

// Loads per super-block and column set (all lanes, one instruction each).
template <int TYPE> constexpr int nloads() {
    return TYPE == TYPE_Q4_K ? 5 : TYPE == TYPE_Q5_K ? 6 : TYPE == TYPE_Q6_K ? 8 : 4;
}

__device__ __forceinline__ u32x4 ld16(const rsrc_t &r, uint32_t voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

// Piece loads of super-block b: woff is this lane's column's byte offset
// (piece 0 of group 0), doff its entry offset in the d plane.  load_head
// takes the scales (and d), load_after the quant pieces whose last use is
// sub-block S.
template <int TYPE>
__device__ __forceinline__ void load_head(W<TYPE> &v, const rsrc_t &r, const rsrc_t &rd, uint32_t woff, uint32_t doff, int b) {
    const int soff = b * slabs_of(TYPE) * 128;
    if constexpr (TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K) v.meta = ld16(r, woff, soff);
    else if constexpr (TYPE == TYPE_Q6_K) {
        v.sc = ld16(r, woff + 128u * 12, soff);
        v.d = __builtin_amdgcn_raw_buffer_load_b16(rd, doff * 2, b * RB * 2, 0);
    } else if constexpr (TYPE == TYPE_Q2_K) {
        v.sc = ld16(r, woff, soff);
        v.d = __builtin_amdgcn_raw_buffer_load_b32(rd, doff * 4, b * RB * 4, 0);
    } else v.meta = ld16(r, woff + 128u * 6, soff);
}
template <int TYPE, int S>
__device__ __forceinline__ void load_after(W<TYPE> &v, const rsrc_t &r, uint32_t woff, int h, int b) {
    const int soff = b * slabs_of(TYPE) * 128;
    const uint32_t voff = woff + 128u * h;
    if constexpr (TYPE == TYPE_Q4_K) {
        if constexpr (S & 1) v.q[S >> 1] = ld16(r, voff + 128u * (1 + (S & ~1)), soff);
    } else if constexpr (TYPE == TYPE_Q5_K) {
        if constexpr (S & 1) v.q[S >> 1] = ld16(r, voff + 128u * (3 + (S & ~1)), soff);
        if constexpr (S == 7) v.qh = ld16(r, voff + 128u, soff);
    } else if constexpr (TYPE == TYPE_Q6_K) {
        if constexpr ((S & 3) >= 2) v.q[2 * (S >> 2) + (S & 1)] = ld16(r, voff + 128u * (4 * (S >> 2) + 2 * (S & 1)), soff);
        if constexpr ((S & 3) == 3) v.qh[S >> 2] = ld16(r, voff + 128u * (8 + 2 * (S >> 2)), soff);
    } else if constexpr (TYPE == TYPE_Q2_K) {
        if constexpr ((S & 3) == 3) v.q[S >> 2] = ld16(r, voff + 128u * (1 + 2 * (S >> 2)), soff);
    } else {
        if constexpr ((S & 3) == 3) v.q[S >> 2] = ld16(r, voff + 128u * (2 + 2 * (S >> 2)), soff);
        if constexpr (S == 7) v.hm = ld16(r, voff, soff);
    }
}
// All of a super-block, NT columns, in the order in which it is used.
template <int TYPE, int NT, int S = 0>
__device__ __forceinline__ void load_rest(W<TYPE> (&v)[NT], const rsrc_t &r, const uint32_t (&woff)[NT], int h, int b) {
#pragma unroll
    for (int u = 0; u < NT; u++) load_after<TYPE, S>(v[u], r, woff[u], h, b);
    __builtin_amdgcn_sched_barrier(0);  // (the loop's order, so that its waits count the same loads)
    if constexpr (S < 7) load_rest<TYPE, NT, S + 1>(v, r, woff, h, b);
}
template <int TYPE, int NT>
__device__ __forceinline__ void load_all(W<TYPE> (&v)[NT], const rsrc_t &r, const rsrc_t &rd, const uint32_t (&woff)[NT],
                                         const uint32_t (&doff)[NT], int h, int b) {
#pragma unroll
    for (int u = 0; u < NT; u++) load_head<TYPE>(v[u], r, rd, woff[u], doff[u], b);
    __builtin_amdgcn_sched_barrier(0);
    load_rest<TYPE, NT>(v, r, woff, h, b);
}

// The scales of one column's super-block, unpacked to bytes, for this lane
// half: Q4_K / Q5_K the eight 6-bit scales and mins (candle's utmp form of
// get_scale_min_k4); Q2_K / Q3_K / Q6_K the scales of groups 2 s + h (byte s
// of sc; Q3_K as s6, Q6_K as the int8 plus 128), Q2_K's mins of its 8 h + i.
struct Scales {
    uint32_t sc[2], mn[2];
};
template <int TYPE>
__device__ __forceinline__ Scales unpack_scales(const W<TYPE> &v, int h) {
    Scales r;
    if constexpr (TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K) {
        const uint32_t u0 = v.meta.y, u1 = v.meta.z, u2 = v.meta.w;
        r.sc[0] = u0 & 0x3F3F3F3Fu;
        r.sc[1] = (u2 & 0x0F0F0F0Fu) | ((u0 >> 2) & 0x30303030u);
        const uint32_t m0 = u1 & 0x3F3F3F3Fu, m1 = ((u2 >> 4) & 0x0F0F0F0Fu) | ((u1 >> 2) & 0x30303030u);
        r.mn[0] = h ? m1 : m0;  // the mins of bsum groups 8 h .. 8 h + 7
    } else {
        // byte 2 s + h of the sixteen: pick the even or odd bytes
        const uint32_t sel = h ? 0x07050301u : 0x06040200u;
        u32x4 a;
        if constexpr (TYPE == TYPE_Q3_K) {
            // s[i] = low nibbles of bytes 0..7 (s 0..7), high nibbles (s 8..15), top two bits from bytes 8..11
            const uint32_t l0 = v.meta.x, l1 = v.meta.y, t = v.meta.z;
            a.x = (l0 & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u);
            a.y = (l1 & 0x0F0F0F0Fu) | ((t << 2) & 0x30303030u);
            a.z = ((l0 >> 4) & 0x0F0F0F0Fu) | (t & 0x30303030u);
            a.w = ((l1 >> 4) & 0x0F0F0F0Fu) | ((t >> 2) & 0x30303030u);
        } else if constexpr (TYPE == TYPE_Q6_K) {
            a = v.sc ^ 0x80808080u;
        } else {
            a = v.sc;
            // mins of groups 8 h .. 8 h + 7
            r.mn[0] = ((h ? a.z : a.x) >> 4) & 0x0F0F0F0Fu;
            r.mn[1] = ((h ? a.w : a.y) >> 4) & 0x0F0F0F0Fu;
            a &= 0x0F0F0F0Fu;
        }
        r.sc[0] = __builtin_amdgcn_perm(a.y, a.x, sel);
        r.sc[1] = __builtin_amdgcn_perm(a.w, a.z, sel);
    }
    return r;
}

// The f16 constants of sub-block s (this lane half): value = f * mul + add of
// f = 1024 + field, one pair per digit (Q6_K: high, low).
template <int TYPE> struct Consts { h2 mul, add; };
template <> struct Consts<TYPE_Q6_K> { h2 mh, ah, ml, al; };
template <int TYPE>
__device__ __forceinline__ Consts<TYPE> consts(const Scales &z, int s) {
    Consts<TYPE> c;
    const uint32_t w = z.sc[s >> 2];
    const int b = s & 3;
    if constexpr (TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K) {
        const h2 sc = pair_of_byte(w, b);
        c.mul = (s & 1) ? sc * splat(0.0625f) : sc;  // high nibbles are taken in place, times 16
        c.add = c.mul * splat(-1024.0f);
    } else if constexpr (TYPE == TYPE_Q2_K) {
        const int jj = s & 3;
        c.mul = pair_of_byte(w, b) * splat(jj == 0 ? 1.0f : jj == 1 ? 0.25f : jj == 2 ? 0.0625f : 0.015625f);
        c.add = c.mul * splat(-1024.0f);
    } else if constexpr (TYPE == TYPE_Q3_K) {
        // fields at bit 2 (jj 0, 1), 4 or 6: value = f * sc / 2^s - (1024 / 2^s + 4) * sc,
        // whose last product has at most 11 bits at these positions
        const int jj = s & 3;
        const float inv = jj <= 1 ? 0.25f : jj == 2 ? 0.0625f : 0.015625f;
        const h2 sc = pair_of_byte(w, b) - splat(32.0f);
        c.mul = sc * splat(inv);
        c.add = sc * splat(-(1024.0f * inv + 4.0f));
    } else {
        // sc + 128 = 16 (sh + 8) + sl
        const int hi = (s & 3) >> 1;  // high nibbles are taken in place, times 16
        const h2 sh = pair_of_byte((w >> 4) & 0x0F0F0F0Fu, b) - splat(8.0f), sl = pair_of_byte(w & 0x0F0F0F0Fu, b);
        c.mh = hi ? sh * splat(0.0625f) : sh;
        c.ml = sl * splat(hi ? 0.00390625f : 0.0625f);
        c.ah = sh * splat(hi ? -96.0f : -1056.0f);
        c.al = sl * splat(hi ? -6.0f : -66.0f);
    }
    return c;
}

template <int SH>
__device__ __forceinline__ uint32_t shl(uint32_t v) {  // by SH bits, to the right when negative
    if constexpr (SH >= 0) return v << SH;
    else return v >> -SH;
}

// 1024 + field as f16 pairs for elements (0, 2) and (1, 3) of dword x (and
// its high-bit dword): sub-block s.
// (magic: 0x64006400 in a vector register, so that and-or takes its mask from
// a scalar one in the same instruction.)
template <int TYPE, int S>
__device__ __forceinline__ void fields(uint32_t w, uint32_t hb, uint32_t magic, uint32_t &e, uint32_t &o) {
    if constexpr (TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K) {
        constexpr uint32_t M = (S & 1) ? 0x00F000F0u : 0x000F000Fu;
        e = (w & M) | magic;
        o = ((w >> 8) & M) | magic;
        if constexpr (TYPE == TYPE_Q5_K) {  // qh bit S to bit 4 (low nibbles) or 8 (in place, times 16)
            constexpr int AT = (S & 1) ? 8 : 4;
            constexpr uint32_t B = 0x00010001u << AT;
            e |= shl<AT - S>(hb) & B;
            o |= shl<AT - S - 8>(hb) & B;
        }
    } else if constexpr (TYPE == TYPE_Q2_K) {
        constexpr uint32_t M = 0x00030003u << (2 * (S & 3));
        e = (w & M) | magic;
        o = ((w >> 8) & M) | magic;
    } else if constexpr (TYPE == TYPE_Q3_K) {  // two bits at 2 jj, the hmask bit 4 hf + jj above them
        constexpr int JJ = S & 3, HB = 4 * (S >> 2) + JJ, AT = JJ == 0 ? 2 : 2 * JJ;
        constexpr uint32_t M = 0x00030003u << AT, B = 0x00040004u << AT;
        e = (shl<AT - 2 * JJ>(w) & M) | magic;
        o = (shl<AT - 2 * JJ - 8>(w) & M) | magic;
        e |= shl<AT + 2 - HB>(hb) & B;
        o |= shl<AT + 2 - HB - 8>(hb) & B;
    } else {  // Q6_K: nibble, and qh bits 2 qq, 2 qq + 1 above it
        constexpr int QQ = S & 3, AT = (QQ >> 1) ? 4 : 0;
        constexpr uint32_t M = 0x000F000Fu << AT, B = 0x00300030u << AT;
        e = (w & M) | magic;
        o = ((w >> 8) & M) | magic;
        e |= shl<4 + AT - 2 * QQ>(hb) & B;
        o |= shl<4 + AT - 2 * QQ - 8>(hb) & B;
    }
}

// The weight dwords of sub-block S, elements 8 i + 4 t .. + 3 of this lane's 16.
template <int TYPE, int S>
__device__ __forceinline__ uint32_t qword(const W<TYPE> &v, int at) {
    if constexpr (TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K) return v.q[S >> 1][at];
    else if constexpr (TYPE == TYPE_Q6_K) return v.q[2 * (S >> 2) + (S & 1)][at];
    else return v.q[S >> 2][at];
}
template <int TYPE, int S>
__device__ __forceinline__ uint32_t hword(const W<TYPE> &v, int at) {
    if constexpr (TYPE == TYPE_Q5_K) return v.qh[at];
    else if constexpr (TYPE == TYPE_Q6_K) return v.qh[S >> 2][at];
    else if constexpr (TYPE == TYPE_Q3_K) return v.hm[at];
    else return 0u;
}

// f16 d (low half) and, for the types that have one, dmin
template <int TYPE>
__device__ __forceinline__ uint32_t d_word(const W<TYPE> &v) {
    if constexpr (TYPE == TYPE_Q6_K || TYPE == TYPE_Q2_K) return v.d;
    else if constexpr (TYPE == TYPE_Q3_K) return v.meta.w;
    else return v.meta.x;
}

// The operands of MFMA (S, i): b[0], and for Q6_K the low digit's b[1].
template <int TYPE, int S>
__device__ __forceinline__ void operands(const W<TYPE> &v, const Consts<TYPE> &c, int i, uint32_t magic, v8h (&b)[TYPE == TYPE_Q6_K ? 2 : 1]) {
    u32x4 r, r2;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        uint32_t e, o;
        fields<TYPE, S>(qword<TYPE, S>(v, 2 * i + t), hword<TYPE, S>(v, 2 * i + t), magic, e, o);
        if constexpr (TYPE == TYPE_Q6_K) {
            r[2 * t] = as_u32(__builtin_elementwise_fma(as_h2(e), c.mh, c.ah));
            r[2 * t + 1] = as_u32(__builtin_elementwise_fma(as_h2(o), c.mh, c.ah));
            r2[2 * t] = as_u32(__builtin_elementwise_fma(as_h2(e), c.ml, c.al));
            r2[2 * t + 1] = as_u32(__builtin_elementwise_fma(as_h2(o), c.ml, c.al));
        } else {
            r[2 * t] = as_u32(__builtin_elementwise_fma(as_h2(e), c.mul, c.add));
            r[2 * t + 1] = as_u32(__builtin_elementwise_fma(as_h2(o), c.mul, c.add));
        }
    }
    b[0] = __builtin_bit_cast(v8h, r);
    if constexpr (TYPE == TYPE_Q6_K) b[1] = __builtin_bit_cast(v8h, r2);
}

// The min product's operand: B[g][n] = the min of bsum group g = 8 h + e
// (Q4_K, Q5_K: of its sub-block).
template <int TYPE>
__device__ __forceinline__ v8h min_operand(const Scales &z) {
    u32x4 bm;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if constexpr (TYPE == TYPE_Q2_K)
            bm[e] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, z.mn[e >> 1], (e & 1) ? 0x04030402u : 0x04010400u)) -
                           splat(1024.0f));
        else
            bm[e] = as_u32(pair_of_byte(z.mn[0], e));
    }
    return __builtin_bit_cast(v8h, bm);
}

// MFMA step J of a super-block: half I of sub-block S.  The sub-blocks that
// share dwords follow each other, so that w >> 8 is formed once.
template <int TYPE, int J>
struct Step {
    static constexpr bool PAIR = TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K, QUAD = TYPE == TYPE_Q2_K || TYPE == TYPE_Q3_K;
    static constexpr int I = QUAD ? (J >> 2) & 1 : (J >> 1) & 1;
    static constexpr int S = PAIR ? 2 * (J >> 2) + (J & 1) : QUAD ? 4 * (J >> 3) + (J & 3)
                                                                  : 4 * (J >> 3) + ((J >> 2) & 1) + 2 * (J & 1);
    static constexpr int SHARE = QUAD ? 4 : 2;                       // sub-blocks of a run
    static constexpr bool LAST = (J & (2 * SHARE - 1)) == 2 * SHARE - 1;  // its pieces are used up
};

// LDS: one stage per half of a super-block; the second also holds bsums and d.
template <int MT>
struct Lds {
    static constexpr int ROWS = 32 * MT;
    static constexpr int QS = ROWS * 256;  // f16 quants: fragments [row tile][8][lane]
    static constexpr int BS = 2 * QS;      // bsums [rows][16] f16
    static constexpr int DX = BS + ROWS * 32;  // d [rows] f32 (a copy writes 256 bytes)
    static constexpr int BYTES = DX + (ROWS * 4 < 256 ? 256 : ROWS * 4);
};

// The body for workgroup bid of the launch, on Lds<MT>::BYTES of LDS.
template <int TYPE, int MT, int NT, int NW, bool DUMP>
__device__ __forceinline__ void body(const KqParams &p, uint8_t *lds, int bid) {
    constexpr bool Q6 = TYPE == TYPE_Q6_K;
    constexpr bool MIN = TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K || TYPE == TYPE_Q2_K;
    constexpr int ND = Q6 ? 2 : 1;  // operands per step (scale digits)
    using L = Lds<MT>;
    const int xcd = bid % NXCD, local = bid / NXCD;
    const int item = xcd * p.per_xcd + local;
    if (local >= p.per_xcd || item >= p.items) return;  // uniform over the workgroup
    const int tile = item / p.splits, split = item - tile * p.splits;
    const int tn = tile / p.ntm, tm = tile - tn * p.ntm;
    const int m0 = tm * L::ROWS;
    const int kb0 = split * p.kbs;
    const int nit = min(p.ng, kb0 + p.kbs) - kb0;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int ng = p.ng, k = p.k;

    // activation copies: a wave copies CI fragments of one row tile per half.
    // Rows past m read zeros (the scalar offset, which the range check leaves
    // out, stays inside the tile).
    const rsrc_t rq = buf_rsrc(p.x16, (uint32_t)((int64_t)p.m * k * 2));
    const rsrc_t rdx = buf_rsrc(p.xd, (uint32_t)((int64_t)p.m * ng * 4));
    const rsrc_t rbs = buf_rsrc(p.xbs, (uint32_t)((int64_t)p.m * (k / 16) * 2));
    const rsrc_t rnone = buf_rsrc(p.x16, 0u);
    constexpr int CI = 8 * MT / NW;  // copies per wave and stage
    static_assert(8 % CI == 0);
    const int trow = m0 + 32 * (CI * wave / 8);  // the tile's first row
    const int trows = min(32, p.m - trow);       // (none: every lane past the range)
    const uint32_t qoff = l32 < trows ? (uint32_t)(trow * k * 2 + (h * trows + l32) * 32) : BUF_OOB;
    const int sbytes = 64 * max(trows, 0);       // of a sub-block
    // bsums: 32 rows per instruction (two lanes a row), wave w those of rows
    // 32 w ..; d: 64 rows per instruction, from wave 3 down.  Every wave
    // issues two small copies, so that all wait on the same counts; the spare
    // ones write to their places again with zero-range descriptors where
    // nothing is to be copied (zeros into rows past the tile are never read).
    const uint32_t bsoff = (uint32_t)(((m0 + 32 * wave + (lane >> 1)) * (k / 16) + 8 * (lane & 1)) * 2);
    const int dxw = wave & 1;  // waves 0, 1 (and 2, 3 again): rows 64 dxw ..
    const uint32_t dxoff = (uint32_t)((m0 + 64 * dxw + lane) * ng * 4);

    // weights: column set u of this wave, column 128 NT tn + 32 (NT wave + u) + l32
    const int nrb = (p.n + RB - 1) / RB;
    const int rb0 = 4 * NW * NT * tn;
    const int rb_here = min(4 * NW * NT, nrb - rb0);
    const rsrc_t rw = buf_rsrc(p.w + (int64_t)rb0 * p.rb_stride, (uint32_t)(rb_here * p.rb_stride));
    constexpr int DB = TYPE == TYPE_Q2_K ? 4 : 2;  // bytes per d-plane entry
    const rsrc_t rwd = (Q6 || TYPE == TYPE_Q2_K)
                           ? buf_rsrc((const uint8_t *)p.wd + (int64_t)rb0 * ng * RB * DB, (uint32_t)(rb_here * ng * RB * DB))
                           : rw;
    uint32_t woff[NT], doff[NT];
#pragma unroll
    for (int u = 0; u < NT; u++) {
        const int rb = 4 * (NT * wave + u) + (l32 >> 3);
        woff[u] = (uint32_t)(rb * p.rb_stride + (l32 & 7) * 16);
        doff[u] = (uint32_t)(rb * ng * RB + (l32 & 7));
    }

    // The weight registers hold one super-block; a piece is loaded again, for
    // the next one, as soon as its last operand is built.
    // Weight loads of the steps of each half (the second half's wait also
    // leaves the heads in flight).
    constexpr int PIECES0 = NT * (TYPE == TYPE_Q6_K ? 3 : TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K ? 2 : 1);
    constexpr int PIECES1 = NT * (TYPE == TYPE_Q6_K || TYPE == TYPE_Q5_K ? 3 : TYPE == TYPE_Q2_K ? 1 : 2);
    constexpr int HEADS = NT * (TYPE == TYPE_Q6_K || TYPE == TYPE_Q2_K ? 2 : 1);
    static_assert(HEADS + PIECES0 + PIECES1 == NT * nloads<TYPE>());
    // VALU instructions between two MFMAs: about those that build a step's operands
    constexpr int VALU_STEP = TYPE == TYPE_Q5_K ? 19 : TYPE == TYPE_Q6_K ? 24 : TYPE == TYPE_Q3_K ? 18 : 13;
    constexpr int VALU_EACH = (VALU_STEP * NT + MT * NT * ND - 1) / (MT * NT * ND);
    using WT = W<TYPE>;
    auto issue = [&](int i, auto HALF) {  // the activation of that half of super-block kb0 + i
        constexpr int HF = decltype(HALF)::value;
        const int b = kb0 + i;
        const bool live = i < nit;
        const rsrc_t r1 = live ? rq : rnone;
#pragma unroll
        for (int c = 0; c < CI; c++)
            buf_to_lds16(r1, lds + HF * L::QS + 1024 * (CI * wave + c), qoff,
                         (b * 8 + 4 * HF + (CI * wave + c) % 8 / 2) * sbytes + 16 * (c & 1));
        if constexpr (HF == 1) {
            if constexpr (MIN) {
                const int bw = wave < MT ? wave : 0;  // (spare waves copy rows 0..31 of the tile again)
                const uint32_t bo = wave < MT ? bsoff : bsoff - (uint32_t)(32 * wave * (k / 16) * 2);
                buf_to_lds16(live ? rbs : rnone, lds + L::BS + 1024 * bw, bo, b * 32);
            }
            if constexpr (MT == 4) buf_to_lds4(live ? rdx : rnone, lds + L::DX + 256 * dxw, dxoff, b * 4);
            else buf_to_lds4(live ? rdx : rnone, lds + L::DX, dxoff - (uint32_t)(64 * dxw * ng * 4), b * 4);
        }
    };

    v16f yacc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int u = 0; u < NT; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) yacc[t][u][r] = 0.0f;

    const uint8_t *frag = lds + 16 * lane;  // this lane's part of fragment 0, row tile 0
    WT v[NT];
    auto super_block = [&](int i) {
        // This wave's copies of the half have landed (those of the other half
        // were issued before; the weight loads stay in flight, the compiler
        // waits for those where they are used) and its LDS reads are done, a
        // barrier (every wave's copies have landed, and every wave has read the
        // other half's stage, which the copies issued now overwrite).
        auto enter = [&](auto HALF) {
            constexpr int HF = decltype(HALF)::value;
            wait_vmcnt<HF == 0 ? PIECES1 : HEADS + PIECES0>();
            lds_barrier();
            issue(HF == 0 ? i : i + 1, std::integral_constant<int, 1 - HF>{});
            // the next wait counts the loads that follow: no copy may sink past one
            // (the compiler moved d's behind the heads)
            __builtin_amdgcn_sched_barrier(0);
        };
        enter(std::integral_constant<int, 0>{});
        v16f acc[MT][NT];
        v16i isum[DUMP ? MT : 1][DUMP ? NT : 1];
        if constexpr (DUMP) {
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int u = 0; u < NT; u++)
#pragma unroll
                    for (int r = 0; r < 16; r++) isum[t][u][r] = 0;
        }
        Scales z[NT];
        uint32_t dd[NT];
        const bool more = i + 1 < nit;
        const rsrc_t r4 = more ? rw : rnone, r5 = more ? rwd : rnone;
#pragma unroll
        for (int u = 0; u < NT; u++) {
            z[u] = unpack_scales<TYPE>(v[u], h);
            dd[u] = d_word<TYPE>(v[u]);
            load_head<TYPE>(v[u], r4, r5, woff[u], doff[u], kb0 + i + 1);
        }
        // The fragments of step J + 1 are read and built while the MFMAs of
        // step J run.
        v8h a[2][MT], b[2][NT][ND];
        Consts<TYPE> c[NT][Step<TYPE, 0>::SHARE];
        uint32_t magic = 0x64006400u;
        opaque(magic);
        auto build = [&](auto JC) {
            constexpr int J = decltype(JC)::value;
            using P = Step<TYPE, J>;
#pragma unroll
            for (int t = 0; t < MT; t++)
                a[J & 1][t] = *(const v8h *)(frag + (J >> 3) * L::QS + 8192 * t + 1024 * ((2 * P::S + P::I) & 7));
#pragma unroll
            for (int u = 0; u < NT; u++) {
                if constexpr (P::I == 0) c[u][J % P::SHARE] = consts<TYPE>(z[u], P::S);
                operands<TYPE, P::S>(v[u], c[u][J % P::SHARE], P::I, magic, b[J & 1][u]);
            }
        };
        auto step = [&](auto JC) {
            constexpr int J = decltype(JC)::value;
            using P = Step<TYPE, J>;
            if constexpr (J % 8 != 7) build(std::integral_constant<int, J + 1>{});
            if constexpr (P::LAST) {
#pragma unroll
                for (int u = 0; u < NT; u++) load_after<TYPE, P::S>(v[u], r4, woff[u], h, kb0 + i + 1);
            }
            // steps per chain
            constexpr int CH = !DUMP ? 16 : TYPE == TYPE_Q4_K ? 8 : TYPE == TYPE_Q5_K ? 4 : Q6 ? 1 : 16;
#pragma unroll
            for (int g = 0; g < ND; g++)
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int u = 0; u < NT; u++) {
                        const v16f zero = {0};
                        acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J & 1][t], b[J & 1][u][g],
                                                                          J % CH == 0 && g == 0 ? zero : acc[t][u], 0, 0, 0);
                    }
            if constexpr (DUMP && J % CH == CH - 1) {
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int u = 0; u < NT; u++)
#pragma unroll
                        for (int r = 0; r < 16; r++) isum[t][u][r] += (int)(Q6 ? 16.0f * acc[t][u][r] : acc[t][u][r]);
            }
            // one MFMA, then a few VALU instructions of the next step's operands, in turn
            __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
            for (int q = 0; q < MT * NT * ND; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VALU_EACH, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        build(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
        enter(std::integral_constant<int, 1>{});
        build(std::integral_constant<int, 8>{});
        step(std::integral_constant<int, 8>{});
        step(std::integral_constant<int, 9>{});
        step(std::integral_constant<int, 10>{});
        step(std::integral_constant<int, 11>{});
        step(std::integral_constant<int, 12>{});
        step(std::integral_constant<int, 13>{});
        step(std::integral_constant<int, 14>{});
        step(std::integral_constant<int, 15>{});

        // The f32 combine of the super-block, tile by tile; the min product
        // of a tile is issued while the one before is combined.
        v8h bmn[NT];
        if constexpr (MIN) {
#pragma unroll
            for (int u = 0; u < NT; u++) bmn[u] = min_operand<TYPE>(z[u]);
        }
        constexpr int NSM = MT * NT > 1 ? 2 : 1;
        v16f sm[NSM];
        auto min_product = [&](int q) {  // tile q = NT t + u
            if constexpr (MIN) {
                const v8h ab = *(const v8h *)(lds + L::BS + (32 * (q / NT) + l32) * 32 + 16 * h);
                const v16f zero = {0};
                sm[q % NSM] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ab, bmn[q % NT], zero, 0, 0, 0);
            }
        };
        min_product(0);
#pragma unroll
        for (int q = 0; q < MT * NT; q++) {
            const int t = q / NT, u = q % NT;
            if (q + 1 < MT * NT) min_product(q + 1);
            const float dw = f16_bits_to_f32(dd[u]) * (Q6 && !DUMP ? 16.0f : 1.0f), dmw = f16_bits_to_f32(dd[u] >> 16);
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const v4f dx4 = *(const v4f *)(lds + L::DX + 4 * (32 * t + 8 * g4 + 4 * h));
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int r = 4 * g4 + e;
                    const float S = DUMP ? (float)isum[DUMP ? t : 0][DUMP ? u : 0][r] : acc[t][u][r];
                    if constexpr (MIN)
                        yacc[t][u][r] = __builtin_fmaf(dx4[e], __builtin_fmaf(-dmw, sm[q % NSM][r], dw * S), yacc[t][u][r]);
                    else
                        yacc[t][u][r] = __builtin_fmaf(dw * dx4[e], S, yacc[t][u][r]);
                    if constexpr (DUMP) {
                        const int row = m0 + 32 * t + 8 * g4 + 4 * h + e;
                        const int col = 32 * NW * NT * tn + 32 * (NT * wave + u) + l32;
                        if (row < p.m && col < p.n) {
                            const int64_t o = ((int64_t)row * p.n + col) * ng + kb0 + i;
                            p.S[o] = isum[DUMP ? t : 0][DUMP ? u : 0][r];
                            p.Smin[o] = MIN ? (int)sm[q % NSM][r] : 0;
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    issue(0, std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    load_all<TYPE, NT>(v, rw, rwd, woff, doff, h, kb0);
    for (int i = 0; i < nit; i++) super_block(i);
    wait_vmcnt<0>();  // copies issued past the last super-block still write LDS

    float *y = p.y + (p.splits > 1 ? (int64_t)split * p.m * p.n : 0);
#pragma unroll
    for (int u = 0; u < NT; u++) {
        const int col = 32 * NW * NT * tn + 32 * (NT * wave + u) + l32;
        if (col >= p.n) continue;
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = m0 + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
                if (row < p.m) y[(int64_t)row * p.n + col] = yacc[t][u][r];
            }
    }
}

// ---------------------------------------------------------------------------
// Few rows (a tile of 32).  The time is the weight stream's, and a column's
// operands feed one MFMA each, so what fills the chip is many wavefronts with
// a short chain each: the NW wavefronts of a workgroup share 32 columns and
// take every NW-th super-block, with no LDS stage and no barrier in between
// (the activation fragments come from the L2 in whole lines, one super-block
// ahead like the weights), then add their sums through LDS in wavefront order.
// ---------------------------------------------------------------------------
template <int TYPE, int NW>
__device__ __forceinline__ void few_body(const KqParams &p, float *dx, float *red, int bid) {
    constexpr bool MIN = TYPE == TYPE_Q4_K || TYPE == TYPE_Q5_K || TYPE == TYPE_Q2_K;
    constexpr int ND = TYPE == TYPE_Q6_K ? 2 : 1;
    const int xcd = bid % NXCD, local = bid / NXCD;
    const int item = xcd * p.per_xcd + local;
    if (local >= p.per_xcd || item >= p.items) return;  // uniform over the workgroup
    const int tile = item / p.splits, split = item - tile * p.splits;
    const int tn = tile / p.ntm, m0 = 32 * (tile - tn * p.ntm);
    const int rows = min(32, p.m - m0);
    const int ng = p.ng, k = p.k;
    const int kb0 = split * p.kbs, kb1 = min(ng, kb0 + p.kbs);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;

    const rsrc_t rq = buf_rsrc(p.x16, (uint32_t)((int64_t)p.m * k * 2));
    const rsrc_t rbs = buf_rsrc(p.xbs, (uint32_t)((int64_t)p.m * (k / 16) * 2));
    const rsrc_t rnone = buf_rsrc(p.x16, 0u);
    const uint32_t qoff = l32 < rows ? (uint32_t)(m0 * k * 2 + (h * rows + l32) * 32) : BUF_OOB;
    const uint32_t bsoff = l32 < rows ? (uint32_t)(((m0 + l32) * (k / 16) + 8 * h) * 2) : BUF_OOB;
    const int sbytes = 64 * rows;  // of a sub-block
    const int nrb = (p.n + RB - 1) / RB, rb0 = 4 * tn, rb_here = min(4, nrb - rb0);
    const rsrc_t rw = buf_rsrc(p.w + (int64_t)rb0 * p.rb_stride, (uint32_t)(rb_here * p.rb_stride));
    constexpr int DB = TYPE == TYPE_Q2_K ? 4 : 2;  // bytes per d-plane entry
    const rsrc_t rwd = (TYPE == TYPE_Q6_K || TYPE == TYPE_Q2_K)
                           ? buf_rsrc((const uint8_t *)p.wd + (int64_t)rb0 * ng * RB * DB, (uint32_t)(rb_here * ng * RB * DB))
                           : rw;
    const uint32_t woff[1] = {(uint32_t)((l32 >> 3) * p.rb_stride + (l32 & 7) * 16)};
    const uint32_t doff[1] = {(uint32_t)((l32 >> 3) * ng * RB + (l32 & 7))};

    // first super-block's loads, then d of the tile's rows into LDS [super-block][row]
    W<TYPE> v[1];
    u32x4 a[16], bs = {0, 0, 0, 0};
    int b = kb0 + wave;
    {
        const bool live = b < kb1;
        const rsrc_t r4 = live ? rw : rnone, r5 = live ? rwd : rnone, r1 = live ? rq : rnone;
        load_all<TYPE, 1>(v, r4, r5, woff, doff, h, b);
#pragma unroll
        for (int f = 0; f < 16; f++) a[f] = ld16(r1, qoff, (b * 8 + f / 2) * sbytes + 16 * (f & 1));
        if constexpr (MIN) bs = ld16(live ? rbs : rnone, bsoff, b * 32);
    }
    for (int e = tid; e < 32 * (kb1 - kb0); e += 64 * NW) {
        const int r = e & 31, g = kb0 + (e >> 5);
        dx[e] = r < rows ? p.xd[(int64_t)(m0 + r) * ng + g] : 0.0f;
    }
    lds_barrier();

    v16f y;
#pragma unroll
    for (int r = 0; r < 16; r++) y[r] = 0.0f;
    uint32_t magic = 0x64006400u;
    opaque(magic);
    for (; b < kb1; b += NW) {  // uniform over the wavefront
        const int nb = b + NW;
        const bool more = nb < kb1;
        const rsrc_t r4 = more ? rw : rnone, r5 = more ? rwd : rnone, r1 = more ? rq : rnone;
        const Scales z = unpack_scales<TYPE>(v[0], h);
        const uint32_t dd = d_word<TYPE>(v[0]);
        load_head<TYPE>(v[0], r4, r5, woff[0], doff[0], nb);
        v16f acc;
        Consts<TYPE> c[Step<TYPE, 0>::SHARE];
        auto step = [&](auto JC) {
            constexpr int J = decltype(JC)::value;
            using P = Step<TYPE, J>;
            constexpr int F = 2 * P::S + P::I;
            if constexpr (P::I == 0) c[J % P::SHARE] = consts<TYPE>(z, P::S);
            v8h w[ND];
            operands<TYPE, P::S>(v[0], c[J % P::SHARE], P::I, magic, w);
#pragma unroll
            for (int g = 0; g < ND; g++) {
                const v16f zero = {0};
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[F]), w[g], J == 0 && g == 0 ? zero : acc, 0, 0, 0);
            }
            a[F] = ld16(r1, qoff, (nb * 8 + P::S) * sbytes + 16 * P::I);
            if constexpr (P::LAST) load_after<TYPE, P::S>(v[0], r4, woff[0], h, nb);
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
        step(std::integral_constant<int, 8>{});
        step(std::integral_constant<int, 9>{});
        step(std::integral_constant<int, 10>{});
        step(std::integral_constant<int, 11>{});
        step(std::integral_constant<int, 12>{});
        step(std::integral_constant<int, 13>{});
        step(std::integral_constant<int, 14>{});
        step(std::integral_constant<int, 15>{});
        v16f sm;
        if constexpr (MIN) {
            const v16f zero = {0};
            sm = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, bs), min_operand<TYPE>(z), zero, 0, 0, 0);
            bs = ld16(more ? rbs : rnone, bsoff, nb * 32);
        }
        const float dw = f16_bits_to_f32(dd) * (TYPE == TYPE_Q6_K ? 16.0f : 1.0f), dmw = f16_bits_to_f32(dd >> 16);
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
            const v4f dx4 = *(const v4f *)(dx + 32 * (b - kb0) + 8 * g4 + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = 4 * g4 + e;
                if constexpr (MIN) y[r] = __builtin_fmaf(dx4[e], __builtin_fmaf(-dmw, sm[r], dw * acc[r]), y[r]);
                else y[r] = __builtin_fmaf(dw * dx4[e], acc[r], y[r]);
            }
        }
    }

    // red [wavefront][row of 32][column of 32]
#pragma unroll
    for (int r = 0; r < 16; r++) red[(wave * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * 32 + l32] = y[r];
    lds_barrier();
    float *out = p.y + (p.splits > 1 ? (int64_t)split * p.m * p.n : 0);
    for (int e = tid; e < 32 * rows; e += 64 * NW) {
        const int r = e >> 5, col = 32 * tn + (e & 31);
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) sum += red[w * 1024 + e];
        if (col < p.n) out[(int64_t)(m0 + r) * p.n + col] = sum;
    }
}

template <int TYPE, int NW>
__global__ __launch_bounds__(64 * NW, 2) void few_kernel(KqParams p) {
    extern __shared__ __align__(16) uint8_t dyn[];  // [NW][32][32] f32, then d
    few_body<TYPE, NW>(p, (float *)(dyn + NW * 4096), (float *)dyn, (int)blockIdx.x);
}

template <int TYPE, int MT, int NT, int NW, int OCC, bool DUMP>
__global__ __launch_bounds__(64 * NW, OCC) void kernel(KqParams p) {
    __shared__ __align__(16) uint8_t lds[Lds<MT>::BYTES];
    body<TYPE, MT, NT, NW, DUMP>(p, lds, (int)blockIdx.x);
}

// A Q4_K weight and another of type T2 on the same activation: workgroups
// [0, g1) run the first (g1 a multiple of the XCD count, so its XCD mapping is
// kept), the rest the second.
template <int T2>
__global__ __launch_bounds__(256, 2) void pair_kernel(KqParams p1, KqParams p2, int g1) {
    __shared__ __align__(16) uint8_t lds[Lds<2>::BYTES];
    if ((int)blockIdx.x < g1) body<TYPE_Q4_K, 2, 1, 4, false>(p1, lds, (int)blockIdx.x);  // uniform
    else body<T2, 2, 1, 4, false>(p2, lds, (int)blockIdx.x - g1);
}

// The launch of one form; the integer dump runs the smallest.
template <int TYPE>
hipError_t launch(const KqParams &p, int form, bool dump, hipStream_t s) {
    const unsigned grid = (unsigned)(p.per_xcd * NXCD);
    if (dump) kernel<TYPE, 1, 1, 4, 1, true><<<grid, 256, 0, s>>>(p);
    else if (form == 0) kernel<TYPE, 1, 1, 4, 2, false><<<grid, 256, 0, s>>>(p);
    else if (form == 1) kernel<TYPE, 2, 1, 4, TYPE == TYPE_Q6_K ? 2 : 3, false><<<grid, 256, 0, s>>>(p);
    else if (form == 2) kernel<TYPE, 4, 1, 8, 2, false><<<grid, 512, 0, s>>>(p);
    else if (form == 3) kernel<TYPE, 4, 1, 4, 2, false><<<grid, 256, 0, s>>>(p);
    else if (form == 4) few_kernel<TYPE, 4><<<grid, 256, 4 * 4096 + 128 * p.kbs, s>>>(p);
    else if (form == 5) few_kernel<TYPE, 8><<<grid, 512, 8 * 4096 + 128 * p.kbs, s>>>(p);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace kq
#endif
}  // namespace aq
