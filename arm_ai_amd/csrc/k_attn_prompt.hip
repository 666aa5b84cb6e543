// k_attn_prompt.hip -- prompt attention on the f16 matrix cores, gfx950.
//
// The same attention as attn_prefill_kernel (k_attn.hip), which runs on the
// f32 matrix cores at a sixteenth of the f16 rate and is bound by them.  Here
// every f32 operand is split into two f16 values, x = hi + lo of 11 bits each,
// and a product of operands into three f16 products with f32 sums,
//   hi hi' + (hi lo' + lo hi');
// what is left out, lo lo', is 2^-22 of the product.  The matrix cores add 16
// products to a sum before they round it (2 on the f32 ones), so the error
// against 64 bits is smaller than before (see launch_attn_prompt).
//
// f16 has five exponent bits, so the operands are scaled by powers of two
// (exact): a query row by its largest value, a block of 32 keys by the block's
// (both to 2^14 .. 2^15), a block of 32 V rows to 2^11 .. 2^15 by a multiple
// of 2^4, and the probabilities by 2^12.  The score scale takes up the first
// two, the output sums are kept in units of the V block last added.
//
// What does not fit goes through plain f32, in the workgroups that would read it.
// attn_rows takes:
// - A query row or a block with a largest value outside 2^-50 .. 2^50 (2^-40 ..
//   2^40 for V) and not zero, or with an infinity or NaN.
// The f32 matrix cores (attn_f32: 2048 rows of 32/8 heads of 128 take 426 us, 391 in
// attn_prefill_kernel, 6900 through attn_rows) take:
// - A block of V with a row or a dim, not zero, whose largest value is below 2^-14
//   of the block's.  f16 ends at 2^-36 of that (2^-40 where it lies high in its
//   2^4), which is 2^-22 of the row's or the dim's: where 22 bits end as well.
// - A query row and a block of keys whose largest values have exponents that add
//   to more than SCORE_EXP: a term of a score could pass 2^15.  f16 ends at 2^-39
//   of a block's largest value, also for the rows far below it, and up to SCORE_EXP
//   that is at most 2^-18 of a base-2 score for each operand (all dims at the worst;
//   2^-24 for normal values beside one key of 2^15).  Scores stay below 2^23, so
//   that their rounding (an exponent is one fma, its reference was rounded) adds at
//   most 1/4 to an exponent, and a probability times 2^P_EXP stays an f16 number.
//
// 1) attn_planes_kernel: one workgroup per 32 keys and kv head rotates the
//    prompt's k rows into the cache, copies its v rows there, and writes the
//    split K and V of the block in the order of the MFMA operands, so that the
//    second kernel copies 1 KiB pieces into LDS and reads 16 bytes a lane.
// 2) attn_prompt_kernel.
#include "aq_internal.h"

#include <climits>
#include <cmath>

namespace aq {

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int KB = 32;                  // keys of a block, queries of a wavefront
constexpr int BAD_EXP = 1 << 20;        // a block for attn_rows
constexpr int WIDE_EXP = 1 << 19;       // a block of V for the f32 matrix cores
constexpr int SCORE_EXP = 16;           // most that the exponents of a query row and a K block add to
constexpr int P_EXP = 12;               // probabilities are kept times 2^12
constexpr float SLACK = 3.0f;           // ... and may exceed 1 by 2^SLACK (attn_prompt_kernel)

struct Prompt {
    const float *q, *k, *v, *cosb, *sinb;
    int64_t ldq, ldk, ldv;
    int index_pos, m, n_head, n_kv, max_seq, nblk;
    float *kc, *vc;
    // [kv head][block]{K hi, K lo, V hi, V lo} of 64 hd bytes each:
    // K [hd / 16][lane] 16 bytes: key lane % 32, dims 16 step + 8 (lane / 32) ..;
    // V [2][hd / 32][lane] 16 bytes: dim lane % 32, keys 16 step + 4 (lane / 32) ..
    // + 3 and the same + 8 .. (the order in which the scores hold the keys)
    uint8_t *planes;
    int2 *exps;  // [kv head][block]: exponents of K and V
    float *out;
};

__device__ __forceinline__ uint32_t mag(float x) { return f32_as_u32(x) & 0x7fffffffu; }

// Exponent by which values of magnitude up to `bits` are divided (zeros: the least).
template <int LIMIT>
__device__ __forceinline__ int scale_exp(uint32_t bits) {
    const int e = (int)(bits >> 23) - 127;
    if (bits == 0) return -LIMIT - 14;
    return e > LIMIT || e < -LIMIT ? BAD_EXP : e - 14;
}

__device__ __forceinline__ void split8(const float (&x)[8], v8h &hi, v8h &lo) {
#pragma unroll
    for (int i = 0; i < 8; i++) hi[i] = (_Float16)x[i];
#pragma unroll
    for (int i = 0; i < 8; i++) lo[i] = (_Float16)__builtin_fmaf((float)hi[i], -1.0f, x[i]);
}

// x 2^P_EXP = hi + lo: hi is hidden from the compiler, which would round x a
// second time for lo.
__device__ __forceinline__ void split_p(const float *x, v8h &hi, v8h &lo) {
    constexpr float UP = 1 << P_EXP;
    u32x4 h;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        const v2h t = {(_Float16)(x[2 * i] * UP), (_Float16)(x[2 * i + 1] * UP)};
        uint32_t u = __builtin_bit_cast(uint32_t, t);
        asm volatile("" : "+v"(u));
        h[i] = u;
    }
    hi = __builtin_bit_cast(v8h, h);
#pragma unroll
    for (int i = 0; i < 8; i++) lo[i] = (_Float16)__builtin_fmaf(x[i], UP, -(float)hi[i]);
}

// v of this lane and of lane ^ 32, combined
__device__ __forceinline__ float max_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(f32_as_u32(v), f32_as_u32(v), false, false);
    return fmaxf(u32_as_f32(r[0]), u32_as_f32(r[1]));
}
__device__ __forceinline__ float sum_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(f32_as_u32(v), f32_as_u32(v), false, false);
    return u32_as_f32(r[0]) + u32_as_f32(r[1]);
}

// The largest of a over the lanes of a wavefront, for eight values a lane: those of
// a[2 q] and a[2 q + 1] in the lanes of 16-lane row q.
__device__ __forceinline__ void wave_max8(const uint32_t (&a)[8], uint32_t (&r)[2]) {
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {  // lanes 0 .. 31: a[i], 32 .. 63: a[i + 4]
        const auto t = __builtin_amdgcn_permlane32_swap(a[i], a[i + 4], false, false);
        h[i] = max((uint32_t)t[0], (uint32_t)t[1]);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {  // rows 0, 2: h[i], 1, 3: h[i + 2]
        const auto t = __builtin_amdgcn_permlane16_swap(h[i], h[i + 2], false, false);
        uint32_t v = max((uint32_t)t[0], (uint32_t)t[1]);
        v = max(v, (uint32_t)dpp_i<DPP_QUAD_XOR1>((int)v));
        v = max(v, (uint32_t)dpp_i<DPP_QUAD_XOR2>((int)v));
        v = max(v, (uint32_t)dpp_i<DPP_HALF_MIRROR>((int)v));
        r[i] = max(v, (uint32_t)dpp_i<DPP_ROW_MIRROR>((int)v));
    }
}

// blockIdx.z 0: K, 1: V of the block.  Bound by latency, so every load is issued
// before the first is used (keys past the end: the last one's, zeroed after).
template <int HD>
__global__ __launch_bounds__(256) void attn_planes_kernel(Prompt p) {
    constexpr int NP = HD / 64;  // pieces of eight values per thread
    __shared__ uint32_t smax[4];
    __shared__ u32x4 img[2][HD * 4];  // K hi, lo; V: the largest of each dim and key
    uint32_t(*const dmax)[HD] = (uint32_t(*)[HD])img, (*const kmax)[32] = (uint32_t(*)[32])(dmax + 4);  // [eight keys], [64 dims]
    const int b = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, kend = p.index_pos + p.m;
    const bool is_v = blockIdx.z;
    int2 *const ex = p.exps + (int64_t)g * p.nblk + b;
    uint8_t *const blk = p.planes + ((int64_t)g * p.nblk + b) * (256 * HD);

    float x[NP][8];
    uint32_t top = 0;
    if (!is_v) {  // consecutive threads along a row
        float c[NP][4], sn[NP][4];
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int piece = tid + 256 * i, key = min(KB * b + piece / (HD / 8), kend - 1), d0 = piece % (HD / 8) * 8;
            const float *src = key < p.index_pos ? p.kc + ((int64_t)g * p.max_seq + key) * HD + d0
                                                 : p.k + (int64_t)(key - p.index_pos) * p.ldk + (int64_t)g * HD + d0;
            const float *cr = p.cosb + (int64_t)key * (HD / 2) + d0 / 2, *sr = p.sinb + (int64_t)key * (HD / 2) + d0 / 2;
#pragma unroll
            for (int j = 0; j < 8; j++) x[i][j] = src[j];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                c[i][j] = cr[j];
                sn[i][j] = sr[j];
            }
        }
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int piece = tid + 256 * i, key = KB * b + piece / (HD / 8), d0 = piece % (HD / 8) * 8;
            if (key >= p.index_pos && key < kend) {
                float4 *row = (float4 *)(p.kc + ((int64_t)g * p.max_seq + key) * HD + d0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float x0 = x[i][2 * j], x1 = x[i][2 * j + 1];
                    x[i][2 * j] = x0 * c[i][j] - x1 * sn[i][j];
                    x[i][2 * j + 1] = x0 * sn[i][j] + x1 * c[i][j];
                }
#pragma unroll
                for (int h = 0; h < 2; h++) row[h] = make_float4(x[i][4 * h], x[i][4 * h + 1], x[i][4 * h + 2], x[i][4 * h + 3]);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (key >= kend) x[i][j] = 0.0f;
                top = max(top, mag(x[i][j]));
            }
        }
    } else {  // consecutive threads along a row, eight keys each
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int piece = tid + 256 * i, dim = piece % HD, st = piece / HD >> 1, hh = piece / HD & 1;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int key = min(KB * b + 16 * st + 4 * hh + (e & 3) + 8 * (e >> 2), kend - 1);
                const float *src = key < p.index_pos ? p.vc + ((int64_t)g * p.max_seq + key) * HD
                                                     : p.v + (int64_t)(key - p.index_pos) * p.ldv + (int64_t)g * HD;
                x[i][e] = src[dim];
            }
        }
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int piece = tid + 256 * i, dim = piece % HD, st = piece / HD >> 1, hh = piece / HD & 1;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int key = KB * b + 16 * st + 4 * hh + (e & 3) + 8 * (e >> 2);
                if (key >= p.index_pos && key < kend) p.vc[((int64_t)g * p.max_seq + key) * HD + dim] = x[i][e];
                if (key >= kend) x[i][e] = 0.0f;
            }
            uint32_t a[8], r[2], of_dim = 0;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                a[e] = mag(x[i][e]);
                of_dim = max(of_dim, a[e]);
            }
            top = max(top, of_dim);
            dmax[2 * st + hh][dim] = of_dim;
            wave_max8(a, r);
            const int e = (tid & 63) >> 4 << 1;  // of a lane's row: values e and e + 1
            if ((tid & 15) < 2) kmax[HD == 128 ? dim >> 6 : 0][16 * st + 4 * hh + (e & 3) + (tid & 15) + 8 * (e >> 2)] = r[tid & 1];
        }
    }
#pragma unroll
    for (int o = 1; o < 64; o *= 2) top = max(top, (uint32_t)__shfl_xor((int)top, o));
    if ((tid & 63) == 0) smax[tid >> 6] = top;
    __syncthreads();
    top = max(max(smax[0], smax[1]), max(smax[2], smax[3]));
    int e = is_v ? scale_exp<40>(top) : scale_exp<50>(top);
    if (is_v) {  // every wavefront looks at every dim and key: no second barrier
        bool low = false;
#pragma unroll
        for (int i = tid & 63; i < HD + 32; i += 64) {
            const uint32_t of = i < HD ? max(max(dmax[0][i], dmax[1][i]), max(dmax[2][i], dmax[3][i]))
                                       : max(kmax[0][i - HD], HD == 128 ? kmax[1][i - HD] : 0u);
            low |= of != 0 && u32_as_f32(of) < u32_as_f32(top) * 0x1p-14f;
        }
        if (e != BAD_EXP) e = __any(low) ? WIDE_EXP : top == 0 ? 0 : (e + 3) & ~3;
    }
    if (tid == 0) *(is_v ? &ex->y : &ex->x) = e;
    if (e >= WIDE_EXP) return;  // uniform over the workgroup; the block's planes are not read

#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int piece = tid + 256 * i;
        v8h hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) x[i][j] = ldexpf(x[i][j], -e);
        split8(x[i], hi, lo);
        if (!is_v) {  // into operand order through LDS
            const int key = piece / (HD / 8), d8 = piece % (HD / 8), at = (d8 >> 1) * 64 + (d8 & 1) * 32 + key;
            img[0][at] = __builtin_bit_cast(u32x4, hi);
            img[1][at] = __builtin_bit_cast(u32x4, lo);
        } else {
            const int dim = piece % HD, sh = piece / HD;
            const int at = ((sh >> 1) * (HD / 32) + dim / 32) * 64 + (sh & 1) * 32 + dim % 32;
            ((u32x4 *)(blk + 128 * HD))[at] = __builtin_bit_cast(u32x4, hi);
            ((u32x4 *)(blk + 192 * HD))[at] = __builtin_bit_cast(u32x4, lo);
        }
    }
    if (is_v) return;  // uniform over the workgroup
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * NP; i++) ((u32x4 *)blk)[tid + 256 * i] = (&img[0][0])[tid + 256 * i];
}

// The tile's rows in plain f32, where an operand does not fit the split: the
// wavefronts take the rows in turn, a lane per key for the scores, the lanes
// along the dims for the output.  Every sum in four chains, as one of hd or of all
// the keys rounds twice as far from 64 bits as attn_prefill_kernel does.
template <int HD>
__device__ void attn_rows(const Prompt &p, int h, int kvh, int qb, int rows, int first, int step, float *qs, float *ps) {
    const int lane = threadIdx.x & 63;
    const float *kh = p.kc + (int64_t)kvh * p.max_seq * HD, *vh = p.vc + (int64_t)kvh * p.max_seq * HD;
    const float sc2 = 1.4426950408889634f / sqrtf((float)HD);
    for (int r = first; r < rows; r += step) {
        const int qpos = p.index_pos + qb + r;
        const float *qr = p.q + (int64_t)(qb + r) * p.ldq + (int64_t)h * HD;
        if (lane < HD / 2) {
            const float a = qr[2 * lane], b = qr[2 * lane + 1];
            const float c = p.cosb[(int64_t)qpos * (HD / 2) + lane], sn = p.sinb[(int64_t)qpos * (HD / 2) + lane];
            qs[2 * lane] = a * c - b * sn;
            qs[2 * lane + 1] = a * sn + b * c;
        }
        __builtin_amdgcn_wave_barrier();
        float mrun = -INFINITY, lrun = 0.0f, acc[HD / 64][4];
        for (int i = 0; i < HD / 16; i++) acc[i / 4][i % 4] = 0.0f;
        for (int k0 = 0; k0 <= qpos; k0 += 64) {
            const int key = k0 + lane;
            float s = -INFINITY;
            if (key <= qpos) {
                const float4 *kr = (const float4 *)(kh + (int64_t)key * HD);
                float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                for (int d = 0; d < HD / 4; d++) {
                    const float4 t = kr[d];
                    c.x = __builtin_fmaf(t.x, qs[4 * d], c.x);
                    c.y = __builtin_fmaf(t.y, qs[4 * d + 1], c.y);
                    c.z = __builtin_fmaf(t.z, qs[4 * d + 2], c.z);
                    c.w = __builtin_fmaf(t.w, qs[4 * d + 3], c.w);
                }
                s = ((c.x + c.y) + (c.z + c.w)) * sc2;
            }
            float bm = s;
            for (int o = 1; o < 64; o *= 2) bm = fmaxf(bm, __shfl_xor(bm, o));
            const float mnew = fmaxf(mrun, bm), msafe = mnew == -INFINITY ? 0.0f : mnew;
            const float scale = __builtin_amdgcn_exp2f(mrun - msafe), e = __builtin_amdgcn_exp2f(s - msafe);
            float sum = e;
            for (int o = 1; o < 64; o *= 2) sum += __shfl_xor(sum, o);
            lrun = __builtin_fmaf(lrun, scale, sum);
            mrun = mnew;
            __builtin_amdgcn_wave_barrier();
            ps[lane] = e;
            __builtin_amdgcn_wave_barrier();
            for (int i = 0; i < HD / 16; i++) acc[i / 4][i % 4] *= scale;
            for (int kk = 0; kk < 64 && k0 + kk <= qpos; kk += 4) {
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (k0 + kk + c <= qpos)
                        for (int d = 0; d < HD / 64; d++)
                            acc[d][c] = __builtin_fmaf(ps[kk + c], vh[(int64_t)(k0 + kk + c) * HD + 64 * d + lane], acc[d][c]);
            }
        }
        for (int d = 0; d < HD / 64; d++)
            p.out[(int64_t)(qb + r) * p.n_head * HD + (int64_t)h * HD + 64 * d + lane] =
                ((acc[d][0] + acc[d][1]) + (acc[d][2] + acc[d][3])) / lrun;
        __builtin_amdgcn_wave_barrier();
    }
}

// The key blocks first, first + step, .. of a unit on the f32 matrix cores, its
// operands from the cache: the running max, sum and output (times 1).
template <int HD>
__device__ __forceinline__ void attn_f32(const Prompt &p, int kvh, int qb, int qpos, int first, int step, const float (&qx)[HD / 16][8],
                                         float &mrun, float &lrun, v16f (&o)[HD / 32]) {
    const int lane = threadIdx.x & 63, j = lane & 31, hh = lane >> 5, last = p.index_pos + p.m - 1;
    const float *kh = p.kc + (int64_t)kvh * p.max_seq * HD, *vh = p.vc + (int64_t)kvh * p.max_seq * HD;
    const float sc2 = 1.4426950408889634f / sqrtf((float)HD);
    for (int k0 = first * KB; k0 <= min(last, p.index_pos + qb + KB - 1); k0 += step * KB) {
        const float4 *kr = (const float4 *)(kh + (int64_t)min(k0 + j, last) * HD + 8 * hh);
        v16f s[2];
#pragma unroll
        for (int r = 0; r < 16; r++) s[0][r] = s[1][r] = 0.0f;
#pragma unroll
        for (int st = 0; st < HD / 16; st++) {
            const float4 a = kr[4 * st], b = kr[4 * st + 1];
            const float kx[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 8; i++) s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[i], qx[st][i], s[i & 1], 0, 0, 0);
        }
        float x[16], bm = -INFINITY, sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            x[r] = k0 + 8 * (r >> 2) + 4 * hh + (r & 3) > qpos ? -INFINITY : (s[0][r] + s[1][r]) * sc2;
            bm = fmaxf(bm, x[r]);
        }
        const float mnew = fmaxf(mrun, max_halves(bm)), msafe = mnew == -INFINITY ? 0.0f : mnew;
        const float scale = __builtin_amdgcn_exp2f(mrun - msafe);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            x[r] = __builtin_amdgcn_exp2f(x[r] - msafe);
            sum += x[r];
        }
        lrun = __builtin_fmaf(lrun, scale, sum_halves(sum));
        mrun = mnew;
#pragma unroll
        for (int b = 0; b < HD / 32; b++) {
#pragma unroll
            for (int r = 0; r < 16; r++) o[b][r] *= scale;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = min(k0 + 8 * (r >> 2) + 4 * hh + (r & 3), last);
                o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(vh[(int64_t)key * HD + 32 * b + j], x[r], o[b], 0, 0, 0);
            }
        }
    }
}

// 2) One workgroup of QW x KG wavefronts takes QW units of a kv head, a unit
//    being 32 query rows of one of its query heads; KG wavefronts share a unit,
//    wavefront group w taking the key blocks w, w + KG, ..., each with a running
//    max, sum and output per query row, combined through LDS at the end.
//    Scores are formed transposed, S^T[key][query] = K . Q^T: lane (j, hh)
//    holds query j against 16 keys, so the softmax of a row needs only its own
//    registers and lane ^ 32, and those registers are the operand of
//    O^T[dim][query] += V^T . P^T after the split.
//    K and V of a block are copied to LDS once for the QW wavefronts that read
//    it.  DB 0: one stage, V copied during the scores and the softmax, the next
//    K during P . V, two barriers a block, and two workgroups of four
//    wavefronts to a CU, which run out of step; DB 1: two stages, the next block
//    copied during this one, one barrier.
template <int HD, int QW, int KG, int DB>
__global__ __launch_bounds__(64 * QW * KG, 2) void attn_prompt_kernel(Prompt p) {
    constexpr int NB = HD / 32, NS = HD / 16, BLK = 256 * HD;  // BLK: bytes of a block's planes
    constexpr int COPIES = HD / 8 / QW;                        // 1 KiB pieces of K (of V) per wavefront
    // [KG][1 + DB]{K hi, lo, V hi, lo}: dynamic, as the compiler waits for every copy
    // in flight before it reads a static array (15 % of the time of the single stage)
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ float sml[KG][QW][2][KB];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qw = wave % QW, kg = wave / QW, j = lane & 31, hh = lane >> 5;
    const int rep = p.n_head / p.n_kv, ntq = (p.m + KB - 1) / KB, units = ntq * rep;
    const int rank = blockIdx.x / p.n_kv, kvh = blockIdx.x % p.n_kv;
    const int u0 = ((units + QW - 1) / QW - 1 - rank) * QW;  // the units with the most keys first
    const int unit = min(u0 + qw, units - 1);                // (a spare wavefront repeats the last, and stores nothing)
    const int qb = unit / rep * KB, h = kvh * rep + unit % rep, rows = min(KB, p.m - qb);
    const int last = min(u0 + QW, units) - 1;
    const int nkb = (p.index_pos + min(p.m, (last / rep + 1) * KB) + KB - 1) / KB, nit = (nkb + KG - 1) / KG;
    const int qpos = p.index_pos + qb + j;

    const rsrc_t rp = buf_rsrc(p.planes + (int64_t)kvh * p.nblk * BLK, (uint32_t)((int64_t)p.nblk * BLK));
    const rsrc_t rnone = buf_rsrc(p.planes, 0u);
    auto issue = [&](int it, int off) {  // off: 0 K, BLK / 2 V
        const int blk = it * KG + kg;
#pragma unroll
        for (int c = 0; c < COPIES; c++) {
            const int at = off + 1024 * (qw * COPIES + c);
            buf_to_lds16(blk < nkb ? rp : rnone, lds + (kg * (1 + DB) + (DB ? it & 1 : 0)) * BLK + at, 16u * lane,
                         blk < nkb ? blk * BLK + at : 0);
        }
    };
    issue(0, 0);
    if constexpr (DB) issue(0, BLK / 2);

    // this lane's query fragment, rotated at qpos: dims 16 step + 8 hh ..
    float qx[NS][8];
    {
        const int row = qb + min(j, rows - 1);  // (spare lanes repeat the last row; nothing of theirs is stored)
        const int pos = p.index_pos + row;
        const float *qr = p.q + (int64_t)row * p.ldq + (int64_t)h * HD + 8 * hh;
        const float *cr = p.cosb + (int64_t)pos * (HD / 2) + 4 * hh, *sr = p.sinb + (int64_t)pos * (HD / 2) + 4 * hh;
        float c[NS][4], sn[NS][4];
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int i = 0; i < 8; i++) qx[s][i] = qr[16 * s + i];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                c[s][i] = cr[8 * s + i];
                sn[s][i] = sr[8 * s + i];
            }
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float a = qx[s][2 * i], b = qx[s][2 * i + 1];
                qx[s][2 * i] = a * c[s][i] - b * sn[s][i];
                qx[s][2 * i + 1] = a * sn[s][i] + b * c[s][i];
            }
    }
    uint32_t qmax = 0;
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int i = 0; i < 8; i++) qmax = max(qmax, mag(qx[s][i]));
    qmax = max(qmax, (uint32_t)__shfl_xor((int)qmax, 32));
    const int eq = scale_exp<50>(qmax);
    const int2 *ex = p.exps + (int64_t)kvh * p.nblk;
    int bad = eq == BAD_EXP, wide = bad;
    const int eqm = scale_exp<50>(f32_as_u32(wave_max_f(u32_as_f32(qmax))));  // of the wavefront's rows
    for (int b = lane; b < nkb; b += 64) {
        const int2 e = ex[b];
        bad |= max(e.x, e.y) == BAD_EXP;
        wide |= e.x + eqm > SCORE_EXP - 28 || e.y >= WIDE_EXP;
    }
    float mrun = -INFINITY, lrun = 0.0f;
    int eo = 0;  // the output is in units of 2^eo
    v16f o[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[b][r] = 0.0f;
    if (__syncthreads_or(wide)) {  // uniform; the copies in flight end before LDS is written again
        wait_vmcnt<0>();
        if (__syncthreads_or(bad)) {
            float *own = (float *)(lds + wave * 1024);
            if (u0 + qw < units) attn_rows<HD>(p, h, kvh, qb, rows, kg, KG, own, own + HD);
            return;
        }
        attn_f32<HD>(p, kvh, qb, qpos, kg, KG, qx, mrun, lrun, o);
        eo = P_EXP;
    } else {
        v8h qh[NS], ql[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int i = 0; i < 8; i++) qx[s][i] = ldexpf(qx[s][i], -eq);
            split8(qx[s], qh[s], ql[s]);
        }

        const float scq = ldexpf(1.4426950408889634f / sqrtf((float)HD), eq);  // log2(e) / sqrt(hd)
        v8h ph[2], pl[2];
        // a block's exponents, loaded a block ahead: before the copies, so that
        // waiting for them does not wait for those
        int2 e, en = ex[min(kg, nkb - 1)];
        auto next_exps = [&](int it) {
            e = make_int2(__builtin_amdgcn_readfirstlane(en.x), __builtin_amdgcn_readfirstlane(en.y));
            en = ex[min((it + 1) * KG + kg, nkb - 1)];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto scores = [&](int blk, const uint8_t *kst) {
            const int k0 = blk * KB;
            v16f s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.0f;
            // the small products first, then the large: one chain, K hi kept
            v8h kh[NS], kl[2];
            auto load = [&](int st) {
                kl[st & 1] = *(const v8h *)(kst + 64 * HD + (st * 64 + lane) * 16);
                kh[st] = *(const v8h *)(kst + (st * 64 + lane) * 16);
            };
            load(0);
#pragma unroll
            for (int st = 0; st < NS; st++) {
                if (st + 1 < NS) load(st + 1);
                __builtin_amdgcn_sched_barrier(0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl[st & 1], qh[st], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh[st], ql[st], s, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int st = 0; st < NS; st++) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh[st], qh[st], s, 0, 0, 0);
            // lane (j, hh) register r: query j, key k0 + 8 (r / 4) + 4 hh + r % 4
            if (k0 + KB - 1 > p.index_pos + qb) {  // the block holds keys past some row
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (k0 + 8 * (r >> 2) + 4 * hh + (r & 3) > qpos) s[r] = -INFINITY;
            }
            float bm = s[0];
#pragma unroll
            for (int r = 1; r < 16; r++) bm = fmaxf(bm, s[r]);
            bm = max_halves(bm);
            const float sc = ldexpf(scq, e.x);
            bm *= sc;
            // the reference follows the max only where it lags by more than
            // SLACK: the sums then need no rescaling in most blocks
            const float mnew = bm > mrun + SLACK ? bm : mrun;
            const float msafe = mnew == -INFINITY ? 0.0f : mnew;  // a block wholly past this query
            const float scale = __builtin_amdgcn_exp2f(mrun - msafe);
            float x[16], sum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                x[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], sc, -msafe));
                sum += x[r];
            }
            lrun = __builtin_fmaf(lrun, scale, sum_halves(sum));
            mrun = mnew;
#pragma unroll
            for (int st = 0; st < 2; st++) split_p(x + 8 * st, ph[st], pl[st]);
            const float os = ldexpf(scale, eo - e.y);
            eo = e.y;
            if (__any(os != 1.0f)) {
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[b][r] *= os;
            }
        };
        auto values = [&](const uint8_t *vst) {
            v8h vh[2], vl[2];
            auto load = [&](int i) {  // fragment i: [2][NB]
                vl[i & 1] = *(const v8h *)(vst + 64 * HD + (i * 64 + lane) * 16);
                vh[i & 1] = *(const v8h *)(vst + (i * 64 + lane) * 16);
            };
            load(0);
#pragma unroll
            for (int i = 0; i < 2 * NB; i++) {
                const int st = i / NB, b = i % NB;
                if (i + 1 < 2 * NB) load(i + 1);
                __builtin_amdgcn_sched_barrier(0);
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[i & 1], ph[st], o[b], 0, 0, 0);
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[i & 1], pl[st], o[b], 0, 0, 0);
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[i & 1], ph[st], o[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto live = [&](int it) {  // uniform over the wavefront
            const int blk = it * KG + kg;
            return blk < nkb && blk * KB <= p.index_pos + qb + KB - 1;
        };
        if constexpr (DB) {
            for (int it = 0; it < nit; it++) {
                wait_vmcnt<0>();  // this block's K and V
                lds_barrier();    // everyone's, and everyone has read the last block's
                next_exps(it);
                issue(it + 1, 0);
                issue(it + 1, BLK / 2);
                const uint8_t *const base = lds + (kg * 2 + (it & 1)) * BLK;
                if (live(it)) {
                    scores(it * KG + kg, base);
                    values(base + BLK / 2);
                }
            }
        } else {
            for (int it = 0; it < nit; it++) {
                wait_vmcnt<0>();  // this block's K
                lds_barrier();    // everyone's, and everyone has read the last block's V
                next_exps(it);
                issue(it, BLK / 2);
                if (live(it)) scores(it * KG + kg, lds + kg * BLK);
                wait_vmcnt<0>();  // this block's V
                lds_barrier();    // everyone's, and everyone has read K
                issue(it + 1, 0);
                if (live(it)) values(lds + kg * BLK + BLK / 2);
            }
        }
        wait_vmcnt<0>();  // (copies past the last block write zeros)
    }

    // combine the KG key ranges: M = max m, out = sum e^(m - M) o / sum e^(m - M) l
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[b][r] = ldexpf(o[b][r], eo - P_EXP);
    if constexpr (KG > 1) {
        if (hh == 0) {
            sml[kg][qw][0][j] = mrun;
            sml[kg][qw][1][j] = lrun;
        }
        __syncthreads();  // the stages are free
        float *so = (float *)lds;
        if (kg > 0) {
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) so[(((kg - 1) * QW + qw) * NB * 16 + 16 * b + r) * 64 + lane] = o[b][r];
        }
        __syncthreads();
        if (kg > 0) return;
        float M = mrun;
#pragma unroll
        for (int w = 1; w < KG; w++) M = fmaxf(M, sml[w][qw][0][j]);
        const float Ms = M == -INFINITY ? 0.0f : M, e0 = __builtin_amdgcn_exp2f(mrun - Ms);
        lrun *= e0;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[b][r] *= e0;
#pragma unroll
        for (int w = 1; w < KG; w++) {
            const float ew = __builtin_amdgcn_exp2f(sml[w][qw][0][j] - Ms);
            lrun = __builtin_fmaf(ew, sml[w][qw][1][j], lrun);
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    o[b][r] = __builtin_fmaf(ew, so[(((w - 1) * QW + qw) * NB * 16 + 16 * b + r) * 64 + lane], o[b][r]);
        }
    }
    if (u0 + qw >= units || j >= rows) return;
    float *orow = p.out + (int64_t)(qb + j) * p.n_head * HD + (int64_t)h * HD + 4 * hh;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
            *(float4 *)(orow + 32 * b + 2 * r) =
                make_float4(o[b][r] / lrun, o[b][r + 1] / lrun, o[b][r + 2] / lrun, o[b][r + 3] / lrun);
}

template <int HD, int QW, int KG, int DB>
hipError_t run(const Prompt &p, hipStream_t s) {
    constexpr int LDS = (1 + DB) * KG * 256 * HD;
    if constexpr (LDS > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void *)attn_prompt_kernel<HD, QW, KG, DB>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return e;
    }
    const int64_t units = (int64_t)((p.m + KB - 1) / KB) * (p.n_head / p.n_kv);
    if (units * p.n_kv > INT_MAX) return hipErrorNotSupported;
    attn_planes_kernel<HD><<<dim3((unsigned)p.nblk, (unsigned)p.n_kv, 2), 256, 0, s>>>(p);
    attn_prompt_kernel<HD, QW, KG, DB><<<(unsigned)((units + QW - 1) / QW * p.n_kv), 64 * QW * KG, LDS, s>>>(p);
    return hipGetLastError();
}

}  // namespace

size_t attn_prompt_workspace_bytes(int64_t kend, int64_t n_kv, int64_t hd) {
    // The split costs a pass over the keys and a longer start: 16 rows and 16
    // keys of 32/4 heads of 64 take 9.1 us on the f32 cores, 10.4 here; 256 rows
    // 13.6 and 13.7, 300 rows 17.3 and 15.5; of 32/8 heads of 128, 128 rows 17.5
    // and 17.5, 256 rows 24.5 and 21.5.
    if (kend * hd <= 20480) return (size_t)-1;
    const int64_t nblk = (kend + KB - 1) / KB;
    if (nblk * 256 * hd >= ((int64_t)1 << 31)) return (size_t)-1;  // (32-bit offsets into a kv head's planes)
    return (size_t)(n_kv * nblk) * (size_t)(256 * hd + sizeof(int2));
}

// The forms (QW, KG), with the first kernel (before its range checks, 0.4 us a
// call); in parentheses attn_prefill_kernel:
//   heads   hd   rows   at     (1, 4)  (2, 2)  (4, 2), two stages
//   32/8    128  2048   0      222.7   131.3   120.7 us  (391)
//   32/8    128  1400   0      132.5    81.0    75.6     (211)
//   32/8    128  1024   0       85.6    54.5    58.2     (126)
//   32/8    128  512    0       39.0    30.6    39.5     (49.6)
//   32/8    128  128    1900    54.4    68.9    85.0     (89)
//   32/4    64   2048   0       98      74.4    75       (216)
//   32/4    64   512    0       19.9    20.0    23.9     (25.7)
//   9/3     64   2048   0       42.9    54.7    63.7     (73.7)
//   32/4    64   128    900     23.7    29.4    35       (31.2)
// Error against 64 bits: 2.2e-7 at the first, 2.7e-7 before; smaller in every row.
// Bound by the f16 matrix cores: the 48 MFMAs of a unit and block at hd 128 take
// 1.77 us of a SIMD with all CUs busy, 37 ns each, and 1.5 us with neither copies
// nor exponentials (a large f16 product reaches 24 ns); a wavefront alone takes
// 1.4 us.  Interleaving the softmax of one block with the products of its
// neighbours in one wavefront was no faster (128 us) and its sums less exact.
hipError_t launch_attn_prompt(const float *q, int64_t ldq, const float *k, int64_t ldk, const float *v, int64_t ldv,
                              const float *cosb, const float *sinb, int64_t index_pos, int64_t m, float *kc, float *vc,
                              int64_t n_head, int64_t n_kv, int64_t hd, int64_t max_seq, float *out, void *ws,
                              size_t ws_bytes, hipStream_t s) {
    if (attn_prompt_workspace_bytes(index_pos + m, n_kv, hd) > ws_bytes || !ws || n_kv > 65535) return hipErrorNotSupported;
    Prompt p{q, k, v, cosb, sinb, ldq, ldk, ldv, (int)index_pos, (int)m, (int)n_head, (int)n_kv, (int)max_seq,
             (int)((index_pos + m + KB - 1) / KB), kc, vc, (uint8_t *)ws, nullptr, out};
    p.exps = (int2 *)(p.planes + n_kv * p.nblk * 256 * hd);
    const int64_t units = (m + KB - 1) / KB * n_head;
    // (1, 4) where the units do not fill the chip, or the chains are long
    if (units <= 256 || (hd == 64 && units <= 768 && units <= 16 * p.nblk))
        return hd == 64 ? run<64, 1, 4, 0>(p, s) : run<128, 1, 4, 0>(p, s);
    if (hd == 64) return run<64, 2, 2, 0>(p, s);
    return units <= 1280 ? run<128, 2, 2, 0>(p, s) : run<128, 4, 2, 1>(p, s);
}

}  // namespace aq
