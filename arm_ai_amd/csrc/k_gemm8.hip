// k_gemm8.hip -- prefill GEMM for Q8_0 weights (and Q4_0 / Q5_0 on their
// expanded copy) on the int8 matrix cores, gfx950.
//
// Replaces the M-row loop of candle-core 0.8.4 k_quants::matmul<BlockQ8_0>
// at prefill (native/arm_ai_nif/src/llama_candle.rs:93; the activation is
// quantised to Q8_0 blocks, BlockQ8_0::vec_dot per 32-element block):
//   y[m][n] = sum_b (f32)S_b * f16(d_w[n,b]) * f16(d_x[m,b]),
//   S_b = sum_{e in b} qw_e * qx_e  (exact in i32).
//
// One v_mfma_i32_32x32x32_i8 covers one block (K = 32) of a 32 x 32 tile.
// The per-block scaling is the whole cost beyond the MFMA, so it is cut to
// two f32 fmas per output:
//   - The MFMA does not start from zero but from the constant C0 = 0x4B400000,
//     the bits of 1.5 * 2^23.  Its i32 result C0 + S, read as f32, is exactly
//     1.5 * 2^23 + S (|S| <= 32 * 128 * 127 < 2^22 keeps the exponent fixed):
//     the int -> float conversion is free.
//   - t = fma(C0 + S, d_w, -1.5 * 2^23 * d_w) rounds S * d_w once, so it is
//     bit-identical to candle's (f32)S * d_w (the constant product is exact:
//     d_w has an 11-bit significand).
//   - acc = fma(t, d_x, acc): one rounding fewer than candle's mul-then-add
//     (within the f32 tolerance of the output; the integer sums are bit-exact,
//     see the dump variant).
// 32 fmas against one MFMA of 32 cycles bind it to VALU issue whatever the
// tile; what a form has to do is to keep two or three wavefronts per SIMD
// issuing.
//
// A lane's weight operand is a 16-byte piece of its own column (column l % 32,
// half h = l / 32: piece 2 j + h of block j), loaded straight into registers
// one group of eight blocks ahead, each again as soon as it is used.  The
// activation comes from planes in the order of the MFMA operands
// (q8_at, dt_at): a block of 32 rows is 1 KiB in lane order.
//
// Tiled form: a workgroup of four wavefronts owns 64 rows x 128 columns, each
// wavefront 32 columns and all the rows; the activation of half a group (four
// blocks) at a time goes global -> LDS by buffer-to-LDS copies, into two
// stages, one half ahead; one s_waitcnt vmcnt and one barrier per half.  The
// eight blocks of a group are summed apart and added to the output once: 2 %
// more fmas' time, and the error against 64 bits stays below that of the
// 128 x 128 tiles before (8.5e-8 against 9.6e-8 at 333 x 4096 x 4096, where one
// chain over K had 1.5e-7); 240 VGPRs, two wavefronts per SIMD.
// 333 x 4096 x 4096: 40.6 us before, 32.6 now (40.9 and 33.2 on another card); 512 x
// 14336 x 4096: 131.6, 105.8; 512 x 5632 x 2048: 43.5, 31.6 (with the quantizer).
// Few-row form (a tile of 32): the wavefronts of a workgroup share 32 columns
// and take every fourth or eighth group each, with no stage and no barrier in
// between, then add their sums through LDS in wavefront order.
// Work items (tile, K split) are dealt so that the row tiles and splits of
// one column tile run on one XCD; split-K partials are added in split order by
// launch_reduce.
#include "aq_internal.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace aq {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int G8XCD = 8;
constexpr int32_t C0 = 0x4B400000;  // bits of 1.5 * 2^23
constexpr float C0F = 12582912.0f;  // 1.5 * 2^23
constexpr int PIECES = 17;          // of a group: 2 j, 2 j + 1 the quants of block j, 16 the eight f16 d

struct Gemm8Params {
    const uint8_t *w;   // row-block tiles
    int64_t rb_stride;
    int ng, nb;         // groups and blocks (k / 32) per row
    const uint8_t *q8;  // activation quants (q8_at)
    const float *dt;    // activation d (dt_at)
    float *y;           // [m][n], or with splits > 1 the partials [splits][m][n]
    int32_t *S, *Smin;  // integer dump [m][n][k/32] (DUMP only)
    int m, n, k;
    int ntm, splits, kgs, items, per_xcd;  // kgs: groups per split
};

__device__ __forceinline__ u32x4 ld16(const rsrc_t &r, uint32_t voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
__device__ __forceinline__ v16i offset_acc() {
    v16i c;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        int v = C0;
        asm volatile("" : "+v"(v));  // held in registers, not rebuilt for each MFMA
        c[r] = v;
    }
    return c;
}
__device__ __forceinline__ uint32_t half_of(const u32x4 &d, int j) { return d[j >> 1] >> (16 * (j & 1)); }

// d_w of block j as f32, converted once: left to the compiler the conversion
// goes into every fma as v_fma_mix_f32 (3 % slower at 512 x 4096 x 4096).
__device__ __forceinline__ float dw_of(const u32x4 &d, int j) {
    float f = f16_bits_to_f32(half_of(d, j));
    asm volatile("" : "+v"(f));
    return f;
}

// y += (S * d_w) * d_x (first: =) for the 16 outputs of a lane; dx: d_x of its rows.
__device__ __forceinline__ void combine(float (&y)[16], const v16i &D, float dw, const v4f (&dx)[4], bool first = false) {
    const float ndw = -C0F * dw;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const float t = __builtin_fmaf(u32_as_f32((uint32_t)D[r]), dw, ndw);
        y[r] = first ? t * dx[r >> 2][r & 3] : __builtin_fmaf(t, dx[r >> 2][r & 3], y[r]);
    }
}

struct Item {
    int tile_n, m0, split;
    bool ok;
};
__device__ __forceinline__ Item item_of(const Gemm8Params &p, int rows) {
    const int xcd = (int)blockIdx.x % G8XCD, local = (int)blockIdx.x / G8XCD;
    const int item = xcd * p.per_xcd + local;
    const int tile = item / p.splits, tn = tile / p.ntm;
    return {tn, rows * (tile - tn * p.ntm), item - tile * p.splits, local < p.per_xcd && item < p.items};
}

// ------------------------------------------------------------ tiled form
template <int MT>
struct L8 {  // two stages, one per half of a group
    static constexpr int QS = MT * 4 * 1024;  // [row tile][4 blocks][lane] 16 bytes
    static constexpr int DX = QS;             // [row tile][4 blocks][32 rows] f32
    static constexpr int STAGE = QS + 1024;
};

template <int MT>
__global__ __launch_bounds__(256, 2) void gemm8_kernel(Gemm8Params p) {
    constexpr int NW = 4;
    using L = L8<MT>;
    __shared__ __align__(16) uint8_t lds[2 * L::STAGE];
    const Item it = item_of(p, 32 * MT);
    if (!it.ok) return;  // uniform over the workgroup
    const int m0 = it.m0, tn = it.tile_n;
    const int g0 = it.split * p.kgs, nit = min(p.ng, g0 + p.kgs) - g0;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int nb = p.nb;

    // activation copies: MT of the stage's 4 MT fragments per wave, of one row
    // tile; d of the workgroup's rows (each wave the same).  Rows past m read
    // zeros (quants) or what the plane's padding holds (d: of rows that are
    // never stored); blocks past the row read zeros.
    const rsrc_t rq = buf_rsrc(p.q8, (uint32_t)((int64_t)p.m * p.k));
    const int mt32 = (p.m + 31) / 32;
    const rsrc_t rd = buf_rsrc(p.dt, (uint32_t)((int64_t)mt32 * 128 * nb));
    const rsrc_t rnone = buf_rsrc(p.q8, 0u);
    const int ct = MT * wave / 4;  // the copied row tile
    const int trow = m0 + 32 * ct, trows = min(32, p.m - trow);
    const uint32_t qoff = l32 < trows ? (uint32_t)(trow * p.k + l32 * 32 + 16 * h) : BUF_OOB;
    const int qblk = 32 * max(trows, 0);
    static_assert(MT == 2);
    const uint32_t doff = (uint32_t)(((m0 / 32 + h) * nb + (l32 >> 3)) * 128 + (lane & 7) * 16);  // row tile h
    const bool d_ok = m0 / 32 + h < mt32;

    const int nrb = (p.n + RB - 1) / RB, rb0 = 16 * tn, rb_here = min(16, nrb - rb0);
    const rsrc_t rw = buf_rsrc(p.w + (int64_t)rb0 * p.rb_stride, (uint32_t)(rb_here * p.rb_stride));
    const uint32_t woff = (uint32_t)((4 * wave + (l32 >> 3)) * p.rb_stride + (l32 & 7) * 16);

    auto issue = [&](int i, auto HALF) {  // that half of group g0 + i
        constexpr int HF = decltype(HALF)::value;
        uint8_t *st = lds + HF * L::STAGE;
        const int b0 = (g0 + i) * 8 + 4 * HF;
#pragma unroll
        for (int c = 0; c < MT; c++) {
            const int f = MT * wave + c, b = b0 + f % 4;
            buf_to_lds16(i < nit && b < nb ? rq : rnone, st + 1024 * f, qoff, b * qblk);
        }
        buf_to_lds16(i < nit ? rd : rnone, st + L::DX, d_ok && b0 + (l32 >> 3) < nb ? doff : BUF_OOB, b0 * 128);
    };

    float y[MT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) y[t][r] = 0.0f;
    const v16i c0 = offset_acc();
    u32x4 q[8], dn;
    auto load_q = [&](const rsrc_t &r, int j, int g) { q[j] = ld16(r, woff + 128u * h, (g * PIECES + 2 * j) * 128); };

    issue(0, std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    dn = ld16(rw, woff, (g0 * PIECES + 16) * 128);
    __builtin_amdgcn_sched_barrier(0);  // (the loop's order, so that its waits count the same loads)
#pragma unroll
    for (int j = 0; j < 8; j++) {
        load_q(rw, j, g0);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int i = 0; i < nit; i++) {
        const rsrc_t r4 = i + 1 < nit ? rw : rnone;
        u32x4 d = dn;
        float gsum[MT][16];  // of the group: eight-term chains, then one term a group
        auto half = [&](auto HALF) {
            constexpr int HF = decltype(HALF)::value;
            // this wave's copies of the half have landed (the weight loads
            // issued since may stay in flight) and its reads of the other stage
            // are done, then every wave's
            wait_vmcnt<HF == 0 ? 4 : 5>();
            lds_barrier();
            issue(HF == 0 ? i : i + 1, std::integral_constant<int, 1 - HF>{});
            // no copy past a load that the next wait counts; arithmetic may pass (held
            // back too, 333 x 4096 x 4096 took 34.2 us, not 33.2)
            __builtin_amdgcn_sched_barrier(0x006);
            if constexpr (HF == 0) dn = ld16(r4, woff, ((g0 + i + 1) * PIECES + 16) * 128);
            const uint8_t *st = lds + HF * L::STAGE;
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int j = 4 * HF + jj;
                const float dw = dw_of(d, j);
                v16i D[MT];
#pragma unroll
                for (int t = 0; t < MT; t++)
                    D[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const v4i *)(st + (4 * t + jj) * 1024 + 16 * lane),
                                                                __builtin_bit_cast(v4i, q[j]), c0, 0, 0, 0);
                load_q(r4, j, g0 + i + 1);
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    v4f dx[4];
#pragma unroll
                    for (int g4 = 0; g4 < 4; g4++) dx[g4] = *(const v4f *)(st + L::DX + (4 * t + jj) * 128 + 4 * (8 * g4 + 4 * h));
                    combine(gsum[t], D[t], dw, dx, j == 0);
                }
            }
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) y[t][r] += gsum[t][r];
    }
    wait_vmcnt<0>();  // copies issued past the last group still write LDS

    float *out = p.y + (p.splits > 1 ? (int64_t)it.split * p.m * p.n : 0);
    const int col = 128 * tn + 32 * wave + l32;
    if (col >= p.n) return;
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = m0 + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row < p.m) out[(int64_t)row * p.n + col] = y[t][r];
        }
}

// ------------------------------------------------------------ few rows
// DUMP: the integer sums of every block instead of the outputs.
template <int NW, bool DUMP>
__global__ __launch_bounds__(64 * NW, 2) void few8_kernel(Gemm8Params p) {
    extern __shared__ __align__(16) uint8_t dyn[];  // [NW][32][32] f32, then d [block][32 rows] f32
    float *red = (float *)dyn;
    float *dx = (float *)(dyn + NW * 4096);
    const Item it = item_of(p, 32);
    if (!it.ok) return;  // uniform over the workgroup
    const int m0 = it.m0, tn = it.tile_n, rows = min(32, p.m - m0);
    const int g0 = it.split * p.kgs, g1 = min(p.ng, g0 + p.kgs);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int nb = p.nb;

    const rsrc_t rq = buf_rsrc(p.q8, (uint32_t)((int64_t)p.m * p.k));
    const rsrc_t rnone = buf_rsrc(p.q8, 0u);
    const uint32_t qoff = l32 < rows ? (uint32_t)(m0 * p.k + l32 * 32 + 16 * h) : BUF_OOB;
    const int qblk = 32 * rows;
    const int nrb = (p.n + RB - 1) / RB, rb0 = 4 * tn, rb_here = min(4, nrb - rb0);
    const rsrc_t rw = buf_rsrc(p.w + (int64_t)rb0 * p.rb_stride, (uint32_t)(rb_here * p.rb_stride));
    const uint32_t woff = (uint32_t)((l32 >> 3) * p.rb_stride + (l32 & 7) * 16);

    u32x4 q[8], a[8], dn;
    int g = g0 + wave;
    auto load = [&](int j, int gg, bool live) {
        q[j] = ld16(live ? rw : rnone, woff + 128u * h, (gg * PIECES + 2 * j) * 128);
        a[j] = ld16(live && gg * 8 + j < nb ? rq : rnone, qoff, (gg * 8 + j) * qblk);
    };
    dn = ld16(g < g1 ? rw : rnone, woff, (g * PIECES + 16) * 128);
#pragma unroll
    for (int j = 0; j < 8; j++) load(j, g, g < g1);
    for (int e = tid; e < 256 * (g1 - g0); e += 64 * NW) {  // blocks past the row: zeros
        const int b = 8 * g0 + (e >> 5), r = e & 31;
        dx[e] = b < nb && r < rows ? p.dt[(int64_t)(m0 / 32) * 32 * nb + b * 32 + r] : 0.0f;
    }
    lds_barrier();

    float y[16];
#pragma unroll
    for (int r = 0; r < 16; r++) y[r] = 0.0f;
    const v16i c0 = offset_acc();
    for (; g < g1; g += NW) {  // uniform over the wavefront
        const bool more = g + NW < g1;
        const u32x4 d = dn;
        dn = ld16(more ? rw : rnone, woff, ((g + NW) * PIECES + 16) * 128);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const v16i D = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(v4i, a[j]), __builtin_bit_cast(v4i, q[j]), c0, 0, 0, 0);
            load(j, g + NW, more);
            v4f dx4[4];
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) dx4[g4] = *(const v4f *)(dx + 256 * (g - g0) + 32 * j + 8 * g4 + 4 * h);
            combine(y, D, dw_of(d, j), dx4);
            if constexpr (DUMP) {
                const int b = 8 * g + j, col = 32 * tn + l32;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = 8 * (r >> 2) + 4 * h + (r & 3);
                    if (row < rows && col < p.n && b < nb) {
                        const int64_t o = ((int64_t)(m0 + row) * p.n + col) * nb + b;
                        p.S[o] = D[r] - C0;
                        p.Smin[o] = 0;
                    }
                }
            }
        }
    }
    if constexpr (DUMP) return;

    // red [wavefront][row of 32][column of 32]
#pragma unroll
    for (int r = 0; r < 16; r++) red[(wave * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * 32 + l32] = y[r];
    lds_barrier();
    float *out = p.y + (p.splits > 1 ? (int64_t)it.split * p.m * p.n : 0);
    for (int e = tid; e < 32 * rows; e += 64 * NW) {
        const int r = e >> 5, col = 32 * tn + (e & 31);
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) sum += red[w * 1024 + e];
        if (col < p.n) out[(int64_t)(m0 + r) * p.n + col] = sum;
    }
}

// ------------------------------------------------------------ plan
struct Gemm8Plan {
    int form, ntm, ntn, splits, kgs;  // form 0: 64 x 128; 1, 2: few rows, 4 or 8 wavefronts
    size_t ws;
};

// The form and K split of least estimated time, as kq_plan's (k_gemm.hip):
// the time of one step (a group, or one group per wavefront) of a workgroup
// alone on its CU, its share when the CU holds more, the workgroups a CU
// holds.  Measured over 576..14336 columns, K of 576..14336, 4..512 rows,
// with the quantizer launch (the 128 x 128 tiles with four K splits before):
//   16 x 4096 x 4096    few rows, eight wavefronts 11.4 us, four 14.9 (23.3)
//   128 x 4096 x 4096   few rows, four wavefronts 18.2 us, eight 19.6, 64 x 128 in four splits 23.2 (26.2)
//   333 x 4096 x 4096   64 x 128 in four splits 32.4 us, in two 36.4 (39.5)
//   512 x 14336 x 4096  64 x 128 101.9 us, in two splits 104 (125)
// (the 64 x 128 figures without the group sums, which add 2 %).
struct FormCost {
    int rows, cols;
    float alone, full;
    int slots, groups;
};
constexpr FormCost COST[] = {{64, 128, 2.4f, 1.45f, 3, 1}, {32, 32, 2.4f, 1.5f, 3, 4}, {32, 32, 3.0f, 3.5f, 1, 8}};

Gemm8Plan gemm8_plan(int64_t m, int64_t n, int64_t k) {
    const int ng = (int)((k / QK8_0 + 7) / 8);
    const int most_splits = m <= 8 ? 1 : 16;  // up to 8 rows no split: those calls never needed a workspace
    Gemm8Plan best{};
    float best_us = 0.0f;
    for (int form = 0; form < 3; form++) {
        const FormCost &t = COST[form];
        const int64_t ntm = (m + t.rows - 1) / t.rows, ntn = (n + t.cols - 1) / t.cols;
        for (int splits = 1; splits <= most_splits && splits * 2 <= std::max(ng, 2); splits *= 2) {
            const int kgs = (ng + splits - 1) / splits, ns = (ng + kgs - 1) / kgs;
            if (form && kgs > Q8_FEW_MAX_GROUPS) continue;
            const float c = (float)((ntm * ntn * ns + 255) / 256);  // workgroups of the busiest CU
            const float step = c <= 1.0f ? t.alone : std::max(t.alone * std::ceil(c / t.slots), t.full * c);
            const float us = ((kgs + t.groups - 1) / t.groups) * step + (ns > 1 ? 2.5f + 8.0f * ns * (float)m * (float)n / 3.5e6f : 0.0f);
            if (best_us == 0.0f || us < best_us) {
                best_us = us;
                best = {form, (int)ntm, (int)ntn, ns, kgs, ns > 1 ? (size_t)ns * m * n * 4 : 0};
            }
        }
    }
    return best;
}

// The same with the partials held to `room` bytes: fewer splits.
Gemm8Plan gemm8_plan_in(int64_t m, int64_t n, int64_t k, size_t room) {
    Gemm8Plan g = gemm8_plan(m, n, k);
    if (g.ws > room) {
        const int ng = (int)((k / QK8_0 + 7) / 8), most = std::max(1, (int)(room / ((size_t)m * n * 4)));
        g.splits = std::min(g.splits, most);
        g.kgs = (ng + g.splits - 1) / g.splits;
        g.splits = (ng + g.kgs - 1) / g.kgs;
        g.ws = g.splits > 1 ? (size_t)g.splits * m * n * 4 : 0;
        if (g.form && g.kgs > Q8_FEW_MAX_GROUPS) {
            g.form = 0;
            g.ntm = (int)((m + COST[0].rows - 1) / COST[0].rows);
            g.ntn = (int)((n + COST[0].cols - 1) / COST[0].cols);
        }
    }
    return g;
}

// Rows per launch: the copies address the activation quants with 32-bit
// offsets (rows * k < 2^31); longer inputs run as several launches.
int64_t gemm8_chunk_rows(int64_t m, int64_t k) {
    const int64_t cap = (((int64_t)1 << 31) - 1) / k / 128 * 128;
    return m < cap ? m : cap;
}

}  // namespace

size_t gemm8_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (m < Q8_MIN_ROWS || n <= 0 || k <= 0 || k % QK8_0 || k > (1 << 24)) return (size_t)-1;
    const int64_t mc = gemm8_chunk_rows(m, k);
    if (mc <= 0) return (size_t)-1;
    const Gemm8Plan g = gemm8_plan(mc, n, k);
    if ((int64_t)g.ntm * g.ntn > GEMM_MAX_TILES) return (size_t)-1;
    size_t ws = g.ws;
    if (m % mc) ws = std::max(ws, gemm8_plan(m % mc, n, k).ws);
    return ws;
}

hipError_t launch_gemm8(const WLayout &w, int64_t n, int64_t k, const ActPlanes &x, int64_t m, float *y, int32_t *S,
                        int32_t *Smin, void *ws, size_t ws_bytes, hipStream_t s) {
    if (w.type != TYPE_Q8_0) return hipErrorNotSupported;
    if (!w.slab || !y || !x.q16 || m < Q8_MIN_ROWS || n <= 0 || k <= 0 || k % QK8_0) return hipErrorInvalidValue;
    if (m > 0x7fffffff || n > 0x7fffffff || k > (1 << 24) || w.ng != (k / QK8_0 + 7) / 8) return hipErrorInvalidValue;
    if ((int64_t)16 * w.rb_stride >= ((int64_t)1 << 31)) return hipErrorNotSupported;
    if ((S == nullptr) != (Smin == nullptr)) return hipErrorInvalidValue;
    const int64_t mc = gemm8_chunk_rows(m, k);
    if (mc <= 0) return hipErrorNotSupported;
    const int64_t nb = k / QK8_0;
    for (int64_t r0 = 0; r0 < m; r0 += mc) {
        const int64_t mm = std::min(mc, m - r0);
        Gemm8Plan g = gemm8_plan_in(mm, n, k, ws ? ws_bytes : 0);
        if (S) {  // the dump's form: few rows, split as far as d in LDS asks
            g = {1, (int)((mm + 31) / 32), (int)((n + 31) / 32), (w.ng + Q8_FEW_MAX_GROUPS - 1) / Q8_FEW_MAX_GROUPS, 0, 0};
            g.kgs = (w.ng + g.splits - 1) / g.splits;
        }
        if ((int64_t)g.ntm * g.ntn > GEMM_MAX_TILES) return hipErrorNotSupported;
        Gemm8Params p;
        p.w = w.slab;
        p.rb_stride = w.rb_stride;
        p.ng = w.ng;
        p.nb = (int)nb;
        p.q8 = (const uint8_t *)x.q16 + r0 * k;
        p.dt = dt_plane(x, k) + r0 * nb;
        p.y = g.splits > 1 ? (float *)ws : y + r0 * n;
        p.S = S ? S + r0 * n * nb : nullptr;
        p.Smin = Smin ? Smin + r0 * n * nb : nullptr;
        p.m = (int)mm;
        p.n = (int)n;
        p.k = (int)k;
        p.ntm = g.ntm;
        p.splits = g.splits;
        p.kgs = g.kgs;
        p.items = g.ntm * g.ntn * g.splits;
        p.per_xcd = (p.items + G8XCD - 1) / G8XCD;
        const unsigned grid = (unsigned)(p.per_xcd * G8XCD);
        if (g.form == 0) gemm8_kernel<2><<<grid, 256, 0, s>>>(p);
        else {
            const int nw = g.form == 1 ? 4 : 8, lds = nw * 4096 + 1024 * p.kgs;
            if (lds > 65536) {  // past what a launch may take unasked
                const void *f = S         ? (const void *)few8_kernel<4, true>
                                : nw == 4 ? (const void *)few8_kernel<4, false>
                                          : (const void *)few8_kernel<8, false>;
                const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
                if (e != hipSuccess) return e;
            }
            if (S) few8_kernel<4, true><<<grid, 256, lds, s>>>(p);
            else if (nw == 4) few8_kernel<4, false><<<grid, 256, lds, s>>>(p);
            else few8_kernel<8, false><<<grid, 512, lds, s>>>(p);
        }
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && g.splits > 1 && !S) e = launch_reduce((const float *)ws, y + r0 * n, mm * n, g.splits, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace aq
