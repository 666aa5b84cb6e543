// k_gemm.hip -- launch plan of the prefill GEMM, and the rows from which it is
// taken (gemm_min_rows).
//
// Replaces the M-row loop of candle-core 0.8.4 k_quants::matmul<T> at
// prefill (native/arm_ai_nif/src/llama_candle.rs:93, forward(&x[1,L], 0)).
// The K-quant kernels are in gemm_kq.h (one instance file per type), the
// Q8_0 kernel in k_gemm8.hip.
//
// Split-K.  When there are too few tiles to fill the CUs, the K loop is cut
// into `splits` ranges of super-blocks.  Each writes its partial sums to the
// workspace, and a second, small launch (splitk_reduce) adds them in split
// order -- so the result does not depend on which workgroup finished first,
// and no workgroup waits on another (a device-scope fence per workgroup costs
// an L2 write-back on this GPU).
#include "gemm_kq.h"

#include <algorithm>
#include <cmath>

namespace aq {

namespace {

// y[e] = sum over splits, in order, of part[s][e], V elements per thread.
template <int V>
__global__ __launch_bounds__(256) void splitk_reduce(const float *__restrict__ part, float *__restrict__ y, int64_t total,
                                                     int splits) {
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (e >= total) return;
    if constexpr (V == 4) {
        float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int s = 0; s < splits; s++) {
            const float4 t = *(const float4 *)(part + s * total + e);
            acc.x += t.x;
            acc.y += t.y;
            acc.z += t.z;
            acc.w += t.w;
        }
        *(float4 *)(y + e) = acc;
    } else {
        float acc = 0.0f;
        for (int s = 0; s < splits; s++) acc += part[s * total + e];
        y[e] = acc;
    }
}

struct Plan {
    int form, ntm, ntn, splits, kbs;
    size_t ws;
};

// The tile form and K split of least estimated time.  Per form, measured on
// Q4_K over 512..14336 columns, K of 1024..14336 and 9..1024 rows: the time of
// one step of a workgroup alone on its CU (bound by its own chain), its share
// when the CU holds more (bound by VALU and MFMA issue), the workgroups a CU
// holds, and the super-blocks of a step (the few-row forms' wavefronts take
// one each).  A split adds the reduce launch and one write and read of its
// partials.  Rows x columns x K, with the quantizer launch:
//   512 x 14336 x 4096  128 x 256 tiles 78 us, 64 x 128 90 (71.4 the former on a faster card)
//   512 x 5632 x 2048   64 x 128 28 us, 128 x 256 in two splits 33
//   128 x 4096 x 4096   few rows 17.5 us, 64 x 128 in four splits 21.1
//   512 x 2048 x 2048   32 x 128 tiles 18.9 us, 64 x 128 21.3, few rows 22.1
//   16 x 14336 x 4096   few rows, four wavefronts 14.6 us, eight 17.7, 32 x 128 in four splits 16.3
//   16 x 4096 x 14336   few rows, eight wavefronts in two splits 17.1 us, unsplit 19.0
struct FormCost {
    float alone, full;
    int slots, blocks;
};
constexpr FormCost COST[] = {{1.4f, 0.84f, 2, 1},  {1.7f, 1.27f, 3, 1}, {4.3f, 4.3f, 1, 1},
                             {2.85f, 2.26f, 2, 1}, {1.3f, 1.4f, 3, 4},   {2.5f, 3.7f, 1, 8}};
constexpr int NFORMS = 6;
constexpr int MAX_SPLITS = 16;
// The time of a step against Q4_K's.  A form of 32 rows builds the weight
// operands for one row tile only, which costs most where they are two digits
// (Q6_K): 512 x 2048 x 5632 takes 49.3 us in 32 x 128 tiles, 40.7 in 64 x 128 with
// two splits; 512 x 4096 x 4096 57.6 and 49.0 us.
constexpr float WEIGHT_Q6K[] = {1.8f, 1.42f, 1.3f, 1.3f, 1.3f, 1.3f};
constexpr float WEIGHT_Q3K[] = {1.3f, 1.25f, 1.2f, 1.2f, 1.05f, 1.05f};
float step_weight(int type, int form) {
    return type == TYPE_Q6_K ? WEIGHT_Q6K[form] : type == TYPE_Q3_K ? WEIGHT_Q3K[form] : type == TYPE_Q5_K ? 1.1f : 1.0f;
}

Plan kq_plan(int type, int64_t m, int64_t n, int64_t k) {
    const int ng = (int)(k / QK_K);
    // up to 8 rows no split: those calls never needed a workspace
    const int most_splits = m <= 8 ? 1 : MAX_SPLITS;
    Plan best{};
    float best_us = 0.0f;
    for (int form = 0; form < NFORMS; form++) {
        const KqForm f = KQ_FORMS[form];
        const FormCost &t = COST[form];
        const int64_t ntm = (m + f.rows - 1) / f.rows, ntn = (n + f.cols - 1) / f.cols;
        if (form == 2 && (int64_t)(f.cols / RB) * slabs_of(type) * ng * 128 >= ((int64_t)1 << 31)) continue;  // 32-bit offsets in a tile
        for (int splits = 1; splits <= most_splits && splits * 2 <= std::max(ng, 2); splits *= 2) {
            const int kbs = (ng + splits - 1) / splits, ns = (ng + kbs - 1) / kbs;
            if (t.blocks > 1 && kbs > KQ_FEW_MAX_NG) continue;
            const float c = (float)((ntm * ntn * ns + 255) / 256);  // workgroups of the busiest CU
            const float step = c <= 1.0f ? t.alone : std::max(t.alone * std::ceil(c / t.slots), t.full * c);
            const float us = step_weight(type, form) * ((kbs + t.blocks - 1) / t.blocks) * step +
                             (ns > 1 ? 2.5f + 8.0f * ns * (float)m * (float)n / 3.5e6f : 0.0f);
            if (best_us == 0.0f || us < best_us) {
                best_us = us;
                best = {form, (int)ntm, (int)ntn, ns, kbs, ns > 1 ? (size_t)ns * m * n * 4 : 0};
            }
        }
    }
    return best;
}

// The same with the partials held to `room` bytes: fewer splits.
Plan kq_plan_in(int type, int64_t m, int64_t n, int64_t k, size_t room) {
    Plan g = kq_plan(type, m, n, k);
    if (g.ws > room) {
        const int ng = (int)(k / QK_K), most = std::max(1, (int)(room / ((size_t)m * n * 4)));
        g.splits = std::min(g.splits, most);
        g.kbs = (ng + g.splits - 1) / g.splits;
        g.splits = (ng + g.kbs - 1) / g.kbs;
        g.ws = g.splits > 1 ? (size_t)g.splits * m * n * 4 : 0;
        if (COST[g.form].blocks > 1 && g.kbs > KQ_FEW_MAX_NG) {
            g.form = 0;
            g.ntm = (int)((m + 31) / 32);
            g.ntn = (int)((n + 127) / 128);
        }
    }
    return g;
}

bool kq_type(int type) {
    return type == TYPE_Q4_K || type == TYPE_Q5_K || type == TYPE_Q6_K || type == TYPE_Q2_K || type == TYPE_Q3_K;
}

// Rows per launch: the copies address the f16 activation with 32-bit offsets;
// longer inputs run as several launches.
int64_t kq_chunk_rows(int64_t m, int64_t k) {
    const int64_t cap = (((int64_t)1 << 31) - 1) / (2 * k) / 128 * 128;
    return std::min(m, cap);
}

KqParams kq_params(const WLayout &w, int64_t n, int64_t k, const ActPlanes &x, int64_t r0, int64_t m, const Plan &g, float *y,
                   int32_t *S, int32_t *Smin) {
    KqParams p;
    p.w = w.slab;
    p.wd = w.d;
    p.rb_stride = w.rb_stride;
    p.ng = w.ng;
    p.x16 = x.q16 + r0 * k;
    p.xd = x.d + r0 * w.ng;
    p.xbs = x.bsum16 + r0 * (k / 16);
    p.y = y;
    p.m = (int)m;
    p.n = (int)n;
    p.k = (int)k;
    p.ntm = g.ntm;
    p.splits = g.splits;
    p.kbs = g.kbs;
    p.items = g.ntm * g.ntn * g.splits;
    p.per_xcd = (p.items + 7) / 8;
    p.S = S;
    p.Smin = Smin;
    return p;
}

}  // namespace

// Q5_K, Q2_K, Q3_K and the Q8_0 family have no matrix-core matvec, and the dot4
// matvec's time grows with the rows: from three to seven rows on the GEMM's
// few-row forms are faster, as far as they take the row length.  The line depends
// on what the matvec reads (Q4_0 and Q5_0 are about half and 0.65 of the copy that
// the GEMM reads), on whether its workgroups take a second turn on the CUs
// (`turns`), and on the GEMM's workgroups of 32 columns: past one a CU beside a
// matvec of one turn (`many`), past three a CU (`wide`); either is not felt in short
// rows.  Matvec and GEMM, us (* turns):
//   Q2_K  3 rows  14336 x 4096 15.0, 11.8   32000 x 2048 11.8, 13.0  128256 x 2048 32.1, 25.3
//         4 rows  14336 x 4096 18.2, 11.8   32000 x 2048 14.2, 13.1   32000 x 4096 25.5, 20.8
//   Q3_K  3 rows  14336 x 4096 16.3, 14.1   32000 x 2048 13.4, 14.8   11008 x 2048  9.2,  9.8
//         4 rows   4096 x 4096 13.8, 10.2   32000 x 2048 15.7, 14.9
//   Q5_K  3 rows  12288 x 4096 14.2, 15.4   16384 x 1024  7.0,  8.2   32000 x 4096 26.3, 29.8
//                *20480 x 4096 24.5, 18.7  *24576 x 2048 14.8, 13.8   4096 x 14336 24.3, 20.6
//         4 rows  14336 x 4096 16.9, 15.3   16384 x 1024  8.0,  8.1   32000 x 4096 30.6, 29.9
//   Q8_0  4 rows  14336 x 4096 19.3, 18.2   11008 x 2048 10.3, 11.6   32000 x 4096 36.0, 38.2
//                *20480 x 4096 33.0, 23.4  *24576 x 1024 14.7, 10.8
//         5 rows  14336 x 4096 22.1, 18.1   16384 x 1024  9.6,  9.2   32000 x 4096 44.0, 38.3
//   Q5_0  4 rows  14336 x 4096 19.5, 18.3   11008 x 2048 10.8, 11.6   32000 x 4096 31.1, 38.6
//         5 rows  14336 x 4096 22.8, 18.1  *49152 x 576  26.5, 14.2   32000 x 4096 41.6, 38.6
//   Q4_0  4 rows  14336 x 4096 17.4, 18.2   11008 x 2048  9.9, 11.6   32000 x 4096 26.8, 38.6
//                *20480 x 4096 25.6, 23.8  *24576 x 1024 12.2, 10.8   13824 x 5120 22.9, 21.0
//         5 rows  14336 x 4096 21.0, 18.1   24576 x 2048 17.6, 15.4   32000 x 4096 32.2, 38.4
//         6 rows  14336 x 4096 23.8, 18.1  *49152 x 576  22.6, 14.2   32000 x 4096 36.5, 38.7
//         8 rows  14336 x 4096 29.6, 18.3                             32000 x 2048 25.0, 20.5
// The matrix-core matvec keeps Q4_K and Q6_K up to its 8 rows (11.0 against 14.1 at
// 8 x 14336 x 4096, 8.3 against 8.9 at 8 x 5632 x 2048).
int gemm_min_rows(int type, int64_t n, int64_t k) {
    const bool wide = n > 3 * 256 * 32 && k >= 1024;
    const bool turns = !wide && matvec_workgroups(type, n, k) > 256;
    const bool many = !wide && !turns && n > 256 * 32 && k >= 1024;
    if (type == TYPE_Q8_0 || type == TYPE_Q4_0 || type == TYPE_Q5_0) {
        if (k > 256 * (int64_t)Q8_FEW_MAX_GROUPS) return 9;
        if (type == TYPE_Q4_0) return wide ? 7 : many && k < 5120 ? 5 : Q8_MIN_ROWS;
        return wide || (many && k <= 2048) ? 5 : Q8_MIN_ROWS;
    }
    if (k > QK_K * (int64_t)KQ_FEW_MAX_NG) return 9;
    if (type == TYPE_Q2_K || type == TYPE_Q3_K) return (wide && k < 4096 && n <= 65536) || (many && k > 1024 && k <= 2048) ? 4 : 3;
    if (type == TYPE_Q5_K) return turns || k >= 5120 ? 3 : 4;
    return 9;
}

hipError_t launch_reduce(const float *part, float *y, int64_t total, int splits, hipStream_t s) {
    if (total % 4 == 0 && (((uintptr_t)y | (uintptr_t)part) & 15) == 0)
        splitk_reduce<4><<<(unsigned)((total / 4 + 255) / 256), 256, 0, s>>>(part, y, total, splits);
    else
        splitk_reduce<1><<<(unsigned)((total + 255) / 256), 256, 0, s>>>(part, y, total, splits);
    return hipGetLastError();
}

size_t gemm_workspace_bytes(int type, int64_t m, int64_t n, int64_t k) {
    if (type == TYPE_Q8_0) return gemm8_workspace_bytes(m, n, k);
    if (!kq_type(type) || m <= 0 || n <= 0 || k <= 0 || k % QK_K || k > (1 << 24)) return (size_t)-1;
    const int64_t mc = kq_chunk_rows(m, k);
    if (mc <= 0) return (size_t)-1;
    const Plan g = kq_plan(type, mc, n, k);
    if ((int64_t)g.ntm * g.ntn > GEMM_MAX_TILES) return (size_t)-1;
    size_t ws = g.ws;
    if (m % mc) ws = std::max(ws, kq_plan(type, m % mc, n, k).ws);
    return ws;
}

hipError_t launch_gemm(const WLayout &w, int64_t n, int64_t k, const ActPlanes &x, int64_t m, float *y, int32_t *S,
                       int32_t *Smin, void *ws, size_t ws_bytes, hipStream_t s) {
    if (w.type == TYPE_Q8_0) return launch_gemm8(w, n, k, x, m, y, S, Smin, ws, ws_bytes, s);
    if (!kq_type(w.type)) return hipErrorNotSupported;
    const bool dplane = w.type == TYPE_Q6_K || w.type == TYPE_Q2_K;
    if (!w.slab || (dplane && !w.d) || !y || !x.q16 || !x.d || !x.bsum16 || m <= 0 || n <= 0 || k <= 0 || k % QK_K)
        return hipErrorInvalidValue;
    if (m > 0x7fffffff || n > 0x7fffffff || k > (1 << 24) || w.ng != k / QK_K) return hipErrorInvalidValue;
    if ((int64_t)16 * w.rb_stride >= ((int64_t)1 << 31)) return hipErrorNotSupported;  // one column tile's weights
    if ((S == nullptr) != (Smin == nullptr)) return hipErrorInvalidValue;
    const int64_t mc = kq_chunk_rows(m, k);
    if (mc <= 0) return hipErrorNotSupported;
    for (int64_t r0 = 0; r0 < m; r0 += mc) {
        const int64_t mm = std::min(mc, m - r0);
        Plan g = kq_plan_in(w.type, mm, n, k, ws ? ws_bytes : 0);
        if (S) g.form = 0, g.ntm = (int)((mm + 31) / 32), g.ntn = (int)((n + 127) / 128);  // the dump's form
        if ((int64_t)g.ntm * g.ntn > GEMM_MAX_TILES) return hipErrorNotSupported;
        const KqParams p = kq_params(w, n, k, x, r0, mm, g, g.splits > 1 ? (float *)ws : y + r0 * n,
                                     S ? S + r0 * n * w.ng : nullptr, Smin ? Smin + r0 * n * w.ng : nullptr);
        hipError_t e = w.type == TYPE_Q4_K   ? launch_kq_q4k(p, g.form, S != nullptr, s)
                       : w.type == TYPE_Q5_K ? launch_kq_q5k(p, g.form, S != nullptr, s)
                       : w.type == TYPE_Q6_K ? launch_kq_q6k(p, g.form, S != nullptr, s)
                       : w.type == TYPE_Q2_K ? launch_kq_q2k(p, g.form, S != nullptr, s)
                                             : launch_kq_q3k(p, g.form, S != nullptr, s);
        if (e == hipSuccess && g.splits > 1) e = launch_reduce((const float *)ws, y + r0 * n, mm * n, g.splits, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Both weights as 64 x 128 tiles, the first unsplit, the second split until its
// steps are at most half as many, and together no more workgroups than the CUs
// hold at once (two each); false where the two do not run as one launch.
static bool pair_plan(int type1, int type2, int64_t m, int64_t n1, int64_t n2, int64_t k, Plan &g1, Plan &g2) {
    if (type1 != TYPE_Q4_K || (type2 != TYPE_Q6_K && type2 != TYPE_Q5_K)) return false;
    if (m <= 0 || n1 <= 0 || n2 <= 0 || k <= 0 || k % QK_K || m > 0x7fffffff || n1 > 0x7fffffff || n2 > 0x7fffffff ||
        k > (1 << 24) || kq_chunk_rows(m, k) < m)
        return false;
    const int ng = (int)(k / QK_K);
    const int64_t ntm = (m + KQ_FORMS[1].rows - 1) / KQ_FORMS[1].rows;
    const int64_t t1 = ntm * ((n1 + 127) / 128), t2 = ntm * ((n2 + 127) / 128);
    int splits = 1;
    while (splits < MAX_SPLITS && t1 + 2 * t2 * splits <= 512 && ng / (2 * splits) >= 2) splits *= 2;
    if (t1 + t2 * splits > 512) return false;
    const int kbs = (ng + splits - 1) / splits, ns = (ng + kbs - 1) / kbs;
    g1 = {1, (int)ntm, (int)((n1 + 127) / 128), 1, ng, 0};
    g2 = {1, (int)ntm, (int)((n2 + 127) / 128), ns, kbs, ns > 1 ? (size_t)ns * m * n2 * 4 : 0};
    return true;
}

size_t gemm_pair_workspace_bytes(int type1, int type2, int64_t m, int64_t n1, int64_t n2, int64_t k) {
    Plan g1, g2;
    return pair_plan(type1, type2, m, n1, n2, k, g1, g2) ? g2.ws : (size_t)-1;
}

hipError_t launch_gemm_pair(const WLayout &w1, int64_t n1, float *y1, const WLayout &w2, int64_t n2, float *y2,
                            int64_t k, const ActPlanes &x, int64_t m, void *ws, size_t ws_bytes, hipStream_t s) {
    Plan g1, g2;
    if (!pair_plan(w1.type, w2.type, m, n1, n2, k, g1, g2) || g2.ws > (ws ? ws_bytes : 0)) return hipErrorNotSupported;
    if (!w1.slab || !w2.slab || (w2.type == TYPE_Q6_K && !w2.d) || !y1 || !y2 || !x.q16 || !x.d || !x.bsum16 ||
        w1.ng != k / QK_K || w2.ng != k / QK_K)
        return hipErrorInvalidValue;
    if ((int64_t)16 * w1.rb_stride >= ((int64_t)1 << 31) || (int64_t)16 * w2.rb_stride >= ((int64_t)1 << 31))
        return hipErrorNotSupported;
    const KqParams p = kq_params(w1, n1, k, x, 0, m, g1, y1, nullptr, nullptr);
    const KqParams q = kq_params(w2, n2, k, x, 0, m, g2, g2.splits > 1 ? (float *)ws : y2, nullptr, nullptr);
    hipError_t e = launch_kq_pair(p, q, w2.type, s);
    if (e == hipSuccess && g2.splits > 1) e = launch_reduce((const float *)ws, y2, m * n2, g2.splits, s);
    return e;
}

}  // namespace aq
