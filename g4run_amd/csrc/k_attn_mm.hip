// k_attn_mm.hip -- causal attention of a prompt batch on the matrix cores:
// attn_kernel (model.c:509-545) for nb new tokens over an f16 KV cache (head
// dims 64 to 512, gemma4's full layers included), the
// tokens of a tile sharing every K and V row they read.
//
// Rows of a tile are (token, query head) pairs of one KV head: 32 / GRP
// tokens x GRP heads = 32 rows.  Token b sits at position p0 + b and attends
// positions j0(b) .. p0 + b, j0 = max(0, p + 1 - window) with a window (else
// 0); on a ring, position j's row is at slot j % ring.  The batch's positions
// are cut at multiples of 128 (score chunks) and 256 (value spans) counted
// from 0, so every sum a row takes -- its scores, its chunk statistics, the
// normaliser over its own chunks (lane k = its k-th chunk), each span's
// weighted values and the spans added in order -- has the same operands in
// the same order whatever other tokens share the batch: a token's row has
// the same bits in any batch, alone included.
//   scores   grid KV head x 128-position chunk x tile, 4 waves x 32
//            positions: S = K_j . fp16(q) (model.c:530-538, no 1/sqrt(d)) as
//            one v_mfma_f32_32x32x16_f16 per 16 head elements (exact
//            products, fp32 sums); per row and chunk the maximum m_c and
//            l_c = sum expf(s - m_c) over the row's positions, summed in
//            double: 16 per lane in order, the two lanes of a row, then the
//            waves in order.
//   values   grid KV head x 256-position span x tile: per row the global
//            maximum M and normaliser (sum_c l_c exp(m_c - M) in double) as in
//            the decode kernels, the weights fp16(expf(s - M) * inv)
//            (model.c:547-555) into LDS (0 outside a row's positions), then
//            sum_j w_j V_j on v_mfma_f32_32x32x16_f16 with the positions as
//            the contraction, 32 columns per wave.
//   combine  per (token, head) its spans' partials added in order.
// With a device position (decode steps replayed from a graph) the grids are
// sized for the most positions a call can span and the workgroups past the
// call's last position return at once.
// Differences from the per-token kernels are the fp32 orders of the score and
// value sums, the grouping of the double normaliser and the exponentials of
// the scores and weights taken in fp32 (expf, about 1 ulp; the reference
// rounds exp in double to float: the weights' fp16 rounding can differ by
// one step where a product lands within ~1e-7 of a rounding boundary):
// within the attention's tolerance of the CPU, not bit-identical to them.  A non-finite
// V row (an f16 overflow) reaches the earlier rows of its tile as 0 * inf.
#include <algorithm>
#include <cmath>

#include "formats.h"
#include "kernels.h"
#include "steps.h"

namespace g4 {

typedef _Float16 am_v8h __attribute__((ext_vector_type(8)));
typedef float am_v16f __attribute__((ext_vector_type(16)));

constexpr int AMM_CH = 128;          // positions per score workgroup
constexpr int AMM_NP = 256;          // positions per value workgroup
constexpr size_t AMM_OFF = 256;      // the decode layout's header (error and epoch words) stays untouched

struct AmmArgs {
    const float *q;                  // [nb][n_head][hd] prepared queries
    float *out;                      // [nb][n_head][hd]
    uint8_t *q8out;                  // optional q8_0 rows of out, q8_stride bytes per token
    size_t q8_stride;
    FewAct few;                      // or (few.qa set) out as q8_0 in k_mm_few's layout
    const uint8_t *kc, *vc;
    int n_head, n_kv, window, ring;
    int p0, nb;                      // token 0's position (or *pos_dev) and the token count
    const int *pos_dev;
    int nch, nchv, ntt;              // the grid: chunks, spans (the strides of Mc / Lc and P), token tiles
    int jb, span;                    // set on the device by amm_view: first position (a multiple of AMM_NP) and count
    float *S;                        // [nb * n_head][nch * AMM_CH]
    float *Mc;                       // [nb * n_head][nch]
    double *Lc;                      // [nb * n_head][nch]
    float *P;                        // [nb * n_head][nchv][hd]
};

static size_t amm_al(size_t v) { return (v + 255) & ~(size_t)255; }
struct AmmWs {
    size_t S, Mc, Lc, P, total;
};
// most positions a batch spans: its last token's window (or all of its
// positions) plus the earlier tokens, from a multiple of AMM_NP
static int amm_span_max(int npos_max, int nb) { return npos_max + nb - 1 + AMM_NP - 1; }
static AmmWs amm_ws(int n_head, int hd, int nb, int span) {
    const size_t R = (size_t)nb * n_head, nch = (span + AMM_CH - 1) / AMM_CH, nchv = (span + AMM_NP - 1) / AMM_NP;
    AmmWs w;
    w.S = AMM_OFF;
    w.Mc = w.S + amm_al(R * nch * AMM_CH * 4);
    w.Lc = w.Mc + amm_al(R * nch * 4);
    w.P = w.Lc + amm_al(R * nch * 8);
    w.total = w.P + amm_al(R * nchv * hd * 4);
    return w;
}
size_t attn_batch_mm_workspace_bytes(int n_head, int hd, int npos_max, int nb) {
    return amm_ws(n_head, hd, nb, amm_span_max(npos_max, nb)).total;
}

// the call's positions: token 0's position, the first position any token
// attends rounded down to a multiple of AMM_NP, and the count from there
__device__ __forceinline__ void amm_view(AmmArgs &c) {
    if (c.pos_dev) c.p0 = *c.pos_dev;
    const int j0 = c.window ? max(0, c.p0 + 1 - c.window) : 0;
    c.jb = j0 / AMM_NP * AMM_NP;
    c.span = c.p0 + c.nb - c.jb;
}

// Workgroup l of a call's n_kv x n position blocks x ntt token tiles runs on XCD
// l % 8.  The tiles that share a block's K or V rows are neighbours on one XCD
// and find them in its L2: each XCD takes an eighth of the tiles, whatever the
// number of blocks.  (With whole blocks dealt to the XCDs in turn, two blocks of
// one KV head kept six XCDs idle: 256 tokens at position 0, 8 q / 1 kv heads of
// 512, 42.6 us, now 23.6; 64 tokens at position 4096, 8 q / 4 kv heads of 128, 26.6
// and 23.7.)  From AMM_ROUNDS tiles whole rounds of 8 blocks are dealt so all the
// same and an eighth of the rest to each: the XCDs then read neighbouring rows at
// any one time (256 tokens at position 16000, 32 q / 4 kv heads of 256, 1005 us
// against 1044).  n counts the blocks up to the call's last position; the grid may
// be sized for more.
constexpr int AMM_ROUNDS = 4096;
__device__ __forceinline__ bool amm_block(const AmmArgs &c, int l, int size, int &kvh, int &blk, int &tt) {
    const int n = (c.span + size - 1) / size, pairs = c.n_kv * n, total = pairs * c.ntt;
    const int rounds = total >= AMM_ROUNDS ? pairs >> 3 : 0, whole = rounds * c.ntt, left = total - 8 * whole, per = (left + 7) >> 3;
    const int x = l & 7, i = l >> 3, item = i < whole ? i : x * per + i - whole, p = item / c.ntt;
    const int pair = i < whole ? p * 8 + x : 8 * rounds + p;
    tt = item - p * c.ntt;
    kvh = pair / n;
    blk = pair - kvh * n;
    return i < whole || (i - whole < per && item < left);
}
static int64_t amm_blocks(const AmmArgs &c, int n) { return ((int64_t)c.n_kv * n * c.ntt + 7) / 8 * 8; }

__device__ __forceinline__ am_v8h amm_ld8(const void *p) { return *(const am_v8h *)p; }
__device__ __forceinline__ am_v16f amm_mma(am_v8h a, am_v8h b, am_v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// tile row i: token b and head h; the row's positions j0 .. p
template <int GRP>
__device__ __forceinline__ void amm_rowinfo(const AmmArgs &c, int kvh, int tt, int i, int &b, int &h, int &j0, int &p) {
    constexpr int T = 32 / GRP;
    b = tt * T + i / GRP;
    h = kvh * GRP + i % GRP;
    p = c.p0 + b;
    j0 = c.window ? std::max(0, p + 1 - c.window) : 0;
}

// Scores, transposed: the positions are the MFMA's rows and the tile's 32
// (token, head) rows its columns, so a lane holds 16 positions of one row and a
// row's statistics are sums within a lane and one exchange (with the positions
// across the lanes they were five exchanges for each of 16 rows, most of them
// of doubles).  A wave's 32 K rows are loaded in runs of adjacent bytes and
// turned into operands through LDS of its own, 128 head elements at a time: an
// operand loaded straight from memory has adjacent lanes in different rows, one
// L1 access each.  64 tokens after 4096 positions, 8 q / 4 kv heads of 256: 17.2
// -> 10.6 us.
template <int HD, int GRP>
__global__ __launch_bounds__(256) void k_amm_scores(AmmArgs c) {
    constexpr int T = 32 / GRP, QS = HD + 8;
    constexpr int KW = HD < 128 ? HD : 128, KH = HD / KW, LPR = KW / 8, RPL = 64 / LPR, NL = 32 / RPL;   // K: columns at a time, lanes per row
    constexpr int KS = KW * 2 + 16;                                 // LDS row stride (bytes)
    __shared__ __align__(16) uint16_t qs[32][QS];                   // fp16 queries of the tile
    __shared__ __align__(16) uint8_t ks[4][32 * KS];
    __shared__ float wm[4][32];
    __shared__ double wl[4][32];
    amm_view(c);
    int kvh, tt, ch;
    if (!amm_block(c, blockIdx.x, AMM_CH, kvh, ch, tt)) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, li = lane & 31, kh = lane >> 5;
    const int jw = ch * AMM_CH + wave * 32;                          // the wave's first position
    const int jfirst = c.window ? max(0, c.p0 + 1 - c.window) : 0, jlast = c.jb + c.span - 1;
    // K rows jfirst .. jlast are one contiguous run of slots (at most `ring` of
    // them, each row stored twice on a ring)
    const uint8_t *kbase = c.kc + ((size_t)(c.ring ? jfirst % c.ring : jfirst) * c.n_kv + kvh) * HD * 2 + 16 * (lane % LPR);
    am_v8h kr[KH][NL];
#pragma unroll
    for (int f = 0; f < KH; f++)
#pragma unroll
        for (int n = 0; n < NL; n++) {
            const int j = std::min(std::max(c.jb + jw + RPL * n + lane / LPR, jfirst), jlast);
            kr[f][n] = amm_ld8(kbase + (size_t)(j - jfirst) * c.n_kv * HD * 2 + f * KW * 2);
        }
    // the tile's queries: all of a thread's loads issued before any conversion
    constexpr int NQ = 32 * HD / 4 / 256;                           // float4 per thread
    float4 qv[NQ];
#pragma unroll
    for (int k = 0; k < NQ; k++) {
        const int x = t + 256 * k, i = x / (HD / 4), e4 = x % (HD / 4), b = tt * T + i / GRP, h = kvh * GRP + i % GRP;
        qv[k] = b < c.nb ? *(const float4 *)(c.q + ((size_t)b * c.n_head + h) * HD + 4 * e4) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int k = 0; k < NQ; k++) {
        const int x = t + 256 * k, i = x / (HD / 4), e4 = x % (HD / 4);
        const uint32_t lo = f2h(qv[k].x) | ((uint32_t)f2h(qv[k].y) << 16), hi = f2h(qv[k].z) | ((uint32_t)f2h(qv[k].w) << 16);
        *(uint2 *)&qs[i][4 * e4] = make_uint2(lo, hi);
    }
    lds_barrier();
    am_v16f acc = {};
    uint8_t *kl = ks[wave];
#pragma unroll
    for (int f = 0; f < KH; f++) {
        // a wave's LDS accesses complete in order; the empty asms keep the
        // compiler from moving them across the hand-over
        asm volatile("" ::: "memory");
#pragma unroll
        for (int n = 0; n < NL; n++) *(am_v8h *)(kl + (RPL * n + lane / LPR) * KS + 16 * (lane % LPR)) = kr[f][n];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int s = 0; s < KW / 16; s++)
            acc = amm_mma(amm_ld8(kl + li * KS + (16 * s + 8 * kh) * 2), amm_ld8(&qs[li][f * KW + 16 * s + 8 * kh]), acc);
    }
    // C[i][li]: positions i = 8 (r / 4) + 4 kh + r % 4 of tile row li
    int b, h, j0, p;
    amm_rowinfo<GRP>(c, kvh, tt, li, b, h, j0, p);
    const bool row = b < c.nb;
    const size_t R = (size_t)(row ? b : 0) * c.n_head + h;
    bool ok[16];
    float m = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int jl = jw + 8 * (r >> 2) + 4 * kh + (r & 3), j = c.jb + jl;
        ok[r] = row && jl < c.span && j >= j0 && j <= p;
        m = fmaxf(m, ok[r] ? acc[r] : -INFINITY);
    }
    m = fmaxf(m, partner<32>(m));
    if (kh == 0) wm[wave][li] = m;
    if (row) {                                                       // whole chunks; k_amm_v gives positions outside a row's own weight 0
        float *Sr = c.S + R * c.nch * AMM_CH + jw + 4 * kh;
#pragma unroll
        for (int q = 0; q < 4; q++) *(float4 *)(Sr + 8 * q) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    }
    lds_barrier();
    const float mc = fmaxf(fmaxf(wm[0][li], wm[1][li]), fmaxf(wm[2][li], wm[3][li]));
    double l = 0.0;
#pragma unroll
    for (int r = 0; r < 16; r++) l += ok[r] ? (double)expf(acc[r] - mc) : 0.0;
    l += partner<32>(l);
    if (kh == 0) wl[wave][li] = l;
    lds_barrier();
    if (t < 32 && row) {
        c.Mc[R * c.nch + ch] = mc;
        c.Lc[R * c.nch + ch] = ((wl[0][t] + wl[1][t]) + wl[2][t]) + wl[3][t];
    }
}

// Values: 8 or 16 waves (NW), each with 4 or 2 of the tile's rows for the weights
// and one unit of 32 columns for the sums (heads of 512 with 8 waves take two
// workgroups, grid y).  Chunk statistics, scores (16 bytes per lane) and half of
// the V rows (in runs of adjacent bytes) are loaded at the start, 20 loads in all
// with 8 waves (V as 128 words per lane took 4.3 us to issue); the other half of
// V goes out once the statistics' registers are free and is in flight while the
// weights are formed.  Scores of a chunk past the call's last one are not loaded;
// scores that a loaded chunk holds outside a row's positions are dropped.  A
// row's statistics and weights are one wave's, handed over in registers; V
// passes through LDS of the wave's own 64 positions at a time and is read there
// transposed (ds_read_b64_tr_b16).  48 or 80 KB of LDS and 128 registers: 16
// waves per CU.  64 tokens after 4096 positions, 8 q / 4 kv heads of 256: 20.8 ->
// 15.6 us.
typedef short am_v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) am_v4s *am_lds4;

template <int HD, int GRP, int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_amm_v(AmmArgs c) {
    constexpr int RW = 32 / NW, NU = HD < 32 * NW ? HD / 32 : NW;   // rows per wave, waves with a column unit
    constexpr int ST = AMM_NP / 16, VP = 4, HP = AMM_NP / VP;       // steps, V parts and their positions
    // fp16 weights of the span, the 16-byte units of row r at unit ^ (r & 7)
    __shared__ __align__(16) uint8_t wsh[32 * AMM_NP * 2];
    __shared__ __align__(16) uint8_t vsh[NW][HP * 64];              // a wave's part of V: rows of 32 columns
    amm_view(c);
    int kvh, tt, cv;
    if (!amm_block(c, blockIdx.x, AMM_NP, kvh, cv, tt)) return;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t) >> 6, li = lane & 31, kh = lane >> 5;
    const int jl0 = cv * AMM_NP, unit = wave + NW * blockIdx.y;
    const int jfirst = c.window ? max(0, c.p0 + 1 - c.window) : 0, jlast = c.jb + c.span - 1;
    // 1. per row the global maximum and normaliser over the row's own chunks
    // (wave w: rows RW w .. RW w + RW - 1; lane k: the row's k-th chunk, 64 per round)
    const int nca = (c.span + AMM_CH - 1) / AMM_CH;                  // >= any row's chunk count
    int nrc[RW], j0r[RW], pr[RW];
    size_t base[RW];
    bool rv[RW], on[RW];
    float mcv[RW];
    double lcv[RW];
    float4 sv[RW];                                                   // the scores of positions 4 lane .. + 3
    const int jt = jl0 + 4 * lane, jg = c.jb + jt;
#pragma unroll
    for (int k = 0; k < RW; k++) {
        int b, h;
        amm_rowinfo<GRP>(c, kvh, tt, wave * RW + k, b, h, j0r[k], pr[k]);
        rv[k] = b < c.nb;
        const int clo = rv[k] ? (j0r[k] - c.jb) / AMM_CH : 0;
        nrc[k] = rv[k] ? (pr[k] - c.jb) / AMM_CH - clo + 1 : 0;
        base[k] = ((size_t)(rv[k] ? b : 0) * c.n_head + h) * c.nch + clo;
        on[k] = lane < nrc[k];
        mcv[k] = on[k] ? c.Mc[base[k] + lane] : -INFINITY;
        lcv[k] = on[k] ? c.Lc[base[k] + lane] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < RW; k++) {
        // whole chunks of scores are stored for the tile's rows; a span's second
        // chunk may lie past the last one
        const bool in = rv[k] && jt < c.nch * AMM_CH;
        sv[k] = in ? *(const float4 *)(c.S + (base[k] - (rv[k] ? (j0r[k] - c.jb) / AMM_CH : 0)) * AMM_CH + jt) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // the unit's columns of the span's V rows, 4 lanes to a row, 16 rows per
    // load.  The attended positions jfirst .. jlast are at most `ring` apart,
    // so on a ring (rows stored at j % ring and again at j % ring + ring) they
    // are one contiguous run of slots from jfirst % ring.  Rows are clamped to
    // them, so every row loaded holds a stored value.
    am_v8h v[ST];
    const size_t rstr = (size_t)c.n_kv * HD * 2;
    const uint8_t *vbase = c.vc + ((size_t)(c.ring ? jfirst % c.ring : jfirst) * c.n_kv + kvh) * HD * 2 + 64 * unit + 16 * (lane & 3);
    auto load_v = [&](int q) __attribute__((always_inline)) {
        const int j = std::min(std::max(c.jb + jl0 + 16 * q + (lane >> 2), jfirst), jlast);
        v[q] = amm_ld8(vbase + (size_t)(j - jfirst) * rstr);
    };
    if (wave < NU) {                                                 // uniform
#pragma unroll
        for (int q = 0; q < ST / 2; q++) load_v(q);
    }
    asm volatile("" ::: "memory");
    float m[RW], inv[RW];
    {
        double sum[RW];
#pragma unroll
        for (int k = 0; k < RW; k++) m[k] = group_max<64>(mcv[k]);
        for (int c1 = 64; c1 < nca; c1 += 64)
#pragma unroll
            for (int k = 0; k < RW; k++) m[k] = fmaxf(m[k], group_max<64>(c1 + lane < nrc[k] ? c.Mc[base[k] + c1 + lane] : -INFINITY));
#pragma unroll
        for (int k = 0; k < RW; k++)                                 // rows outside the batch (uniform) skip the exp
            sum[k] = rv[k] ? group_sum_t<64>(on[k] ? lcv[k] * exp((double)mcv[k] - (double)m[k]) : 0.0) : 1.0;
        for (int c1 = 64; c1 < nca; c1 += 64)
#pragma unroll
            for (int k = 0; k < RW; k++) {
                const bool o = c1 + lane < nrc[k];
                const float mc = o ? c.Mc[base[k] + c1 + lane] : 0.0f;
                const double lc = o ? c.Lc[base[k] + c1 + lane] : 0.0;
                sum[k] += group_sum_t<64>(o ? lc * exp((double)mc - (double)m[k]) : 0.0);
            }
#pragma unroll
        for (int k = 0; k < RW; k++) inv[k] = (float)(1.0 / sum[k]);
    }
    asm volatile("" ::: "memory");
    if (wave < NU) {                                                 // the second half, the statistics' registers free
#pragma unroll
        for (int q = ST / 2; q < ST; q++) load_v(q);
    }
    asm volatile("" ::: "memory");
    // 2. the weights (0 outside a row's positions)
#pragma unroll
    for (int k = 0; k < RW; k++) {
        uint2 w = make_uint2(0, 0);
        if (rv[k]) {                                                 // uniform
            const float e[4] = {sv[k].x, sv[k].y, sv[k].z, sv[k].w};
            uint32_t hw[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bool ok = jt + i < c.span && jg + i >= j0r[k] && jg + i <= pr[k];
                hw[i] = f2h(ok ? expf(e[i] - m[k]) * inv[k] : 0.0f);
            }
            w = make_uint2(hw[0] | (hw[1] << 16), hw[2] | (hw[3] << 16));
        }
        const int r = wave * RW + k;
        *(uint2 *)(wsh + r * (AMM_NP * 2) + 16 * ((lane >> 1) ^ (r & 7)) + 8 * (lane & 1)) = w;
    }
    lds_barrier();
    if (wave >= NU) return;                                          // uniform
    // 3. sum_j w_j V_j over the span's 16 steps of 16 positions, in step order
    // (the MFMA's accumulation).  The operand of step q: lane (c, half) holds
    // column c of positions 8 half .. + 7, two transposed reads in which 16
    // lanes give 4 rows of 16 columns and get 4 rows of their own column
    uint8_t *vl = vsh[wave];
    const int g4 = lane >> 4, i16 = lane & 15;
    const uint32_t tr = (8 * (g4 >> 1) + (i16 >> 2)) * 64 + 32 * (g4 & 1) + 8 * (i16 & 3);
    am_v16f acc = {};
#pragma unroll
    for (int f = 0; f < VP; f++) {
        asm volatile("" ::: "memory");                               // a wave's LDS accesses complete in order
#pragma unroll
        for (int q = 0; q < ST / VP; q++) *(am_v8h *)(vl + (16 * q + (lane >> 2)) * 64 + 16 * (lane & 3)) = v[f * (ST / VP) + q];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < ST / VP; q++) {
            const am_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((am_lds4)(vl + tr + 16 * q * 64));
            const am_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((am_lds4)(vl + tr + (16 * q + 4) * 64));
            typedef short v8s __attribute__((ext_vector_type(8)));
            const v8s bv = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const int un = 2 * (f * (ST / VP) + q) + kh;
            acc = amm_mma(amm_ld8(wsh + li * (AMM_NP * 2) + 16 * (un ^ (li & 7))), __builtin_bit_cast(am_v8h, bv), acc);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int i = 8 * (r >> 2) + 4 * kh + (r & 3);
        int b, h, j0, p;
        amm_rowinfo<GRP>(c, kvh, tt, i, b, h, j0, p);
        if (b < c.nb) c.P[(((size_t)b * c.n_head + h) * c.nchv + cv) * HD + 32 * unit + li] = acc[r];
    }
}

// grid (n_head, nb), 256 threads (elements e and e + 256): the spans'
// partials in order; with q8out (or few), the head row as q8_0 blocks too
// (quants.c:74-109)
template <int HD>
__global__ __launch_bounds__(256) void k_amm_combine(AmmArgs c) {
    constexpr int EP = (HD + 255) / 256;                             // elements per thread
    __shared__ float row[HD];
    amm_view(c);
    const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    const size_t R = (size_t)b * c.n_head + h;
    const int p = c.p0 + b, j0 = c.window ? max(0, p + 1 - c.window) : 0;
    const int first = (j0 - c.jb) / AMM_NP, last = (p - c.jb) / AMM_NP;   // the token's spans
#pragma unroll
    for (int q = 0; q < EP; q++) {
        const int e = t + 256 * q;
        if (e < HD) {
            const float *src = c.P + R * c.nchv * HD + e;
            float r = 0.0f;
            for (int c0 = first; c0 <= last; c0 += 8) {              // eight loads in flight, added in order
                float v[8];
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = c0 + k <= last ? src[(size_t)(c0 + k) * HD] : 0.0f;
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (c0 + k <= last) r += v[k];
            }
            c.out[R * HD + e] = r;
            row[e] = r;
        }
    }
    if (c.q8out || c.few.qa) {
        __syncthreads();
        const bool own = t < HD / 4;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (own)
            for (int k = 0; k < 4; k++) v[k] = row[4 * t + k];
        if (t < (HD / 4 + 63) / 64 * 64) {
            if (c.few.qa) q8_store4_few(v, h * (HD / 4) + t, own, c.few, b);
            else q8_store4(v, t, own, c.q8out + (size_t)b * c.q8_stride + (size_t)h * (HD / 32) * 34);
        }
    }
}

bool attn_batch_mm_ok(const QkvArgs &a) {
    const int grp = a.n_kv > 0 ? a.n_head / a.n_kv : 0;
    return a.kv_type == F16 && (a.hd == 64 || a.hd == 128 || a.hd == 256 || a.hd == 512) && a.n_kv > 0 && a.n_head % a.n_kv == 0 &&
           (grp == 1 || grp == 2 || grp == 4 || grp == 8);
}

template <int HD, int GRP>
static void amm_go(const AmmArgs &c, hipStream_t s) {
    hipLaunchKernelGGL((k_amm_scores<HD, GRP>), dim3((unsigned)amm_blocks(c, c.nch)), dim3(256), 0, s, c);
    // heads of 512, 16 column units: two workgroups of 8 waves, or from 320 blocks
    // one of 16, which forms the weights once (us a call, 8 q / 1 kv heads, two / one:
    // one token at position 1000 16.5 / 17.3, 64 tokens at 4096 44.4 / 45.5, at 8192
    // 74.9 / 71.3, 256 at 16000 502 / 454; the per-tile launch before both 478)
    const unsigned blocks = (unsigned)amm_blocks(c, c.nchv);
    if (HD == 512 && blocks >= 320) hipLaunchKernelGGL((k_amm_v<HD, GRP, HD == 512 ? 16 : 8>), dim3(blocks), dim3(1024), 0, s, c);
    else hipLaunchKernelGGL((k_amm_v<HD, GRP, 8>), dim3(blocks, HD == 512 ? 2 : 1), dim3(512), 0, s, c);
    hipLaunchKernelGGL(k_amm_combine<HD>, dim3(c.n_head, c.nb), dim3(256), 0, s, c);
}

hipError_t launch_attn_batch_mm(const float *q, const QkvArgs &a, int npos0, int nb, float *out, uint8_t *q8out, uint8_t *ws,
                                size_t ws_bytes, hipStream_t s, size_t q8_stride, const int *pos_dev, int npos_max,
                                const FewAct &few) {
    if (!attn_batch_mm_ok(a) || !q || !out || !ws || nb < 1 || nb > 65535 || (!pos_dev && npos0 < 1) || (pos_dev && npos_max < 1) ||
        (few.qa && nb > 16 * few.mt))
        return hipErrorInvalidValue;
    if (a.ring && (a.window <= 0 || a.window > a.ring || nb > a.ring - a.window + 1)) return hipErrorInvalidValue;
    AmmArgs c{};
    c.q = q;
    c.out = out;
    c.q8out = q8out;
    c.q8_stride = q8_stride ? q8_stride : (size_t)a.n_head * (a.hd / 32) * 34;
    c.few = few;
    c.kc = a.kc;
    c.vc = a.vc;
    c.n_head = a.n_head;
    c.n_kv = a.n_kv;
    c.window = a.window;
    c.ring = a.ring;
    c.p0 = npos0 - 1;
    c.nb = nb;
    c.pos_dev = pos_dev;
    // the grid: this call's positions, or with a device position the most a
    // call can span (npos_max positions attended by its last token)
    int span;
    if (pos_dev) {
        span = amm_span_max(a.window ? std::min(a.window, npos_max) : npos_max, nb);
    } else {
        const int j0 = a.window ? std::max(0, c.p0 + 1 - a.window) : 0;
        span = c.p0 + nb - j0 / AMM_NP * AMM_NP;
    }
    c.nch = (span + AMM_CH - 1) / AMM_CH;
    c.nchv = (span + AMM_NP - 1) / AMM_NP;
    const int grp = a.n_head / a.n_kv;
    c.ntt = (nb + 32 / grp - 1) / (32 / grp);
    const AmmWs w = amm_ws(a.n_head, a.hd, nb, span);
    if (ws_bytes < w.total || amm_blocks(c, c.nch) > max_grid(256) || amm_blocks(c, c.nchv) > max_grid(a.hd == 512 ? 1024 : 512)) return hipErrorInvalidValue;
    c.S = (float *)(ws + w.S);
    c.Mc = (float *)(ws + w.Mc);
    c.Lc = (double *)(ws + w.Lc);
    c.P = (float *)(ws + w.P);
#define G4_AMM(HD_, G_) \
    if (a.hd == HD_ && grp == G_) amm_go<HD_, G_>(c, s);
    G4_AMM(64, 1) G4_AMM(64, 2) G4_AMM(64, 4) G4_AMM(64, 8)
    G4_AMM(128, 1) G4_AMM(128, 2) G4_AMM(128, 4) G4_AMM(128, 8)
    G4_AMM(256, 1) G4_AMM(256, 2) G4_AMM(256, 4) G4_AMM(256, 8)
    G4_AMM(512, 1) G4_AMM(512, 2) G4_AMM(512, 4) G4_AMM(512, 8)
#undef G4_AMM
    return hipGetLastError();
}

}  // namespace g4
