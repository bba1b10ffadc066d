// k_mfma_k.hip -- batched-prefill matmul on the int8 matrix cores for K-quant
// weights (q4_K, q6_K) against q8_K activations: the many-token form of
// matmul_b (model.c:191-270) for the formats real gemma GGUFs carry, whose
// batched dots are x1 dots four times (quants.c:1535-1547).
//
// A workgroup owns a 32-token x 32-row output tile; its MMK_NW waves split
// the row's superblocks (wave w takes s = w, w + MMK_NW, ...), two
// superblocks' operands loaded at a time, and their partial tiles are summed
// through LDS in wave order.
// Per superblock every integer the reference forms is exact:
//   q4_K (quants.c:713-762): isum = sum_j sc_j * sum_32 q4 * q8 over the 8
//     sub-blocks j of 32 -- one v_mfma_i32_32x32x32_i8 per sub-block, each
//     tile scaled by the lane's row's 6-bit sc_j on the VALU (a 24-bit
//     multiply-add); summ = sum_g m_{g/2} * bsum_g over the q8_K row's 16
//     sums of 16 -- one v_mfma_f32_32x32x16_f16 whose operands (|bsum| <=
//     2048, m <= 63) and partial sums (< 2^24) are integers fp16 and fp32
//     hold exactly.  y += (d_a * d) * isum - (d_a * dmin) * summ.
//   q6_K (quants.c:582-622): per 16-element sub-block s, sum (q6 - 32) * q8 *
//     sc_s = sc_s * sum q6u * q8 - 32 * sc_s * bsum_s with q6u = q6 + 32 in
//     0..63: each sub-block is one v_mfma_i32_32x32x16_i8, scaled by sc_s on
//     the VALU; the correction sum_s sc_s * bsum_s (|.| < 2^23) is one exact
//     f16 MFMA.  y += (d_a * d) * (isum - 32 * corr).
// The fp32 products d_a * d (and d_a * dmin) of a superblock come from one
// fp32 MFMA whose only nonzero k term is each product (rounded once), in the
// integer tiles' layout.  Each wave accumulates its
// superblocks in increasing order and the waves' tiles are added in wave
// order, so a token's result does not depend on the batch size (the x4
// contract of g4run.h:148-157 within this family); the fp32 order differs
// from the CPU dots' within the path's tolerance.
//
// Two kernels with the same arithmetic and the same bits: k_mmk reads given
// q8_K rows as they are (d f32 | 256 int8 | 16 int16 bsums, 292 bytes a
// superblock; a lane's 16-byte operand slices are 4-byte-aligned loads) and
// needs no scratch; k_mmk_tile takes fp32 tokens through the quantizer launch,
// which writes them in operand order.
#include <algorithm>
#include <cstdio>

#include "formats.h"
#include "kernels.h"

namespace g4 {

typedef int mk_v2i __attribute__((ext_vector_type(2)));
typedef int mk_v4i __attribute__((ext_vector_type(4)));
typedef int mk_v16i __attribute__((ext_vector_type(16)));
typedef float mk_v16f __attribute__((ext_vector_type(16)));
typedef float mk_v32f __attribute__((ext_vector_type(32)));
typedef _Float16 mk_v8h __attribute__((ext_vector_type(8)));

constexpr int MMK_NW = 8;             // waves per workgroup, splitting the superblocks of one 32 x 32 tile

__device__ __forceinline__ mk_v4i mk_ld(const uint8_t *p) { return *(const mk_v4i *)p; }
// activations: given q8_K rows, and the ragged last tile of the operand layout,
// are 4-byte aligned (one global load all the same)
typedef int mk_v4i4 __attribute__((ext_vector_type(4), aligned(4)));
typedef int mk_v2i4 __attribute__((ext_vector_type(2), aligned(4)));
static_assert(alignof(mk_v4i4) == 4 && alignof(mk_v2i4) == 4, "superblocks of 292 bytes");
__device__ __forceinline__ mk_v4i mk_ld_act(const uint8_t *p) { return *(const mk_v4i4 *)p; }
__device__ __forceinline__ mk_v16i mk_mma(mk_v4i a, mk_v4i b, mk_v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ mk_v16i mk_mma16(mk_v2i a, mk_v2i b, mk_v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x16_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}
__device__ __forceinline__ mk_v16f mk_mma_h(mk_v8h a, mk_v8h b) {
    const mk_v16f z = {};
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, z, 0, 0, 0);
}

// the lane's slice of one q8_K superblock of its token: quants 32 j + 16 kh
// .. + 15 of every sub-block j, bsums 8 kh .. 8 kh + 7, and d
struct MkAct {
    mk_v4i q[8], bs;
    float d;
};
__device__ __forceinline__ void mk_load_act(MkAct &a, const uint8_t *ab, int kh) {
#pragma unroll
    for (int j = 0; j < 8; j++) a.q[j] = mk_ld_act(ab + 4 + 32 * j + 16 * kh);
    a.bs = mk_ld_act(ab + 260 + 16 * kh);
    a.d = *(const float *)ab;
}
// the 8 int16 bsums as fp16 (exact: |bsum| <= 16 * 128)
__device__ __forceinline__ mk_v8h mk_bsums(const mk_v4i &bs) {
    mk_v8h h;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        h[2 * k] = (_Float16)(short)(bs[k] & 0xffff);
        h[2 * k + 1] = (_Float16)(short)((uint32_t)bs[k] >> 16);
    }
    return h;
}

// one q4_K superblock: exact isum tile, exact summ tile, and the scale
// products (P[0..15] = d_a d, P[16..31] = d_a dmin)
struct Q4KSb {
    static constexpr int T = Q4_K, SEG = 2;                              // superblocks whose loads go out together
    // the lane's row: 16-byte header (d | dmin | 12 scale bytes) and its
    // k-half of the 4 nibble rows of 32 bytes
    struct W {
        mk_v4i hdr, q[4];
    };
    static __device__ __forceinline__ void load(W &w, const g4h_tensor &Wt, int64_t row, int s, int kh) {
        const uint8_t *b = Wt.qs + ((size_t)row * Wt.nb + s) * 144;
        w.hdr = mk_ld(b);
#pragma unroll
        for (int p = 0; p < 4; p++) w.q[p] = mk_ld(b + 16 + 32 * p + 16 * kh);
    }
    // 6-bit scale and min of sub-block j (quants.c:417-423, get_scale_min_k4)
    static __device__ __forceinline__ void scale_min(const mk_v4i &hdr, int j, int &sc, int &m) {
        const uint32_t w0 = (uint32_t)hdr.y, w1 = (uint32_t)hdr.z, w2 = (uint32_t)hdr.w;   // scale bytes 0..11
        auto byte = [&](int i) -> int { return (int)(((i < 4 ? w0 : i < 8 ? w1 : w2) >> (8 * (i & 3))) & 0xff); };
        if (j < 4) {
            sc = byte(j) & 63;
            m = byte(j + 4) & 63;
        } else {
            sc = (byte(j + 4) & 0xF) | ((byte(j - 4) >> 6) << 4);
            m = (byte(j + 4) >> 4) | ((byte(j) >> 6) << 4);
        }
    }
    static __device__ __forceinline__ void load_act(MkAct &a, const uint8_t *ab, int kh) { mk_load_act(a, ab, kh); }
    static __device__ __forceinline__ void mul(const W &w, const MkAct &a, int kh, mk_v16f &acc) {
        const mk_v16i z = {};
        mk_v16i isum = {};
        int mn[8];
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const mk_v4i lo = w.q[p] & 0x0F0F0F0F, hi = (w.q[p] >> 4) & 0x0F0F0F0F;
            int sc0, sc1;
            scale_min(w.hdr, 2 * p, sc0, mn[2 * p]);
            scale_min(w.hdr, 2 * p + 1, sc1, mn[2 * p + 1]);
            const mk_v16i i0 = mk_mma(a.q[2 * p], lo, z), i1 = mk_mma(a.q[2 * p + 1], hi, z);
#pragma unroll
            for (int r = 0; r < 16; r++) isum[r] = __mul24(sc1, i1[r]) + (__mul24(sc0, i0[r]) + isum[r]);
        }
        // weight operand of summ: m of bsums 8 kh .. 8 kh + 7, sub-blocks 4 kh .. 4 kh + 3
        mk_v8h mh;
#pragma unroll
        for (int t = 0; t < 4; t++) mh[2 * t] = mh[2 * t + 1] = (_Float16)(kh ? mn[4 + t] : mn[t]);
        const mk_v16f summ = mk_mma_h(mk_bsums(a.bs), mh);
        const float dw = h2f((uint16_t)((uint32_t)w.hdr.x & 0xffff)), dm = h2f((uint16_t)((uint32_t)w.hdr.x >> 16));
        const mk_v32f zf = {};
        const mk_v32f P = __builtin_amdgcn_mfma_f32_32x32x1f32(a.d, kh ? dm : dw, zf, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            acc[r] = __builtin_fmaf(P[r], (float)isum[r], acc[r]);
            acc[r] = __builtin_fmaf(-P[16 + r], summ[r], acc[r]);
        }
    }
};

// one q6_K superblock: ql [128], qh [64], int8 scales [16], fp16 d in the
// resident planes.  Group (h, j) of 32 elements 128 h + 32 j + e takes
// ql[64 h + 32 (j & 1) + e] (low nibble for j < 2, high for j >= 2) and bits
// 2 j, 2 j + 1 of qh[32 h + e]; its sub-blocks of 16 are 8 h + 2 j and
// 8 h + 2 j + 1 (quants.c:582-622).  Lane half kh holds elements 8 kh .. + 7
// and 16 + 8 kh .. + 7 of every group, activations and weights alike, so
// each sub-block is one v_mfma_i32_32x32x16_i8 on 8 bytes of each operand.
struct Q6KSb {
    static constexpr int T = Q6_K, SEG = 1;
    struct W {
        mk_v4i l0[2], l1[2], hb[2], sc;
        uint16_t d;
    };
    static __device__ __forceinline__ mk_v4i ld_split(const uint8_t *p) {
        const mk_v2i a = *(const mk_v2i *)p, b = *(const mk_v2i *)(p + 16);
        return mk_v4i{a.x, a.y, b.x, b.y};
    }
    static __device__ __forceinline__ void load(W &w, const g4h_tensor &Wt, int64_t row, int s, int kh) {
        const size_t j = (size_t)row * Wt.nb + s;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint8_t *ql = Wt.qs + j * 128 + 64 * h + 8 * kh;
            w.l0[h] = ld_split(ql);
            w.l1[h] = ld_split(ql + 32);
            w.hb[h] = ld_split(Wt.ex + j * 64 + 32 * h + 8 * kh);
        }
        w.sc = mk_ld(Wt.sc + j * 16);
        w.d = ((const uint16_t *)Wt.dd)[j];
    }
    static __device__ __forceinline__ void load_act(MkAct &a, const uint8_t *ab, int kh) {
#pragma unroll
        for (int g = 0; g < 8; g++) {
            const mk_v2i lo = *(const mk_v2i4 *)(ab + 4 + 32 * g + 8 * kh), hi = *(const mk_v2i4 *)(ab + 20 + 32 * g + 8 * kh);
            a.q[g] = mk_v4i{lo.x, lo.y, hi.x, hi.y};
        }
        a.bs = mk_ld_act(ab + 260 + 16 * kh);
        a.d = *(const float *)ab;
    }
    static __device__ __forceinline__ void mul(const W &w, const MkAct &a, int kh, mk_v16f &acc) {
        const mk_v16i z = {};
        auto scb = [&](int s) { return (int)(int8_t)(((uint32_t)w.sc[s >> 2] >> (8 * (s & 3))) & 0xff); };
        mk_v16i isum = {};
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const mk_v4i &L = (j & 1) ? w.l1[h] : w.l0[h];
                mk_v4i q = ((L >> (j >= 2 ? 4 : 0)) & 0x0F0F0F0F) | (((w.hb[h] >> (2 * j)) & 0x03030303) << 4);
                const int s0 = 8 * h + 2 * j;
                const int c0 = scb(s0), c1 = scb(s0 + 1);
                const mk_v4i &x = a.q[4 * h + j];
                // the group's weight operand waits for the previous group's
                // multiply-adds: the compiler would otherwise issue all 16
                // MFMAs first and hold 256 result registers
                asm volatile("" : "+v"(q) : "v"(isum[15]));
                const mk_v16i i0 = mk_mma16(x.xy, q.xy, z), i1 = mk_mma16(x.zw, q.zw, z);
#pragma unroll
                for (int r = 0; r < 16; r++) isum[r] = __mul24(c1, i1[r]) + (__mul24(c0, i0[r]) + isum[r]);
            }
        }
        // weight operand of the correction: sc of bsums (= sub-blocks) 8 kh .. 8 kh + 7
        mk_v8h ch;
#pragma unroll
        for (int t = 0; t < 8; t++) ch[t] = (_Float16)(kh ? scb(8 + t) : scb(t));
        const mk_v16f corr = mk_mma_h(mk_bsums(a.bs), ch);
        // d_a * d in the tiles' layout: one k term of two, the other zero
        const mk_v16f zf = {};
        const mk_v16f P = __builtin_amdgcn_mfma_f32_32x32x2f32(kh ? 0.0f : a.d, h2f(w.d), zf, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = __builtin_fmaf(P[r], (float)(isum[r] - 32 * (int)corr[r]), acc[r]);
    }
};

// One workgroup per (row tile, token tile) of 32 x 32.  Workgroup b runs on
// XCD b % 8: row tiles r with r % 8 == b % 8 go there, the token tiles of a
// row tile consecutively, so they find its weights in that XCD's L2.  The
// grid is padded to whole groups of 8 row tiles; padding workgroups return.
template <class S>
__global__ __launch_bounds__(64 * MMK_NW) void k_mmk(g4h_tensor W, const uint8_t *__restrict__ act, size_t stride, int M,
                                                     float *__restrict__ Y, int ntok) {
    __shared__ float part[MMK_NW][32][33];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 31, kh = lane >> 5;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int64_t rt = (int64_t)(l / ntok) * 8 + x;
    const int m0 = (l % ntok) * 32;
    if (rt * 32 >= W.nrows) return;                                      // uniform over the workgroup
    const int64_t n0 = rt * 32;
    const int64_t row = std::min<int64_t>(n0 + li, W.nrows - 1);
    const uint8_t *arow = act + (size_t)std::min(m0 + li, M - 1) * stride;
    const int nb = (int)W.nb;
    mk_v16f acc = {};
    // the wave's superblocks s = wave, wave + MMK_NW, .. two at a time: both
    // superblocks' operands are loaded before the first multiply, in
    // straight-line code (a register ring carried around the loop was undone
    // by the compiler: its loads sank to their uses, several round trips per
    // superblock)
    // q4_K: a lone last superblock is loaded twice; its second multiply gets the
    // activation scale 0, so its products add +0 to an accumulator that never
    // holds -0 (no branch: the compiler would sink that superblock's loads
    // into it).
    for (int s0 = wave; s0 < nb; s0 += S::SEG * MMK_NW) {               // uniform over the wave
        if constexpr (S::SEG == 2) {
            const bool two = s0 + MMK_NW < nb;
            const int s1 = two ? s0 + MMK_NW : s0;
            typename S::W w0, w1;
            MkAct a0, a1;
            S::load(w0, W, row, s0, kh);
            S::load_act(a0, arow + (size_t)s0 * 292, kh);
            S::load(w1, W, row, s1, kh);
            S::load_act(a1, arow + (size_t)s1 * 292, kh);
            if (!two) a1.d = 0.0f;
            __builtin_amdgcn_sched_barrier(0);
            S::mul(w0, a0, kh, acc);
            __builtin_amdgcn_sched_barrier(0);
            S::mul(w1, a1, kh, acc);
        } else {                                                          // q6_K: two superblocks' operands spill
            typename S::W w0;
            MkAct a0;
            S::load(w0, W, row, s0, kh);
            S::load_act(a0, arow + (size_t)s0 * 292, kh);
            S::mul(w0, a0, kh, acc);
        }
    }
    // C[i][j]: j = lane % 32 (weight row), i = 8 (r / 4) + 4 kh + r % 4 (token)
#pragma unroll
    for (int r = 0; r < 16; r++) part[wave][8 * (r >> 2) + 4 * kh + (r & 3)][li] = acc[r];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 32 * 32 / (64 * MMK_NW); h++) {
        const int o = threadIdx.x + 64 * MMK_NW * h, i = o >> 5, j = o & 31;
        float v = part[0][i][j];
#pragma unroll
        for (int w = 1; w < MMK_NW; w++) v += part[w][i][j];
        const int m = m0 + i;
        const int64_t n = n0 + j;
        if (m < M && n < W.nrows) Y[(size_t)m * W.nrows + n] = v;
    }
}

// The same sums from fp32 tokens (the usual call): the quantizer launch writes
// the activations in operand order (k_quantize_q8_K_tile), so a wave's operand
// load is 1 KB of adjacent bytes, and each wave owns MT token tiles of its row
// tile, whose weights it loads in runs of adjacent bytes and turns into
// operands through LDS of its own (no barrier).  k_mmk's operand loads have
// adjacent lanes in different rows, one L1 access per lane, and the L1's one
// access per clock bounds it.  Measured at 4096 x 11008, quantizer included
// (us, k_mmk / this): q4_K at 9 / 64 / 128 / 509 tokens 20.4 / 25.8 / 45.4 /
// 165 -> 15.8 / 18.3 / 25.1 / 82.8 (554 TOPS); q6_K at 9 / 64 / 509 tokens 30.3
// / 38.5 / 250 -> 21.6 / 23.2 / 112; q6_K 2048 x 6144 at 64 26.9 -> 14.3.  What
// bounds it at 509 tokens: 1.0 GB of operands from L2 and 38 us of VALU issue
// (the scale multiply-adds), partly overlapped.
// The waves split the superblocks as k_mmk's do, each superblock's integers
// and scale products are the same, and the partial tiles are added in the same
// order: k_mmk's bits.  The next superblock's operands are loaded as the
// current one's are used up.  q6_K's sub-blocks take the signed q6 - 32
// directly: the integers of sum q6u q8 - 32 bsum.
struct Q4KTile {
    static constexpr int T = Q4_K, WL = 5, ROW = 144, LDSB = 32 * ROW;   // loads per lane, LDS bytes per row and wave
    struct W {
        mk_v4i v[WL];
    };
    struct Ptr {
        const uint8_t *p[WL];
    };
    struct Head {
        mk_v4i hdr;
        uint32_t sc[2], mn[2];
    };
    // 9 lanes per row of 144 bytes; past the 288 pieces the last one again
    static __device__ __forceinline__ void piece(int lane, int i, int &r, int &c) {
        const int f = min(64 * i + lane, 287);
        r = f / 9, c = f - 9 * r;
    }
    static __device__ __forceinline__ void init(Ptr &P, const g4h_tensor &Wt, int64_t n0, int lane) {
#pragma unroll
        for (int i = 0; i < WL; i++) {
            int r, c;
            piece(lane, i, r, c);
            P.p[i] = Wt.qs + (size_t)std::min<int64_t>(n0 + r, Wt.nrows - 1) * Wt.nb * 144 + 16 * c;
        }
    }
    static __device__ __forceinline__ void load(W &w, const Ptr &P, int s) {
#pragma unroll
        for (int i = 0; i < WL; i++) w.v[i] = mk_ld(P.p[i] + (size_t)s * 144);
    }
    static __device__ __forceinline__ void put(const W &w, uint8_t *lds, int lane) {
#pragma unroll
        for (int i = 0; i < WL; i++) {
            int r, c;
            piece(lane, i, r, c);
            *(mk_v4i *)(lds + r * ROW + 16 * c) = w.v[i];
        }
    }
    // the row's 6-bit scales and mins (quants.c:417-423), four to a word
    static __device__ __forceinline__ Head head(const uint8_t *lds, int li) {
        Head h;
        h.hdr = *(const mk_v4i *)(lds + li * ROW);
        const uint32_t w0 = (uint32_t)h.hdr.y, w1 = (uint32_t)h.hdr.z, w2 = (uint32_t)h.hdr.w;
        h.sc[0] = w0 & 0x3f3f3f3fu;
        h.mn[0] = w1 & 0x3f3f3f3fu;
        h.sc[1] = (w2 & 0x0f0f0f0fu) | ((w0 >> 2) & 0x30303030u);
        h.mn[1] = ((w2 >> 4) & 0x0f0f0f0fu) | ((w1 >> 2) & 0x30303030u);
        return h;
    }
};

struct Q6KTile {
    static constexpr int T = Q6_K, WL = 7, QL = 144, QH = 80, LDSB = 32 * (QL + QH);
    struct W {
        mk_v4i v[WL];                                                // ql, qh, scales
        uint16_t d;
    };
    struct Ptr {
        const uint8_t *ql[4], *qh[2], *sc, *dd;
    };
    static __device__ __forceinline__ void init(Ptr &P, const g4h_tensor &Wt, int64_t n0, int lane) {
        auto row = [&](int r) { return (size_t)std::min<int64_t>(n0 + r, Wt.nrows - 1) * Wt.nb; };
#pragma unroll
        for (int i = 0; i < 4; i++) P.ql[i] = Wt.qs + row(8 * i + (lane >> 3)) * 128 + 16 * (lane & 7);
#pragma unroll
        for (int i = 0; i < 2; i++) P.qh[i] = Wt.ex + row(16 * i + (lane >> 2)) * 64 + 16 * (lane & 3);
        P.sc = Wt.sc + row(lane & 31) * 16;
        P.dd = Wt.dd + row(lane & 31) * 2;
    }
    static __device__ __forceinline__ void load(W &w, const Ptr &P, int s) {
#pragma unroll
        for (int i = 0; i < 4; i++) w.v[i] = mk_ld(P.ql[i] + (size_t)s * 128);
#pragma unroll
        for (int i = 0; i < 2; i++) w.v[4 + i] = mk_ld(P.qh[i] + (size_t)s * 64);
        w.v[6] = mk_ld(P.sc + (size_t)s * 16);
        w.d = *(const uint16_t *)(P.dd + (size_t)s * 2);
    }
    static __device__ __forceinline__ void put(const W &w, uint8_t *lds, int lane) {
#pragma unroll
        for (int i = 0; i < 4; i++) *(mk_v4i *)(lds + (8 * i + (lane >> 3)) * QL + 16 * (lane & 7)) = w.v[i];
#pragma unroll
        for (int i = 0; i < 2; i++) *(mk_v4i *)(lds + 32 * QL + (16 * i + (lane >> 2)) * QH + 16 * (lane & 3)) = w.v[4 + i];
    }
    static __device__ __forceinline__ mk_v4i split(const uint8_t *p) {
        const mk_v2i a = *(const mk_v2i *)p, b = *(const mk_v2i *)(p + 16);
        return mk_v4i{a.x, a.y, b.x, b.y};
    }
};

// isum += c * i over a result tile, one v_mad_i32_i24 per value: the empty asm
// keeps the compiler from splitting two of them into two multiplies and a
// three-operand add
__device__ __forceinline__ void mk_mad(mk_v16i &isum, int c, const mk_v16i &i) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
        int v = __mul24(c, i[r]) + isum[r];
        asm("" : "+v"(v));
        isum[r] = v;
    }
}

// Workgroup b runs on XCD b % 8: row tiles r with r % 8 == b % 8, the token
// tiles of a row tile consecutively (as k_mmk).
template <class S, int MT>
__global__ __launch_bounds__(64 * MMK_NW) void k_mmk_tile(g4h_tensor W, const uint8_t *__restrict__ act, int M, float *__restrict__ Y,
                                                          int ntok) {
    constexpr int PB = MMK_NW * MT * 32 * 33 * 4, WBYTES = MMK_NW * S::LDSB;
    __shared__ __align__(16) uint8_t lds[PB > WBYTES ? PB : WBYTES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
    const int li = lane & 31, kh = lane >> 5;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int64_t n0 = ((int64_t)(l / ntok) * 8 + x) * 32;
    const int m0 = (l % ntok) * (32 * MT);
    if (n0 >= W.nrows) return;                                           // uniform over the workgroup
    const int nb = (int)W.nb;
    uint8_t *wl = lds + wave * S::LDSB;
    // activation tiles (a second tile past the last token repeats the first)
    const uint8_t *ab[MT];
    int TL[MT], ao[MT], tl[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int t0 = m0 + 32 * m < M ? m0 + 32 * m : m0;
        TL[m] = min(32, M - t0);
        ab[m] = act + (size_t)t0 * nb * 292;
        tl[m] = min(li, TL[m] - 1);
        ao[m] = (kh * TL[m] + tl[m]) * 16;
    }
    typename S::Ptr P;
    S::init(P, W, n0, lane);
    typename S::W w;
    mk_v4i a[MT][8], bs[MT];
    float d[MT];
    auto load_a = [&](int m, int j, int s) __attribute__((always_inline)) {
        a[m][j] = mk_ld_act(ab[m] + (size_t)s * TL[m] * 292 + 2 * j * TL[m] * 16 + ao[m]);
    };
    auto load_s = [&](int m, int s) __attribute__((always_inline)) {
        const uint8_t *b = ab[m] + (size_t)s * TL[m] * 292;
        if constexpr (S::T == Q4_K) bs[m] = mk_ld_act(b + TL[m] * 256 + ao[m]);
        d[m] = *(const float *)(b + TL[m] * 288 + 4 * tl[m]);
    };
    mk_v16f acc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) acc[m] = mk_v16f{};
    const mk_v16i z = {};
    if (wave < nb) {
        S::load(w, P, wave);
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int j = 0; j < 8; j++) load_a(m, j, wave);
            load_s(m, wave);
        }
    }
    for (int s = wave; s < nb; s += MMK_NW) {                            // uniform over the wave
        const int sn = s + MMK_NW < nb ? s + MMK_NW : s;                 // the next one (the last again at the end)
        S::put(w, wl, lane);
        typename S::W wc;                                                // q6_K: scales and d of this superblock
        if constexpr (S::T == Q6_K) wc.v[6] = w.v[6], wc.d = w.d;
        asm volatile("" ::: "memory");                                   // a wave's LDS accesses complete in order
        S::load(w, P, sn);
        asm volatile("" ::: "memory");
        mk_v16i isum[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) isum[m] = z;
        if constexpr (S::T == Q4_K) {
            const auto h = S::head(wl, li);
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const mk_v4i q = *(const mk_v4i *)(wl + li * S::ROW + 16 + 32 * p + 16 * kh);
                const mk_v4i lo = q & 0x0F0F0F0F, hi = (q >> 4) & 0x0F0F0F0F;
                int sc0 = (h.sc[p >> 1] >> (16 * (p & 1))) & 0xff, sc1 = (h.sc[p >> 1] >> (16 * (p & 1) + 8)) & 0xff;
                asm("" : "+v"(sc0), "+v"(sc1));                          // no byte select inside the multiplies
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const mk_v16i i0 = mk_mma(a[m][2 * p], lo, z), i1 = mk_mma(a[m][2 * p + 1], hi, z);
                    load_a(m, 2 * p, sn);
                    load_a(m, 2 * p + 1, sn);
                    asm volatile("" ::: "memory");
                    mk_mad(isum[m], sc0, i0);
                    mk_mad(isum[m], sc1, i1);
                }
            }
            // weight operand of summ: m of bsums 8 kh .. 8 kh + 7, sub-blocks 4 kh .. 4 kh + 3
            const uint32_t mn = kh ? h.mn[1] : h.mn[0];
            mk_v8h mh;
#pragma unroll
            for (int t = 0; t < 4; t++) mh[2 * t] = mh[2 * t + 1] = (_Float16)(float)((mn >> (8 * t)) & 0xff);
            const float dw = h2f((uint16_t)((uint32_t)h.hdr.x & 0xffff)), dm = h2f((uint16_t)((uint32_t)h.hdr.x >> 16));
            const mk_v32f zf = {};
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const mk_v16f summ = mk_mma_h(__builtin_bit_cast(mk_v8h, bs[m]), mh);
                const mk_v32f P2 = __builtin_amdgcn_mfma_f32_32x32x1f32(d[m], kh ? dm : dw, zf, 0, 0, 0);
                load_s(m, sn);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    acc[m][r] = __builtin_fmaf(P2[r], (float)isum[m][r], acc[m][r]);
                    acc[m][r] = __builtin_fmaf(-P2[16 + r], summ[r], acc[m][r]);
                }
            }
        } else {
            auto scb = [&](int k) { return (int)(int8_t)(((uint32_t)wc.v[6][k >> 2] >> (8 * (k & 3))) & 0xff); };
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                const mk_v4i l0 = S::split(wl + li * S::QL + 64 * hh + 8 * kh), l1 = S::split(wl + li * S::QL + 64 * hh + 32 + 8 * kh);
                const mk_v4i hb = S::split(wl + 32 * S::QL + li * S::QH + 32 * hh + 8 * kh);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const mk_v4i &L = (j & 1) ? l1 : l0;
                    mk_v4i q = ((L >> (j >= 2 ? 4 : 0)) & 0x0F0F0F0F) | (((hb >> (2 * j)) & 0x03030303) << 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) q[e] = (int)(((uint32_t)q[e] + 0x60606060u) ^ 0x80808080u);   // per byte: q - 32
                    int c0 = scb(8 * hh + 2 * j), c1 = scb(8 * hh + 2 * j + 1);
                    asm("" : "+v"(c0), "+v"(c1));                        // no byte select inside the multiplies
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const mk_v4i &xa = a[m][4 * hh + j];
                        const mk_v16i i0 = mk_mma16(xa.xy, q.xy, z), i1 = mk_mma16(xa.zw, q.zw, z);
                        load_a(m, 4 * hh + j, sn);
                        asm volatile("" ::: "memory");
                        mk_mad(isum[m], c0, i0);
                        mk_mad(isum[m], c1, i1);
                    }
                }
            }
            const mk_v16f zf = {};
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const mk_v16f P1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kh ? 0.0f : d[m], h2f(wc.d), zf, 0, 0, 0);
                load_s(m, sn);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int r = 0; r < 16; r++) acc[m][r] = __builtin_fmaf(P1[r], (float)isum[m][r], acc[m][r]);
            }
        }
    }
    __syncthreads();
    // C[i][j]: j = lane % 32 (weight row), i = 8 (r / 4) + 4 kh + r % 4 (token)
    float (*part)[MT * 32][33] = (float (*)[MT * 32][33])lds;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < 16; r++) part[wave][32 * m + 8 * (r >> 2) + 4 * kh + (r & 3)][li] = acc[m][r];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < MT * 32 * 32 / (64 * MMK_NW); h++) {
        const int o = threadIdx.x + 64 * MMK_NW * h, i = o >> 5, j = o & 31;
        float v = part[0][i][j];
#pragma unroll
        for (int k = 1; k < MMK_NW; k++) v += part[k][i][j];
        const int m = m0 + i;
        const int64_t n = n0 + j;
        if (m < M && n < W.nrows) Y[(size_t)m * W.nrows + n] = v;
    }
}

bool mmk_capable(int type) { return type == Q4_K || type == Q6_K; }

static void mmk_grid(const g4h_tensor &W, int M, int64_t &grid, int &ntok) {
    ntok = (M + 31) / 32;
    grid = (W.nrows + 255) / 256 * 8 * ntok;
}

hipError_t launch_matmul_mfma_k(const g4h_tensor &W, const uint8_t *act, size_t stride, int M, float *Y, hipStream_t s) {
    if (!mmk_capable(W.type) || M < 1 || !act || !Y || stride % 4 || stride < (size_t)W.nb * 292) return hipErrorInvalidValue;
    int64_t grid;
    int ntok;
    mmk_grid(W, M, grid, ntok);
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    if (W.type == Q4_K) hipLaunchKernelGGL(k_mmk<Q4KSb>, dim3((unsigned)grid), dim3(64 * MMK_NW), 0, s, W, act, stride, M, Y, ntok);
    else hipLaunchKernelGGL(k_mmk<Q6KSb>, dim3((unsigned)grid), dim3(64 * MMK_NW), 0, s, W, act, stride, M, Y, ntok);
    return hipGetLastError();
}

// token tiles per wave: two (each weight load and unpack serving 64 tokens)
// once there are two and that still gives every CU a workgroup.  Measured (us,
// one / two): q4_K 4096 x 11008 at 64 tokens 18.7 / 25.3, at 128 31.1 / 25.9;
// q4_K 8192 x 4096 at 33 tokens 14.8 / 12.6.  Up to 32 tokens the second tile is
// all padding: q4_K 10240 x 4096 at 9 tokens 13.9 / 18.9, q6_K 20480 x 4096 at
// 32 30.5 / 40.8.
static int mmk_mt(const g4h_tensor &W, int M) { return M > 32 && (W.nrows + 31) / 32 * ((M + 63) / 64) >= 256 ? 2 : 1; }

// fp32 tokens that k_mmk takes all the same, quantized to rows: q6_K rows of one
// superblock, where one wave of eight works and the time is its longest chain,
// shorter by the LDS pass in k_mmk.  Up to 64 tokens, or while every CU has at
// most one workgroup (us, k_mmk / k_mmk_tile: 4096 x 256 at 9 / 64 tokens 6.8 / 7.1,
// 7.2 / 7.4; 20480 x 256 at 9 11.4 / 12.4; 256 x 256 at 512 7.2 / 7.4); past both
// the loads decide (4096 x 256 at 100 tokens 9.8 / 9.0).  q4_K is faster in
// k_mmk_tile everywhere.
static bool mmk_from_rows(const g4h_tensor &W, int M) {
    return W.type == Q6_K && W.nb == 1 && (M <= 64 || (W.nrows + 31) / 32 * ((M + 31) / 32) <= 256);
}

hipError_t launch_matmul_mfma_kx(const g4h_tensor &W, const float *x, size_t xs, int M, float *Y, uint8_t *ws, hipStream_t s) {
    if (!mmk_capable(W.type) || M < 1 || !x || !Y || (uintptr_t)ws % 64) return hipErrorInvalidValue;
    if (mmk_from_rows(W, M)) {
        const size_t stride = 292;                                   // one superblock
        if (hipError_t e = launch_quantize_q8_K(x, xs, ws, stride, W.ncols, M, s)) return e;
        return launch_matmul_mfma_k(W, ws, stride, M, Y, s);
    }
    if (hipError_t e = launch_quantize_q8_K_tile(x, xs, ws, W.ncols, M, W.type, s)) return e;
    const int mt = mmk_mt(W, M), ntok = (M + 32 * mt - 1) / (32 * mt);
    const int64_t grid = (W.nrows + 255) / 256 * 8 * ntok;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 g((unsigned)grid), b(64 * MMK_NW);
    if (W.type == Q4_K) {
        if (mt == 1) hipLaunchKernelGGL((k_mmk_tile<Q4KTile, 1>), g, b, 0, s, W, ws, M, Y, ntok);
        else hipLaunchKernelGGL((k_mmk_tile<Q4KTile, 2>), g, b, 0, s, W, ws, M, Y, ntok);
    } else {
        if (mt == 1) hipLaunchKernelGGL((k_mmk_tile<Q6KTile, 1>), g, b, 0, s, W, ws, M, Y, ntok);
        else hipLaunchKernelGGL((k_mmk_tile<Q6KTile, 2>), g, b, 0, s, W, ws, M, Y, ntok);
    }
    return hipGetLastError();
}

void mmk_describe(const g4h_tensor &W, int M, char *buf, size_t len) {
    const char *type = W.type == Q4_K ? "q4_K" : "q6_K";
    if (mmk_from_rows(W, M)) {
        int64_t grid;
        int ntok;
        mmk_grid(W, M, grid, ntok);
        snprintf(buf, len, "k_mmk<%s> grid=%lld block=%d (int8 MFMA, 32x32 tiles, %d waves split the superblocks; fp32 x quantized to rows)", type,
                 (long long)grid, 64 * MMK_NW, MMK_NW);
        return;
    }
    const int mt = mmk_mt(W, M), ntok = (M + 32 * mt - 1) / (32 * mt);
    snprintf(buf, len, "k_mmk_tile<%s,mt=%d> grid=%lld block=%d (int8 MFMA, %dx32 tiles, %d waves split the superblocks; given rows take k_mmk)",
             type, mt, (long long)((W.nrows + 255) / 256 * 8 * ntok), 64 * MMK_NW, 32 * mt, MMK_NW);
}

}  // namespace g4
