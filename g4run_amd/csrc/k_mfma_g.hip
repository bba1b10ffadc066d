// k_mfma_g.hip -- prompt batches over q5_K, q3_K, q2_K and tq2_0 weights on the
// int8 matrix cores with the GEMV family's sums: the bits of the GEMV kernels
// (gemv.h), so the two are one kernel family (g4run.h:148-157).
//
// A GEMV row's LPR lanes each take every LPR-th unit of 64 elements (a quarter
// superblock) in increasing order, one or two fmas per unit on exact integers,
// and the lanes are added in a butterfly over 1, 2, 4, ..  Unit 4 s + p goes to
// lane (4 s + p) % LPR, so the superblocks s of one class s % (LPR / 4) feed four
// neighbouring lanes.  Here a wave owns whole classes of a 32-token x 32-row
// tile: four accumulator tiles (one per p) take the units' integers from the
// MFMAs through the same fmas, (p0 + p1) + (p2 + p3) is the butterfly's first two
// levels, and the classes are added in the butterfly's order, the last levels
// through LDS.
//
// Integers of a unit (all exact):
//   q5_K  (quants.c:764-818): sc0 * i0 + sc1 * i1, one v_mfma_i32_32x32x32_i8
//         per 32 elements, scaled on the VALU (q * sc needs 11 bits).
//   q2_K  (quants.c:425-445): q * sc <= 45 fits the operand's byte, so the unit
//         is two v_mfma_i32_32x32x32_i8 on scaled weights.
//   q3_K  (quants.c:447-477): sc * (4 - t) lies in -128 .. 124 (sc -32 .. 31, t =
//         0 .. 7), so the same two MFMAs give minus the unit's integer.
//   tq2_0 (quants.c:564-580): t - 1 as bytes, no scales.
// The minima times the activation's sums of 16 (q5_K, q2_K) are one f16 MFMA
// whose operands and sums are integers that fp16 and fp32 hold exactly.
//
// The GEMV family ran a batch as one launch per 8 tokens or fewer (4 at 11008
// columns), each reading the weights again and bounded by its LDS reads of the
// activations.  Measured at 4096 x 11008, quantizer included (us, GEMV chunks /
// this): q5_K at 9 / 64 / 509 tokens 37.1 / 214 / 1684 -> 20.7 / 23.2 / 160,
// q3_K 33.2 / 198 / 1535 -> 22.1 / 23.5 / 159, q2_K 28.6 / 173 / 1351 -> 16.2 /
// 18.8 / 125, tq2_0 24.2 / 147 / 1149 -> 12.4 / 15.0 / 94.5 (486 TOPS).  What
// bounds it at 509 tokens: the VALU, with four units' conversions and fmas per
// superblock and output (the GEMV's roundings) and the scale products, at two
// waves per SIMD (four accumulator tiles, 165 to 256 registers; q5_K's form of
// 16 classes spills 4 of them, 20 bytes of scratch, and its form of 4 classes
// takes 276, one wave per SIMD).
#include <algorithm>
#include <cstdio>

#include "formats.h"
#include "kernels.h"

namespace g4 {

typedef int mg_v2i __attribute__((ext_vector_type(2)));
typedef int mg_v4i __attribute__((ext_vector_type(4)));
typedef int mg_v16i __attribute__((ext_vector_type(16)));
typedef float mg_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 mg_v8h __attribute__((ext_vector_type(8)));
typedef unsigned short mg_v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ mg_v4i mg_ld(const uint8_t *p) { return *(const mg_v4i *)p; }
// activations: the ragged last tile of the layout is 4-byte aligned (one global
// load all the same)
typedef int mg_v4i4 __attribute__((ext_vector_type(4), aligned(4)));
static_assert(alignof(mg_v4i4) == 4, "superblocks of TL * 292 bytes");
__device__ __forceinline__ mg_v4i mg_ld_act(const uint8_t *p) { return *(const mg_v4i4 *)p; }
__device__ __forceinline__ mg_v16i mg_mma(mg_v4i a, mg_v4i b, mg_v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ uint32_t mg_pkmul(uint32_t a, uint32_t b) {   // 16-bit halves, modulo 2^16
    return __builtin_bit_cast(uint32_t, (mg_v2u)(__builtin_bit_cast(mg_v2u, a) * __builtin_bit_cast(mg_v2u, b)));
}
__device__ __forceinline__ uint32_t mg_pkadd(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (mg_v2u)(__builtin_bit_cast(mg_v2u, a) + __builtin_bit_cast(mg_v2u, b)));
}

// a wave's weights of one superblock: 32 rows, loaded in runs of adjacent bytes
// (q5_K: the GGUF block, 11 lanes per row; the others: 4 lanes per row of 64
// quant bytes, and for q3_K 2 per row of 32 hmask bytes) and passed through LDS;
// scales and d straight from the lane's row
template <int T>
struct MgW {
    static constexpr bool Q5 = T == Q5_K;
    static constexpr int WL = Q5 ? 6 : T == Q3_K ? 3 : 2, ROW = Q5 ? 176 : 80, HM = 48, LDSB = 32 * (ROW + (T == Q3_K ? HM : 0));
    mg_v4i v[WL];
    mg_v4i sc;
    uint32_t dd;
    static __device__ __forceinline__ void piece(int lane, int i, int &r, int &c) {
        if constexpr (Q5) {
            const int f = min(64 * i + lane, 351);                       // past the 352 pieces the last one again
            r = f / 11, c = f - 11 * r;
        } else {
            r = 16 * i + (lane >> 2), c = lane & 3;
        }
    }
    struct Ptr {
        const uint8_t *p[WL], *sc, *dd;
    };
    static __device__ __forceinline__ void init(Ptr &P, const g4h_tensor &Wt, int64_t n0, int lane) {
        auto blk = [&](int r) { return (size_t)std::min<int64_t>(n0 + r, Wt.nrows - 1) * Wt.nb; };
#pragma unroll
        for (int i = 0; i < (Q5 ? 6 : 2); i++) {
            int r, c;
            piece(lane, i, r, c);
            P.p[i] = Wt.qs + blk(r) * (Q5 ? 176 : 64) + 16 * c;
        }
        if constexpr (T == Q3_K) P.p[2] = Wt.ex + blk(lane >> 1) * 32 + 16 * (lane & 1);
        if constexpr (T == Q2_K) P.sc = Wt.sc + blk(lane & 31) * 16, P.dd = Wt.ex + blk(lane & 31) * 4;
        if constexpr (T == Q3_K) P.sc = Wt.sc + blk(lane & 31) * 12, P.dd = Wt.dd + blk(lane & 31) * 2;
        if constexpr (T == TQ2_0) P.dd = Wt.sc + blk(lane & 31) * 2;
    }
    __device__ __forceinline__ void load(const Ptr &P, int s) {
#pragma unroll
        for (int i = 0; i < (Q5 ? 6 : 2); i++) v[i] = mg_ld(P.p[i] + (size_t)s * (Q5 ? 176 : 64));
        if constexpr (T == Q3_K) {
            v[2] = mg_ld(P.p[2] + (size_t)s * 32);
            const uint32_t *w = (const uint32_t *)(P.sc + (size_t)s * 12);
            sc.x = (int)w[0], sc.y = (int)w[1], sc.z = (int)w[2];
        }
        if constexpr (T == Q2_K) sc = mg_ld(P.sc + (size_t)s * 16), dd = *(const uint32_t *)(P.dd + (size_t)s * 4);
        if constexpr (T == Q3_K || T == TQ2_0) dd = *(const uint16_t *)(P.dd + (size_t)s * 2);
    }
    __device__ __forceinline__ void put(uint8_t *lds, int lane) const {
#pragma unroll
        for (int i = 0; i < (Q5 ? 6 : 2); i++) {
            int r, c;
            piece(lane, i, r, c);
            *(mg_v4i *)(lds + r * ROW + 16 * c) = v[i];
        }
        if constexpr (T == Q3_K) *(mg_v4i *)(lds + 32 * ROW + (lane >> 1) * HM + 16 * (lane & 1)) = v[2];
    }
};

// NC classes of superblocks (LPR / 4) over NW waves.  Workgroup b runs on XCD
// b % 8: row tiles r with r % 8 == b % 8, the token tiles of a row tile
// consecutively, so they find its weights in that XCD's L2; padding workgroups
// return.  Activations: launch_quantize_q8_K_tile's layout for T.
template <int T, int NC>
__global__ __launch_bounds__(NC < 8 ? 256 : 512) void k_mmg(g4h_tensor W, const uint8_t *__restrict__ act, int M, float *__restrict__ Y,
                                                            int ntok) {
    using WT = MgW<T>;
    constexpr int NW = NC < 8 ? NC : 8, CPW = NC / NW;
    constexpr bool MINS = T == Q5_K || T == Q2_K;
    constexpr int PB = NW * 32 * 33 * 4, WB = NW * WT::LDSB;
    __shared__ __align__(16) uint8_t lds[PB > WB ? PB : WB];
    __shared__ __align__(16) float dl[NW][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
    const int li = lane & 31, kh = lane >> 5;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int64_t n0 = ((int64_t)(l / ntok) * 8 + x) * 32;
    const int m0 = (l % ntok) * 32;
    if (n0 >= W.nrows) return;                                           // uniform over the workgroup
    const int nb = (int)W.nb;
    uint8_t *wl = lds + wave * WT::LDSB;
    const int TL = min(32, M - m0), tl = min(li, TL - 1), ao = (kh * TL + tl) * 16;
    const uint8_t *ab = act + (size_t)m0 * nb * 292;
    typename WT::Ptr P;
    WT::init(P, W, n0, lane);
    WT w;
    mg_v4i a[8], bs;
    float d;
    const mg_v16i z = {};
    const mg_v16f zf = {};
    auto load_a = [&](int j, int s) __attribute__((always_inline)) { a[j] = mg_ld_act(ab + (size_t)s * TL * 292 + 2 * j * TL * 16 + ao); };
    auto load_s = [&](int s) __attribute__((always_inline)) {
        const uint8_t *b = ab + (size_t)s * TL * 292;
        if constexpr (MINS) bs = mg_ld_act(b + TL * 256 + ao);
        d = *(const float *)(b + TL * 288 + 4 * tl);
    };
    if (wave * CPW < nb) {
        w.load(P, wave * CPW);
#pragma unroll
        for (int j = 0; j < 8; j++) load_a(j, wave * CPW);
        load_s(wave * CPW);
    }
    mg_v16f tot;
#pragma unroll 1
    for (int ci = 0; ci < CPW; ci++) {
        const int cls = wave * CPW + ci;
        mg_v16f acc[4] = {};
        for (int s = cls; s < nb; s += NC) {                             // uniform over the wave
            // the wave's next superblock (the last again at the end)
            const int sn = s + NC < nb ? s + NC : ci + 1 < CPW && cls + 1 < nb ? cls + 1 : s;
            w.put(wl, lane);
            if (kh == 0) dl[wave][li] = d;
            const mg_v4i sc = w.sc;
            uint32_t dd = w.dd;
            asm volatile("" ::: "memory");                               // a wave's LDS accesses complete in order
            w.load(P, sn);
            asm volatile("" ::: "memory");
            mg_v4i hdr;
            if constexpr (T == Q5_K) hdr = mg_ld(wl + li * WT::ROW), dd = (uint32_t)hdr.x;
            const float dw = h2f((uint16_t)(dd & 0xffff)), dm = h2f((uint16_t)(dd >> 16));
            float da[16];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 f = *(const float4 *)&dl[wave][8 * q + 4 * kh];
                da[4 * q] = f.x, da[4 * q + 1] = f.y, da[4 * q + 2] = f.z, da[4 * q + 3] = f.w;
            }
            // q5_K: 6-bit scales and mins, four to a word (quants.c:417-423)
            uint32_t s5[2], m5[2];
            mg_v4i hb;
            if constexpr (T == Q5_K) {
                const uint32_t w0 = (uint32_t)hdr.y, w1 = (uint32_t)hdr.z, w2 = (uint32_t)hdr.w;
                s5[0] = w0 & 0x3f3f3f3fu;
                m5[0] = w1 & 0x3f3f3f3fu;
                s5[1] = (w2 & 0x0f0f0f0fu) | ((w0 >> 2) & 0x30303030u);
                m5[1] = ((w2 >> 4) & 0x0f0f0f0fu) | ((w1 >> 2) & 0x30303030u);
                hb = mg_ld(wl + li * WT::ROW + 16 + 16 * kh);
            }
            mg_v2i hm[2];
            if constexpr (T == Q3_K) {
#pragma unroll
                for (int k = 0; k < 2; k++) hm[k] = *(const mg_v2i *)(wl + 32 * WT::ROW + li * WT::HM + 16 * k + 8 * kh);
            }
            // minima as fp16 pairs against the lane's activation sums 8 kh .. + 7
            uint32_t mh[4];
            if constexpr (MINS) {
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    if constexpr (T == Q5_K) {
                        const uint32_t h = f2h((float)(((kh ? m5[1] : m5[0]) >> (8 * t)) & 0xff));
                        mh[t] = h | (h << 16);                           // sub-block 4 kh + t: two sums of 16
                    } else {
                        const uint32_t b = (uint32_t)(t < 2 ? (kh ? sc.z : sc.x) : (kh ? sc.w : sc.y)) >> (16 * (t & 1));
                        mh[t] = f2h((float)((b >> 4) & 15)) | ((uint32_t)f2h((float)((b >> 12) & 15)) << 16);
                    }
                }
            }
#pragma unroll
            for (int p = 0; p < 4; p++) {
                mg_v16i is;
                if constexpr (T == Q5_K) {
                    const mg_v4i q = mg_ld(wl + li * WT::ROW + 48 + 32 * p + 16 * kh);
                    const mg_v4i lo = (q & 0x0F0F0F0F) | (((hb >> (2 * p)) & 0x01010101) << 4);
                    const mg_v4i hi = ((q >> 4) & 0x0F0F0F0F) | (((hb >> (2 * p + 1)) & 0x01010101) << 4);
                    int sc0 = (s5[p >> 1] >> (16 * (p & 1))) & 0xff, sc1 = (s5[p >> 1] >> (16 * (p & 1) + 8)) & 0xff;
                    asm("" : "+v"(sc0), "+v"(sc1));                      // no byte select inside the multiplies
                    const mg_v16i i0 = mg_mma(a[2 * p], lo, z), i1 = mg_mma(a[2 * p + 1], hi, z);
#pragma unroll
                    for (int r = 0; r < 16; r++) is[r] = __mul24(sc1, i1[r]) + __mul24(sc0, i0[r]);
                } else {
                    const int h = p >> 1, k = p & 1;
                    const mg_v2i q = *(const mg_v2i *)(wl + li * WT::ROW + 16 * p + 8 * kh);
                    mg_v4i o[2];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int g = 8 * h + 2 * j + k;                 // 16-element group
                        int c = 0;
                        if constexpr (T == Q2_K) {
                            c = ((uint32_t)sc[g >> 2] >> (8 * (g & 3))) & 15;
                            c |= c << 16;
                        }
                        if constexpr (T == Q3_K) {
                            const uint32_t lo = ((uint32_t)((g & 7) < 4 ? sc.x : sc.y) >> (8 * (g & 3) + (g >= 8 ? 4 : 0))) & 15;
                            c = (int)(lo | ((((uint32_t)sc.z >> (8 * (g & 3) + 2 * (g >> 2))) & 3) << 4)) - 32;
                        }
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            uint32_t t = ((uint32_t)q[e] >> (2 * j)) & 0x03030303u;
                            if constexpr (T == TQ2_0) t = (t + 0x7f7f7f7fu) ^ 0x80808080u;   // per byte: t - 1
                            if constexpr (T == Q2_K) t = mg_pkmul(t, (uint32_t)c);           // bytes <= 45: no carry
                            if constexpr (T == Q3_K) {
                                // per byte 4 c - c t modulo 256, even and odd bytes apart
                                t |= (((uint32_t)hm[k][e] >> (4 * h + j)) & 0x01010101u) << 2;
                                const uint32_t nc = (uint32_t)(-c & 0xffff) * 0x10001u, c4 = (uint32_t)((4 * c) & 0xffff) * 0x10001u;
                                const uint32_t ev = mg_pkadd(mg_pkmul(t & 0x00ff00ffu, nc), c4);
                                const uint32_t od = mg_pkadd(mg_pkmul((t >> 8) & 0x00ff00ffu, nc), c4);
                                t = (ev & 0x00ff00ffu) | ((od << 8) & 0xff00ff00u);
                            }
                            o[j >> 1][2 * (j & 1) + e] = (int)t;
                        }
                    }
                    is = mg_mma(a[2 * p + 1], o[1], mg_mma(a[2 * p], o[0], z));
                }
                load_a(2 * p, sn);
                load_a(2 * p + 1, sn);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int r = 0; r < 16; r++) acc[p][r] = __builtin_fmaf(T == Q3_K ? -(da[r] * dw) : da[r] * dw, (float)is[r], acc[p][r]);
                if constexpr (MINS) {
                    // unit p's four sums of 16: q5_K 4 p .. + 3, q2_K 8 h + 2 j + k
                    uint32_t mo[4];
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const bool on = kh == (p >> 1) && (T == Q2_K || (t >> 1) == (p & 1));
                        const uint32_t keep = T == Q2_K ? (p & 1 ? 0xffff0000u : 0x0000ffffu) : 0xffffffffu;
                        mo[t] = on ? mh[t] & keep : 0u;
                    }
                    const mg_v4i mv = {(int)mo[0], (int)mo[1], (int)mo[2], (int)mo[3]};
                    const mg_v16f ms = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mg_v8h, bs), __builtin_bit_cast(mg_v8h, mv), zf, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[p][r] = __builtin_fmaf(-(da[r] * dm), ms[r], acc[p][r]);
                }
            }
            load_s(sn);
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float v = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
            tot[r] = ci ? tot[r] + v : v;
        }
    }
    __syncthreads();
    // C[i][j]: j = lane % 32 (weight row), i = 8 (r / 4) + 4 kh + r % 4 (token)
    float (*part)[32][33] = (float (*)[32][33])lds;
#pragma unroll
    for (int r = 0; r < 16; r++) part[wave][8 * (r >> 2) + 4 * kh + (r & 3)][li] = tot[r];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 32 * 32 / (64 * NW); h++) {
        const int o = threadIdx.x + 64 * NW * h, i = o >> 5, j = o & 31;
        float v = (part[0][i][j] + part[1][i][j]) + (part[2][i][j] + part[3][i][j]);
        if constexpr (NW == 8) v += (part[4][i][j] + part[5][i][j]) + (part[6][i][j] + part[7][i][j]);
        if (m0 + i < M && n0 + j < W.nrows) Y[(size_t)(m0 + i) * W.nrows + n0 + j] = v;
    }
}

// the GEMV shapes it reproduces: 16, 32 or 64 lanes per row.  From 9 tokens,
// where the GEMV takes a second launch (up to 8 it takes one, two at wide
// rows): faster at every size there, the smallest included (GEMV chunks / this,
// us, 9 tokens: q5_K 256 x 256 11.9 / 7.5, 256 x 2048 14.6 / 8.3, 256 x 11008
// 49.2 / 19.2, 1024 x 4096 15.4 / 9.9; tq2_0 256 x 256 12.3 / 8.4, 1024 x 4096
// 15.2 / 8.3)
static int mmg_classes(const g4h_tensor &W) {
    int lpr, upl;
    gemv_shape(W.type, W.nb, &lpr, &upl);
    return lpr == 16 || lpr == 32 || lpr == 64 ? lpr / 4 : 0;
}
// token tiles of one launch (all of them, but for outputs of 2^33 values and more)
static int mmg_tok(const g4h_tensor &W, int M) {
    return (int)std::min<int64_t>((M + 31) / 32, max_grid(mmg_classes(W) < 8 ? 256 : 512) / ((W.nrows + 255) / 256 * 8));
}
bool mmg_fits(const g4h_tensor &W, int M) {
    if (W.type != Q5_K && W.type != Q3_K && W.type != Q2_K && W.type != TQ2_0) return false;
    return M > 8 && mmg_classes(W) && mmg_tok(W, M) > 0;
}

template <int T>
static hipError_t mmg_go(const g4h_tensor &W, const uint8_t *ws, int M, float *Y, int nc, hipStream_t s) {
    const int nt = mmg_tok(W, M);
    for (int64_t m0 = 0; m0 < M; m0 += (int64_t)nt * 32) {              // one launch as a rule
        const int m = (int)std::min<int64_t>(M - m0, (int64_t)nt * 32), ntok = (m + 31) / 32;
        const dim3 g((unsigned)((W.nrows + 255) / 256 * 8 * ntok));
        const uint8_t *a = ws + (size_t)m0 * W.nb * 292;
        float *y = Y + (size_t)m0 * W.nrows;
        if (nc == 4) hipLaunchKernelGGL((k_mmg<T, 4>), g, dim3(256), 0, s, W, a, m, y, ntok);
        else if (nc == 8) hipLaunchKernelGGL((k_mmg<T, 8>), g, dim3(512), 0, s, W, a, m, y, ntok);
        else hipLaunchKernelGGL((k_mmg<T, 16>), g, dim3(512), 0, s, W, a, m, y, ntok);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

hipError_t launch_matmul_mfma_gx(const g4h_tensor &W, const float *x, size_t xs, int M, float *Y, uint8_t *ws, hipStream_t s) {
    if (!mmg_fits(W, M) || !x || !Y || (uintptr_t)ws % 64) return hipErrorInvalidValue;
    if (hipError_t e = launch_quantize_q8_K_tile(x, xs, ws, W.ncols, M, W.type, s)) return e;
    const int nc = mmg_classes(W);
    switch (W.type) {
    case Q5_K: return mmg_go<Q5_K>(W, ws, M, Y, nc, s);
    case Q3_K: return mmg_go<Q3_K>(W, ws, M, Y, nc, s);
    case Q2_K: return mmg_go<Q2_K>(W, ws, M, Y, nc, s);
    default: return mmg_go<TQ2_0>(W, ws, M, Y, nc, s);
    }
}

void mmg_describe(const g4h_tensor &W, int M, char *buf, size_t len) {
    const int nc = mmg_classes(W), nt = mmg_tok(W, M);
    snprintf(buf, len, "k_mmg<%s,classes=%d> grid=%lld block=%d (x%d launches; int8 MFMA in the GEMV's order, fp32 x; given rows take the GEMV chunks)",
             W.type == Q5_K ? "q5_K" : W.type == Q3_K ? "q3_K" : W.type == Q2_K ? "q2_K" : "tq2_0", nc,
             (long long)((W.nrows + 255) / 256 * 8 * nt), nc < 8 ? 256 : 512, ((M + 31) / 32 + nt - 1) / nt);
}

}  // namespace g4
