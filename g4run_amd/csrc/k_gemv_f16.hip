// k_gemv_f16.hip -- GEMV over f16 / bf16 weight rows (matmul_b's G4_F16 and
// G4_BF16 cases, model.c:238-239, over g4_dot_f16 / g4_dot_bf16,
// quants.c:1319-1347) and the activation conversions of prep_act's AC_F16 /
// AC_BF16 classes (model.c:163-180).
//
// Floating-point weights carry no block scales and no integer sums: each lane
// widens 8 weights (one 16-byte load) and 8 activations to fp32 and fma's them
// into one accumulator per token, lanes stride the row, and the wave sums its
// lanes.  The fp32 order differs from the CPU's 8-lane AVX2 order (within the
// path's fp32 tolerance) but does not depend on the token count, so a batch
// gives every token the single-token bits.
#include <cstdio>

#include "common.h"
#include "kernels.h"

namespace g4 {

// g4_fp32_to_bf16 (g4run.h:64-68): a NaN keeps its high half with the quiet
// bit set; everything else rounds to nearest even by the header's add-and-shift.
__device__ __forceinline__ uint16_t f2bf(float f) {
    const uint32_t x = __float_as_uint(f);
    if ((x & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x >> 16) | 64u);
    return (uint16_t)((x + (0x7fffu + ((x >> 16) & 1u))) >> 16);
}

// x fp32 [nb][ncols] (row stride xs floats) -> f16 rows (AC_F16) or bf16-rounded
// fp32 rows (AC_BF16) at `os` bytes per token
__global__ __launch_bounds__(256) void k_act_float(int wtype, const float *__restrict__ x, size_t xs, int64_t ncols,
                                                   uint8_t *__restrict__ out, size_t os) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int b = blockIdx.y;
    if (i >= ncols) return;
    const float v = x[(size_t)b * xs + i];
    if (wtype == F16) ((uint16_t *)(out + (size_t)b * os))[i] = f2h(v);
    else ((float *)(out + (size_t)b * os))[i] = __uint_as_float((uint32_t)f2bf(v) << 16);
}

template <int WT>
__device__ __forceinline__ void widen8(const uint4 w, float (&f)[8]) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if constexpr (WT == F16) {
            f[2 * k] = h2f((uint16_t)(u[k] & 0xffff));
            f[2 * k + 1] = h2f((uint16_t)(u[k] >> 16));
        } else {                                            // bf16 -> fp32: the high half of a word
            f[2 * k] = __uint_as_float(u[k] << 16);
            f[2 * k + 1] = __uint_as_float(u[k] & 0xffff0000u);
        }
    }
}

// One wave per row.  W rows at `ws` bytes, activations of NB tokens at `as`
// bytes (f16 for F16 weights, fp32 for BF16), 16-byte aligned, ncols % 8 == 0.
// XF: `act` holds the tokens as fp32 rows instead, converted on load with
// k_act_float's arithmetic (f16 round-to-nearest-even, or bf16 rounding), so
// the sums are those of converting first -- one launch instead of two.
template <int WT, int NB, bool XF, bool OUT>
__global__ __launch_bounds__(256) void k_gemv_float(const uint8_t *__restrict__ W, size_t ws, int64_t nrows, int64_t ncols,
                                                    const uint8_t *__restrict__ act, size_t as, float *__restrict__ Y,
                                                    size_t ys, GemvOut out) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= nrows) return;                                       // wave-uniform
    const uint8_t *wr = W + (size_t)row * ws;
    const int64_t ng = ncols / 8;
    float acc[NB];
#pragma unroll
    for (int t = 0; t < NB; t++) acc[t] = 0.0f;
#pragma unroll 4
    for (int64_t g = lane; g < ng; g += 64) {
        float wf[8];
        widen8<WT>(*(const uint4 *)(wr + 16 * g), wf);
#pragma unroll
        for (int t = 0; t < NB; t++) {
            float af[8];
            if constexpr (XF) {
                const float4 a0 = *(const float4 *)(act + (size_t)t * as + 32 * g);
                const float4 a1 = *(const float4 *)(act + (size_t)t * as + 32 * g + 16);
                const float xr[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
                for (int e = 0; e < 8; e++)
                    af[e] = WT == F16 ? h2f(f2h(xr[e])) : __uint_as_float((uint32_t)f2bf(xr[e]) << 16);
            } else if constexpr (WT == F16) {
                widen8<F16>(*(const uint4 *)(act + (size_t)t * as + 16 * g), af);
            } else {
                const float4 a0 = *(const float4 *)(act + (size_t)t * as + 32 * g);
                const float4 a1 = *(const float4 *)(act + (size_t)t * as + 32 * g + 16);
                af[0] = a0.x; af[1] = a0.y; af[2] = a0.z; af[3] = a0.w;
                af[4] = a1.x; af[5] = a1.y; af[6] = a1.z; af[7] = a1.w;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) acc[t] = __builtin_fmaf(wf[e], af[e], acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const float s = group_sum<64>(acc[t]);
        if (lane == 0) Y[(size_t)t * ys + row] = OUT ? gemv_out_value(out, row, s) : s;
    }
}

template <int WT, bool XF>
static hipError_t gf_go(const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const uint8_t *act, size_t as, float *Y,
                        size_t ys, int nb, hipStream_t s, const GemvOut &out) {
    if (out.mode != OUT_STORE && nb != 1) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((nrows + 3) / 4));
    if (out.mode != OUT_STORE) {
        hipLaunchKernelGGL((k_gemv_float<WT, 1, XF, true>), grid, dim3(256), 0, s, W, ws, nrows, ncols, act, as, Y, ys, out);
        return hipGetLastError();
    }
    switch (nb) {
    case 1: hipLaunchKernelGGL((k_gemv_float<WT, 1, XF, false>), grid, dim3(256), 0, s, W, ws, nrows, ncols, act, as, Y, ys, out); break;
    case 2: hipLaunchKernelGGL((k_gemv_float<WT, 2, XF, false>), grid, dim3(256), 0, s, W, ws, nrows, ncols, act, as, Y, ys, out); break;
    case 4: hipLaunchKernelGGL((k_gemv_float<WT, 4, XF, false>), grid, dim3(256), 0, s, W, ws, nrows, ncols, act, as, Y, ys, out); break;
    case 8: hipLaunchKernelGGL((k_gemv_float<WT, 8, XF, false>), grid, dim3(256), 0, s, W, ws, nrows, ncols, act, as, Y, ys, out); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_gemv_float(int wtype, const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const uint8_t *act, size_t as,
                             float *Y, size_t ys, int nb, hipStream_t s, const GemvOut &out) {
    if (ncols % 8 || ws % 16 || as % 16 || (uintptr_t)W % 16 || (uintptr_t)act % 16) return hipErrorInvalidValue;
    return wtype == F16 ? gf_go<F16, false>(W, ws, nrows, ncols, act, as, Y, ys, nb, s, out)
         : wtype == BF16 ? gf_go<BF16, false>(W, ws, nrows, ncols, act, as, Y, ys, nb, s, out)
                         : hipErrorInvalidValue;
}

// the same from fp32 tokens x (row stride xs floats), converted on load
hipError_t launch_gemv_float_x(int wtype, const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const float *x, size_t xs,
                               float *Y, size_t ys, int nb, hipStream_t s, const GemvOut &out) {
    if (ncols % 8 || ws % 16 || xs % 4 || (uintptr_t)W % 16 || (uintptr_t)x % 16) return hipErrorInvalidValue;
    const uint8_t *a = (const uint8_t *)x;
    return wtype == F16 ? gf_go<F16, true>(W, ws, nrows, ncols, a, xs * 4, Y, ys, nb, s, out)
         : wtype == BF16 ? gf_go<BF16, true>(W, ws, nrows, ncols, a, xs * 4, Y, ys, nb, s, out)
                         : hipErrorInvalidValue;
}

// Prompt batches on the matrix cores (g4h_matmul path 2): Y[t][r] = sum_k
// W[r][k] a[t][k], one v_mfma_f32_16x16x32_f16 / _bf16 per 32 columns of a
// 16-token x 16-row tile.  The operands are the GEMV family's: f16 weights
// against f16-rounded activations, bf16 weights against bf16-rounded ones
// (prep_act's AC_F16 / AC_BF16, model.c:163-180), so every product is exact
// in fp32 (11 x 11 or 8 x 8 significant bits) and only the fp32 order of the
// sums differs from the CPU's and from the GEMV family's (within the path's
// tolerance).  A workgroup owns MT x NT such tiles; its MMF_W waves split the
// 64-column chunks (wave w takes chunks w, w + MMF_W, ..., each chained into
// its accumulators in increasing order, a last partial chunk included) and
// the waves' tiles are added in wave order through LDS: a token's result
// depends neither on the batch size nor on MT and NT.
//
// What bounds it: the CU's L1 serves one 64-byte access per clock, and lanes
// reading different rows are one access each.  An MFMA operand has adjacent
// lanes in different rows, so loading it straight from memory costs 57
// accesses per 1 KB instruction (measured).  Here adjacent lanes load adjacent
// 16 bytes of one row, fp32 activations are rounded on the way, and each wave
// turns its own chunk into operands through LDS of its own (no barrier), the
// next chunk's loads in flight meanwhile.  LDS rows of 128 bytes, the 16-byte
// columns of row r at column ^ (r & 7).  Measured against operands loaded
// straight from memory for 32 x 32 tiles (fp32 tokens, us): f16 4096 x 4096 at
// 64 / 201 / 512 tokens 29.4 / 83.0 / 177.9 -> 15.9 / 23.9 / 46.7 (141, 282 and
// 368 TFLOP/s), f16 256 x 2048 at 64 tokens 13.4 -> 5.6, bf16 2560 x 10240 at
// 64 / 300 tokens 74.8 / 212.8 -> 33.6 / 51.5.
// Operand layout: lane l holds A[l % 16][8 (l / 16) .. + 7] and
// B[l % 16][8 (l / 16) .. + 7]; C[i][j] with j = l % 16 (weight row), i = 4
// (l / 16) + r (token).
typedef _Float16 mf_v8h __attribute__((ext_vector_type(8)));
typedef __bf16 mf_v8bf __attribute__((ext_vector_type(8)));
typedef float mf_v4f __attribute__((ext_vector_type(4)));

constexpr int MMF_W = 8;              // waves per workgroup

// two fp32 activations rounded with k_act_float's arithmetic by the packed
// conversion instructions (round to nearest even; bf16-rounded rows keep their
// values)
template <int WT>
__device__ __forceinline__ uint32_t mmf_round2(uint32_t x, uint32_t y) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    const v2f v = {__uint_as_float(x), __uint_as_float(y)};
    if constexpr (WT == F16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2h));
    else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2bf));
}

// A32: activation rows of fp32 (row stride `as` bytes), rounded on the way to
// LDS; else f16 rows.  Workgroup b runs on XCD b % 8: the token tiles of one
// row tile go to one XCD, consecutively, and find its weights in that XCD's L2.
template <int WT, bool A32, int MT, int NT>
__global__ __launch_bounds__(64 * MMF_W) void k_mm_float(const uint8_t *__restrict__ W, size_t ws, int64_t nrows, int64_t ncols,
                                                         const uint8_t *__restrict__ act, size_t as, int M, float *__restrict__ Y,
                                                         int ntok) {
    constexpr int AL = A32 ? 4 * MT : 2 * MT, WL = 2 * NT;          // 16-byte loads per lane and chunk
    // chunks per stage: 40 to 96 registers of loads, at most 16 KB of LDS per wave
    constexpr int CR = AL + WL >= 12 ? 1 : AL + WL >= 8 ? 2 : 4, CH = CR * (MT + NT) <= 8 ? CR : CR / 2;
    constexpr int LW = CH * (MT + NT) * 2048;                       // LDS bytes per wave
    constexpr int PW = MT * NT * 1024;                              // partial tiles per wave
    __shared__ __align__(16) uint8_t lds[MMF_W * (LW > PW ? LW : PW)];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
    const int li = lane & 15, kg = lane >> 4;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int64_t n0 = ((int64_t)(l / ntok) * 8 + x) * (16 * NT);
    const int m0 = (l % ntok) * (16 * MT);
    if (n0 >= nrows) return;                                        // uniform over the workgroup
    uint8_t *sl = lds + wave * LW;
    // 16-byte loads: eight lanes per 128-byte row of W (and of f16
    // activations), sixteen per 256-byte fp32 row
    const int wr = lane >> 3, wc = lane & 7, ar = A32 ? lane >> 4 : wr, ac = A32 ? lane & 15 : wc;
    constexpr int AQ = A32 ? 4 : 8;                                 // activation rows per load
    const uint8_t *wp[WL], *ap[AL];
#pragma unroll
    for (int q = 0; q < WL; q++) wp[q] = W + (size_t)min(n0 + 8 * q + wr, nrows - 1) * ws + 16 * wc;
#pragma unroll
    for (int q = 0; q < AL; q++) ap[q] = act + (size_t)min(m0 + AQ * q + ar, M - 1) * as + 16 * ac;
    const int nc = (int)(ncols >> 6);                               // whole chunks
    const int nj = (nc - wave + MMF_W - 1) / MMF_W;                 // this wave's (uniform)
    struct Stage {
        uint4 w[CH][WL], a[CH][AL];
    };
    Stage S;
    auto load = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const size_t k = (size_t)(wave + MMF_W * min(j0 + c, nj - 1));
#pragma unroll
            for (int q = 0; q < WL; q++) S.w[c][q] = *(const uint4 *)(wp[q] + 128 * k);
#pragma unroll
            for (int q = 0; q < AL; q++) S.a[c][q] = *(const uint4 *)(ap[q] + (A32 ? 256 : 128) * k);
        }
    };
    auto put = [&](int c) __attribute__((always_inline)) {          // chunk c of the stage into LDS
        uint8_t *la = sl + c * (MT + NT) * 2048, *lw = la + MT * 2048;
#pragma unroll
        for (int q = 0; q < WL; q++) *(uint4 *)(lw + (8 * q + wr) * 128 + 16 * (wc ^ wr)) = S.w[c][q];
#pragma unroll
        for (int q = 0; q < AL; q++) {
            const uint4 v = S.a[c][q];
            const int r = AQ * q + ar;
            if constexpr (A32)
                *(uint2 *)(la + r * 128 + 16 * ((ac >> 1) ^ (r & 7)) + 8 * (ac & 1)) =
                    make_uint2(mmf_round2<WT>(v.x, v.y), mmf_round2<WT>(v.z, v.w));
            else
                *(uint4 *)(la + r * 128 + 16 * (ac ^ (r & 7))) = v;
        }
    };
    mf_v4f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[m][n] = mf_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto mul = [&](int c) __attribute__((always_inline)) {
        const uint8_t *la = sl + c * (MT + NT) * 2048 + li * 128, *lw = la + MT * 2048;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int o = 16 * ((4 * h + kg) ^ (li & 7));
            uint4 a[MT], w[NT];
#pragma unroll
            for (int m = 0; m < MT; m++) a[m] = *(const uint4 *)(la + 2048 * m + o);
#pragma unroll
            for (int n = 0; n < NT; n++) w[n] = *(const uint4 *)(lw + 2048 * n + o);
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if constexpr (WT == F16)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mf_v8h, a[m]), __builtin_bit_cast(mf_v8h, w[n]),
                                                                           acc[m][n], 0, 0, 0);
                    else
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_v8bf, a[m]),
                                                                            __builtin_bit_cast(mf_v8bf, w[n]), acc[m][n], 0, 0, 0);
                }
        }
    };
    // a wave's LDS accesses complete in order; the empty asms keep the
    // compiler from moving any access across a hand-over
    if (nj > 0) {
        load(0);
        for (int j0 = 0; j0 < nj; j0 += CH) {
            const int left = nj - j0;                               // uniform
#pragma unroll
            for (int c = 0; c < CH; c++) put(c);
            asm volatile("" ::: "memory");
            load(j0 + CH);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int c = 0; c < CH; c++)
                if (c < left) mul(c);
            asm volatile("" ::: "memory");
        }
    }
    // a last chunk of ncols % 64 columns, zeros past them
    if ((ncols & 63) && wave == nc % MMF_W) {                       // uniform
        const int lw = (int)(ncols & 63) / 8, la = A32 ? 2 * lw : lw;   // 16-byte columns
        const size_t k = nc;
        const uint4 z = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < WL; q++) {
            S.w[0][q] = *(const uint4 *)(wp[q] + 128 * k - 16 * (wc < lw ? 0 : wc));   // past them the chunk's first column
            if (wc >= lw) S.w[0][q] = z;
        }
#pragma unroll
        for (int q = 0; q < AL; q++) {
            S.a[0][q] = *(const uint4 *)(ap[q] + (A32 ? 256 : 128) * k - 16 * (ac < la ? 0 : ac));
            if (ac >= la) S.a[0][q] = z;
        }
        put(0);
        asm volatile("" ::: "memory");
        mul(0);
    }
    __syncthreads();
    float *part = (float *)lds;                                     // [wave][register][lane]
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) part[(wave * MT * NT * 4 + (m * NT + n) * 4 + r) * 64 + lane] = acc[m][n][r];
    __syncthreads();
    // the waves' tiles in wave order; wave w stores registers w, w + 8, ..
    for (int u = wave; u < MT * NT * 4; u += MMF_W) {
        float o = part[u * 64 + lane];
#pragma unroll
        for (int w = 1; w < MMF_W; w++) o += part[(w * MT * NT * 4 + u) * 64 + lane];
        const int m = m0 + 16 * (u / (4 * NT)) + 4 * kg + (u & 3);
        const int64_t n = n0 + 16 * ((u >> 2) % NT) + li;
        if (m < M && n < nrows) Y[(size_t)m * nrows + n] = o;
    }
}

// Tiles of a call: the shape with the least L1 traffic per CU, rounds of
// workgroups x the bytes a workgroup loads per column (fp32 activation rows 4,
// f16 rows and weights 2 each).  Measured with fp32 activations (us): f16 4096
// x 4096 at 64 tokens 2 x 2 15.9, 4 x 1 21.0, 2 x 4 20.2; at 128 tokens 2 x 4
// 19.0, 4 x 2 22.9; at 201 tokens 4 x 4 25.1, 2 x 4 32.0, 4 x 2 36.2.
static void mmf_tiles(bool a32, int64_t nrows, int M, int &mt, int &nt, int &ntok, int64_t &grid) {
    const int tm = (M + 15) / 16;
    const int64_t tn = (nrows + 15) / 16;
    int64_t best = INT64_MAX;
    for (int m = tm > 2 ? 4 : tm; m >= 1; m >>= 1)
        for (int n = 4; n >= 1; n >>= 1) {
            const int64_t cost = ((tm + m - 1) / m * ((tn + n - 1) / n) + 255) / 256 * ((a32 ? 2 : 1) * m + n);
            if (cost < best) best = cost, mt = m, nt = n;
        }
    ntok = (tm + mt - 1) / mt;
    grid = ((tn + nt - 1) / nt + 7) / 8 * 8 * ntok;
}

void mmf_describe(int wtype, int64_t nrows, int M, char *buf, size_t len) {
    int mt, nt, ntok;
    int64_t grid;
    mmf_tiles(true, nrows, M, mt, nt, ntok, grid);
    snprintf(buf, len, "k_mm_float<%s,mt=%d,nt=%d> grid=%lld block=%d (matrix cores, 16x16 tiles, %d waves split the columns)",
             wtype == F16 ? "f16" : "bf16", mt, nt, (long long)grid, 64 * MMF_W, MMF_W);
}

template <int WT, bool A32>
static hipError_t mmf_go(const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const uint8_t *a, size_t ab, int M, float *Y,
                         hipStream_t s) {
    int mt, nt, ntok;
    int64_t grid;
    mmf_tiles(A32, nrows, M, mt, nt, ntok, grid);
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
#define G4_MMF(MT_, NT_)                                                                                                       \
    if (mt == MT_ && nt == NT_) {                                                                                              \
        hipLaunchKernelGGL((k_mm_float<WT, A32, MT_, NT_>), dim3((unsigned)grid), dim3(64 * MMF_W), 0, s, W, ws, nrows, ncols, a, ab, \
                           M, Y, ntok);                                                                                        \
        return hipGetLastError();                                                                                              \
    }
    G4_MMF(1, 1) G4_MMF(1, 2) G4_MMF(1, 4) G4_MMF(2, 1) G4_MMF(2, 2) G4_MMF(2, 4) G4_MMF(4, 1) G4_MMF(4, 2) G4_MMF(4, 4)
#undef G4_MMF
    return hipErrorInvalidValue;
}

// M tokens of f16 / bf16 weight rows (ws bytes apart, ncols % 16 == 0) on the
// matrix cores: x fp32 rows (xs floats apart) or prepared activation rows at
// `as` bytes (exactly one of x, act)
hipError_t launch_mm_float(int wtype, const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const float *x, size_t xs,
                           const uint8_t *act, size_t as, int M, float *Y, hipStream_t s) {
    if ((wtype != F16 && wtype != BF16) || ncols % 16 || ws % 16 || (uintptr_t)W % 16 || M < 1 || (x == nullptr) == (act == nullptr))
        return hipErrorInvalidValue;
    if (x ? ((uintptr_t)x % 16 || xs % 4) : ((uintptr_t)act % 16 || as % 16)) return hipErrorInvalidValue;
    const uint8_t *a = x ? (const uint8_t *)x : act;
    const size_t ab = x ? xs * 4 : as;
    // prepared bf16 rows are bf16-rounded fp32: rounding them again keeps them
    if (wtype == BF16) return mmf_go<BF16, true>(W, ws, nrows, ncols, a, ab, M, Y, s);
    return x ? mmf_go<F16, true>(W, ws, nrows, ncols, a, ab, M, Y, s) : mmf_go<F16, false>(W, ws, nrows, ncols, a, ab, M, Y, s);
}

hipError_t launch_act_float(int wtype, const float *x, size_t xs, int64_t ncols, int nb, uint8_t *out, size_t os, hipStream_t s) {
    hipLaunchKernelGGL(k_act_float, dim3((unsigned)((ncols + 255) / 256), (unsigned)nb), dim3(256), 0, s, wtype, x, xs, ncols, out, os);
    return hipGetLastError();
}

}  // namespace g4
