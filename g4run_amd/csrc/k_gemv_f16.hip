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
#include <algorithm>
#include <cstdio>
#include <type_traits>

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
// W[r][k] a[t][k], one v_mfma_f32_32x32x16_f16 / _bf16 per 16 columns of a
// 32-token x 32-row tile.  The operands are the GEMV family's: f16 weights
// against f16-rounded activations, bf16 weights against bf16-rounded ones
// (prep_act's AC_F16 / AC_BF16, model.c:163-180), so every product is exact
// in fp32 (11 x 11 or 8 x 8 significant bits) and only the fp32 order of the
// sums differs from the CPU's and from the GEMV family's (within the path's
// tolerance).  A workgroup owns MR tokens x NR rows; its MMF_W waves split the
// 16-column steps (wave w takes steps w, w + MMF_W, ..., each chained into its
// accumulators in increasing order) and the waves' tiles are added in wave
// order through LDS: a token's result depends neither on the batch size nor on
// MR and NR (a tile of 16 repeats its rows in the MFMA's other half).
//
// What bounds it: the CU's L1 serves one 64-byte access per clock, and lanes
// reading different rows are one access each.  An MFMA operand has adjacent
// lanes in different rows, so loading it straight from memory costs 57
// accesses per 1 KB instruction (measured).  Here the workgroup loads chunks
// of 256 columns, adjacent lanes adjacent 16 bytes of a row, rounds fp32
// activations on the way into LDS and reads the operands there, the next
// chunk's loads in flight meanwhile.  LDS rows of 512 bytes, the 16-byte
// columns of row r at column ^ (r & 7).  Measured against operands loaded
// straight from memory for 32 x 32 tiles, the same bits (fp32 tokens, us): f16
// 4096 x 4096 at 9 / 64 / 201 / 512 tokens 19.5 / 29.4 / 83.0 / 177.9 -> 10.9 /
// 16.8 / 25.7 / 55.5 (310 TFLOP/s), f16 256 x 2048 at 64 13.4 -> 5.4, bf16 2560 x
// 10240 at 64 / 300 tokens 74.8 / 212.8 -> 33.6 / 60.2.  Each wave turning its
// own 64-column chunks into operands without a barrier was faster at 512
// tokens (46.7 us), but its other order of the sums moves every 16-bit
// projection of a model by a last bit.
// Operand layout: lane l holds A[l % 32][8 (l / 32) .. + 7] and
// B[l % 32][8 (l / 32) .. + 7]; C[i][j] with j = l % 32 (weight row), i = 8
// (r / 4) + 4 (l / 32) + r % 4 (token).
typedef _Float16 mf_v8h __attribute__((ext_vector_type(8)));
typedef __bf16 mf_v8bf __attribute__((ext_vector_type(8)));
typedef float mf_v16f __attribute__((ext_vector_type(16)));
typedef uint32_t mf_v4u __attribute__((ext_vector_type(4)));

constexpr int MMF_W = 8;              // waves per workgroup
constexpr int MMF_KC = 256;           // columns per chunk: two steps per wave
// rows of many chunks, of one, and past 32-bit byte offsets (16 x 16 tiles only)
enum { MMF_LOOP, MMF_ONE, MMF_LONG };
static bool mmf_long(int64_t ncols) { return ncols >= (int64_t)1 << 29; }

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

// FORM MMF_ONE: rows of one chunk (up to 256 columns), which is loaded once and takes
// one buffer; the loop's loads ahead would all be of the last piece again (us, loop /
// this, the same tiles: f16 65536 x 256 at 9 / 17 / 80 tokens 14.5 / 16.4 / 40.3 ->
// 8.1 / 10.3 / 37.3).
// A32: activation rows of fp32 (row stride `as` bytes), rounded on the way to
// LDS; else f16 rows.  Workgroup b runs on XCD b % 8: the token tiles of one
// row tile go to one XCD, consecutively, and find its weights in that XCD's L2.
template <int WT, bool A32, int FORM, int MR, int NR>
__global__ __launch_bounds__(64 * MMF_W) void k_mm_float(const uint8_t *__restrict__ W, size_t ws, int64_t nrows, int64_t ncols,
                                                         const uint8_t *__restrict__ act, size_t as, int M, float *__restrict__ Y,
                                                         int ntok) {
    constexpr int MT = (MR + 31) / 32, NT = (NR + 31) / 32, NTH = 64 * MMF_W, RB = 2 * MMF_KC;
    constexpr int AU = A32 ? 64 : 32, AL = MR * AU / NTH, WL = NR * 32 / NTH;   // 16-byte pieces per row, loads per thread
    static_assert(MR * AU % NTH == 0 && NR * 32 % NTH == 0, "whole loads");
    constexpr int BUF = (MR + NR) * RB, PART = MMF_W * MT * NT * 4096;
    constexpr bool ONE = FORM == MMF_ONE;
    constexpr int STAGED = ONE ? BUF : 2 * BUF;
    __shared__ __align__(16) uint8_t lds[STAGED > PART ? STAGED : PART];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t) >> 6;
    const int li = lane & 31, kh = lane >> 5;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int64_t n0 = ((int64_t)(l / ntok) * 8 + x) * NR;
    const int m0 = (l % ntok) * MR;
    if (n0 >= nrows) return;                                        // uniform over the workgroup
    const int wr = t >> 5, wc = t & 31, ar = A32 ? t >> 6 : wr, ac = A32 ? t & 63 : wc;
    constexpr int WQ = NTH / 32, AQ = NTH / AU;                     // rows per load of the workgroup
    const uint8_t *wp[WL], *ap[AL];
#pragma unroll
    for (int q = 0; q < WL; q++) wp[q] = W + (size_t)min(n0 + WQ * q + wr, nrows - 1) * ws;
#pragma unroll
    for (int q = 0; q < AL; q++) ap[q] = act + (size_t)min(m0 + AQ * q + ar, M - 1) * as;
    const int ns = (int)(ncols >> 4), nc = (ns + 15) >> 4;          // steps, chunks
    using Off = std::conditional_t<FORM == MMF_LONG, uint64_t, uint32_t>;
    const Off wlast = (Off)ncols * 2 - 16, alast = (Off)ncols * (A32 ? 4 : 2) - 16;
    struct Stage {
        mf_v4u w[WL], a[AL];
    };
    // stages of loads in flight, 48 to 96 registers (64 x 64 workgroups were
    // slower with two: f16 4096 x 4096 at 512 tokens 55.6 / 58.7 us)
    constexpr int D = ONE || AL + WL >= 12 ? 1 : AL + WL >= 8 ? 2 : 4;
    Stage st[D];
    auto load = [&](Stage &S, int c) __attribute__((always_inline)) {   // past the row's end its last piece again, never used
        const Off wo = std::min((Off)c * RB + 16 * wc, wlast), ao = std::min((Off)c * (A32 ? 2 * RB : RB) + 16 * ac, alast);
#pragma unroll
        for (int q = 0; q < WL; q++) S.w[q] = *(const mf_v4u *)(wp[q] + wo);
#pragma unroll
        for (int q = 0; q < AL; q++) S.a[q] = *(const mf_v4u *)(ap[q] + ao);
        // the loads go out here: left alone the compiler sinks them to their
        // use behind the multiplies
        asm volatile("" ::: "memory");
    };
    auto put = [&](const Stage &S, int b) __attribute__((always_inline)) {
        uint8_t *la = lds + b * BUF, *lw = la + MR * RB;
#pragma unroll
        for (int q = 0; q < WL; q++) {
            const int r = WQ * q + wr;
            *(mf_v4u *)(lw + r * RB + 16 * (wc ^ (r & 7))) = S.w[q];
        }
#pragma unroll
        for (int q = 0; q < AL; q++) {
            const mf_v4u v = S.a[q];
            const int r = AQ * q + ar;
            if constexpr (A32)
                *(uint2 *)(la + r * RB + 16 * ((ac >> 1) ^ (r & 7)) + 8 * (ac & 1)) =
                    make_uint2(mmf_round2<WT>(v.x, v.y), mmf_round2<WT>(v.z, v.w));
            else
                *(mf_v4u *)(la + r * RB + 16 * (ac ^ (r & 7))) = v;
        }
    };
    mf_v16f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[m][n] = mf_v16f{};
    auto mul = [&](int b, int c) __attribute__((always_inline)) {
        const uint8_t *la = lds + b * BUF, *lw = la + MR * RB;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int q = wave + MMF_W * h;                         // the chunk's step (uniform)
            mf_v4u a[MT], w[NT];
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const int r = MR < 32 ? li & (MR - 1) : 32 * m + li;
                a[m] = *(const mf_v4u *)(la + r * RB + 16 * ((2 * q + kh) ^ (r & 7)));
            }
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const int r = NR < 32 ? li & (NR - 1) : 32 * n + li;
                w[n] = *(const mf_v4u *)(lw + r * RB + 16 * ((2 * q + kh) ^ (r & 7)));
            }
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if (16 * c + q >= ns) break;                   // uniform
                    if constexpr (WT == F16)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mf_v8h, a[m]), __builtin_bit_cast(mf_v8h, w[n]),
                                                                           acc[m][n], 0, 0, 0);
                    else
                        acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mf_v8bf, a[m]),
                                                                            __builtin_bit_cast(mf_v8bf, w[n]), acc[m][n], 0, 0, 0);
                }
        }
    };
    // chunk c: its stage into one LDS buffer, the stage reloaded D chunks on,
    // one barrier, the multiplies; the other buffer's readers have passed the
    // barrier before it.  Every load is issued on every pass, so the memory
    // counter waits before a store cover only the stage stored.
#pragma unroll
    for (int d = 0; d < D; d++) load(st[d], d);
    if constexpr (ONE) {
        put(st[0], 0);
        lds_barrier();
        mul(0, 0);
    } else {
        for (int c0 = 0; c0 < nc; c0 += D) {                        // uniform
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (c0 + d >= nc) break;
                put(st[d], (c0 + d) & 1);
                load(st[d], c0 + d + D);
                lds_barrier();
                mul((c0 + d) & 1, c0 + d);
            }
        }
    }
    __syncthreads();
    float *part = (float *)lds;                                     // [wave][tile register][lane]
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int r = 0; r < 16; r++) part[((wave * MT * NT + m * NT + n) * 16 + r) * 64 + lane] = acc[m][n][r];
    __syncthreads();
    // the waves' tiles in wave order; wave w stores tile registers w, w + 8, ..
    for (int u = wave; u < MT * NT * 16; u += MMF_W) {
        float o = part[u * 64 + lane];
#pragma unroll
        for (int w = 1; w < MMF_W; w++) o += part[(w * MT * NT * 16 + u) * 64 + lane];
        const int r = u & 15, i = 32 * (u / (16 * NT)) + 8 * (r >> 2) + 4 * kh + (r & 3), j = 32 * ((u >> 4) % NT) + li;
        if (i < MR && j < NR && m0 + i < M && n0 + j < nrows) Y[(size_t)(m0 + i) * nrows + n0 + j] = o;
    }
}

// Tokens and rows per workgroup: the shape with the least L1 traffic per CU,
// rounds of workgroups x the bytes a workgroup loads per column (fp32
// activation rows 4, f16 rows and weights 2 each).  Measured with fp32
// activations (us): f16 4096 x 4096 at 64 tokens 32 x 32 16.1, 64 x 32 21.3, 64 x 64
// 25.3; at 200 tokens 64 x 64 26.4, 64 x 32 38.5; 10240 x 4096 at 9 tokens 16 x 64
// 18.3, 16 x 32 23.7.  Past one 16 x 64 workgroup per CU, 16 x 32 keeps more loads in
// flight instead: 20480 x 1040 at 9 tokens 16.1 / 12.3, 65536 x 1040 37.3 / 29.6.
// Rows of one chunk wait for one round trip and the sums' LDS pass, so small
// workgroups, many per CU, are best: at most 32 x 32 (f16 20480 x 256 at 48 tokens
// 64 x 64 10.0, 32 x 32 7.0; 65536 x 256 at 80 37.4 / 19.7).
// Shapes that this never finds best are not built (fp32: fewer rows than tokens;
// one chunk: past 32 x 32).
static void mmf_tiles(bool a32, int64_t nrows, int64_t ncols, int M, int &mr, int &nr, int &ntok, int64_t &grid) {
    const int most = mmf_long(ncols) ? 16 : ncols <= MMF_KC ? 32 : 64;
    int64_t best = INT64_MAX;
    for (int m = std::min(most, M > 32 ? 64 : M > 16 ? 32 : 16); m >= 16; m >>= 1)
        for (int n = most; n >= (a32 ? m : std::max(16, m / 2)); n >>= 1) {
            if (m == 16 && n == 64 && nrows > 256 * 64) continue;   // 16 x 32 above
            const int64_t cost = ((M + m - 1) / m * ((nrows + n - 1) / n) + 255) / 256 * ((a32 ? 2 : 1) * m + n);
            if (cost < best) best = cost, mr = m, nr = n;
        }
    ntok = (M + mr - 1) / mr;
    grid = ((nrows + nr - 1) / nr + 7) / 8 * 8 * ntok;
}
// token tiles of one launch (all of them, but for outputs of 2^33 values and more)
static int mmf_tok(int64_t grid, int ntok) { return (int)std::min<int64_t>(ntok, max_grid(64 * MMF_W) / (grid / ntok)); }

void mmf_describe(int wtype, int64_t nrows, int64_t ncols, int M, char *buf, size_t len) {
    int mr, nr, ntok, pm, pn;
    int64_t grid, pgrid;
    mmf_tiles(wtype != F16, nrows, ncols, M, pm, pn, ntok, pgrid);
    mmf_tiles(true, nrows, ncols, M, mr, nr, ntok, grid);
    const int nt = mmf_tok(grid, ntok);
    snprintf(buf, len, "k_mm_float<%s,%dx%d> grid=%lld block=%d (x%d launches; matrix cores, %d waves split the columns; given rows %dx%d)",
             wtype == F16 ? "f16" : "bf16", mr, nr, (long long)(grid / ntok * nt), 64 * MMF_W, nt ? (ntok + nt - 1) / nt : 0, MMF_W, pm, pn);
}

template <int WT, bool A32, int MR, int NR>
static void mmf_run(dim3 g, const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const uint8_t *a, size_t ab, int M, float *Y, int ntok,
                    hipStream_t s) {
    if (ncols <= MMF_KC) {
        if constexpr (MR <= 32 && NR <= 32)
            hipLaunchKernelGGL((k_mm_float<WT, A32, MMF_ONE, MR, NR>), g, dim3(64 * MMF_W), 0, s, W, ws, nrows, ncols, a, ab, M, Y, ntok);
    } else if (mmf_long(ncols)) {
        if constexpr (MR == 16 && NR == 16)
            hipLaunchKernelGGL((k_mm_float<WT, A32, MMF_LONG, MR, NR>), g, dim3(64 * MMF_W), 0, s, W, ws, nrows, ncols, a, ab, M, Y, ntok);
    } else hipLaunchKernelGGL((k_mm_float<WT, A32, MMF_LOOP, MR, NR>), g, dim3(64 * MMF_W), 0, s, W, ws, nrows, ncols, a, ab, M, Y, ntok);
}

template <int WT, bool A32>
static hipError_t mmf_go(const uint8_t *W, size_t ws, int64_t nrows, int64_t ncols, const uint8_t *a, size_t ab, int M, float *Y,
                         hipStream_t s) {
    int mr, nr, ntok;
    int64_t grid;
    mmf_tiles(A32, nrows, ncols, M, mr, nr, ntok, grid);
    const int nt = mmf_tok(grid, ntok);
    if (nt < 1) return hipErrorInvalidValue;
    for (int64_t m0 = 0; m0 < M; m0 += (int64_t)nt * mr) {          // one launch as a rule
        const int m = (int)std::min<int64_t>(M - m0, (int64_t)nt * mr), n = (m + mr - 1) / mr;
        const dim3 g((unsigned)(grid / ntok * n));
        bool run = false;
#define G4_MMF(MR_, NR_)                                                                                          \
        if constexpr (!A32 || NR_ >= MR_)                                                                         \
            if (mr == MR_ && nr == NR_) mmf_run<WT, A32, MR_, NR_>(g, W, ws, nrows, ncols, a + m0 * ab, ab, m, Y + m0 * nrows, n, s), run = true;
        G4_MMF(16, 16) G4_MMF(16, 32) G4_MMF(16, 64) G4_MMF(32, 16) G4_MMF(32, 32) G4_MMF(32, 64) G4_MMF(64, 32) G4_MMF(64, 64)
#undef G4_MMF
        if (!run) return hipErrorInvalidValue;
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
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
