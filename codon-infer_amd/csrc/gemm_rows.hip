// Quantized GEMM for a few dozen rows: Y = epi(X W^T + b), X in f16 limbs
// (AF_H2, M <= GEMM_ROWS_MAX rows), W in Q8_0 / Q4_0 blocks or an FP32
// matrix's f16 pair copy.
//
// Same arithmetic as the other limb GEMMs (per 32-wide block tmp = hi x q +
// lo x q on f16 MFMA with FP32 accumulation, acc += d * tmp;
// matmul_tiled_q8/q4_parallel, codon-infer src/lib.rs:4870, 4937), for
// shapes that are bound by reading the weights once and by the latency of
// each launch: one short protein, or a few dozen decode rows.
//
//   * A workgroup owns 16 CT columns and all M rows; its 8 waves take every
//     8th k-block with the block's weights (straight from the compact quants,
//     each byte read by one wave) and activations in registers, several
//     blocks requested together.  No LDS and no barrier before the MFMAs.
//   * v_mfma_f32_16x16x32_f16 covers one k-block of 16 rows x 16 columns per
//     limb.  The waves' sums meet in LDS and are added in wave order, then the
//     epilogue: no partial sums in memory and no reduction kernel, except for
//     residual projections, whose K is cut across workgroups as well (their
//     N alone would not fill the CUs; the LayerNorm after them adds the
//     splits).
//   * Every workgroup reads all activations of its k-range, and a CU takes
//     about 45 B/ns from L2, so CT and the split are chosen for the fewest
//     bytes per CU (rows_plan).
//
// Against the register-staged GEMM, traced inside a 650M Q8_0 forward (us;
// before: QKV and FC1 with the reduction kernel of their splits; the LayerNorm
// that adds Wo's and FC2's is apart, 5.8 -> 4.9): at 41 rows QKV 13.7 -> 12.5,
// Wo 6.1 -> 5.1, FC1 15.8 -> 13.4, FC2 10.6 -> 7.6; at 9 rows 11.6 -> 5.4, 5.4
// -> 4.8, 12.2 -> 8.1, 7.7 -> 4.8.  Timed alone, with their activations read
// before, QKV and FC1 of 41 rows take 9.9 and 10.9.  Floors at 41 rows: 1.2 us
// for QKV's 5.5 MB at the 4.8 TB/s of a large copy, about 2.5 us for the
// launch.  One 41-token sequence of 650M Q8_0: 2.33 -> 2.00 ms per forward.
// Tried, alone: activations staged in LDS for 64-column workgroups with K
// split over the device and a fold kernel (QKV 10.9 us at 41 rows: the fold's
// 4.6 us eats the gain), 8 rows x 2 limbs per MFMA (10.1), workgroups starting
// at different k-blocks (no change).
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "kernels.h"
#include "x3.h"

namespace cih {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// One lane's 8 weights of k-block blk / N, column blk % N (k-group g): the raw
// bytes (Q8_0 / Q4_0) or the f16 values (pair copy)
template <int WF> struct WRaw {
    u32x2 q;
    __device__ __forceinline__ void load(const unsigned char *W, size_t blk, int g) {
        if constexpr (WF == WF_Q8) q = *reinterpret_cast<const u32x2 *>(W + blk * 32 + 8 * g);
        else q = *reinterpret_cast<const u32x2 *>(W + blk * 16 + 8 * (g & 1));
    }
    __device__ __forceinline__ f16x8 f16(int g) const {
        return __builtin_bit_cast(f16x8, quants_f16<WF>(q, (g >> 1) * 4));  // Q4_0: g = 2, 3 take the high nibbles
    }
};
template <> struct WRaw<WF_F16P> {
    f16x8 v;
    __device__ __forceinline__ void load(const unsigned char *W, size_t blk, int g) {
        v = *reinterpret_cast<const f16x8 *>(W + blk * 64 + 16 * g);
    }
    __device__ __forceinline__ f16x8 f16(int) const { return v; }
};

}  // namespace

// G: groups of 16 rows.  Grid (ceil(N / (16 CT)), splits); split y covers
// k-blocks [y kps, (y + 1) kps) and, when part is given, leaves its raw sums
// in part + y M N.  KBX: activation blocks per row (a pair copy's weight
// block kb meets activation block kb mod KBX).
template <int WF, int G, int CT>
__global__ __launch_bounds__(512) void k_gemm_rows(const unsigned short *__restrict__ X, int M, int KB, int KBX,
                                                   const unsigned char *__restrict__ Wq,
                                                   const float *__restrict__ Wsc, int N,
                                                   const float *__restrict__ bias, void *__restrict__ Yv, int ldy,
                                                   int epi, float *__restrict__ part, int kps) {
    constexpr int NW = 8, U = G * CT > 8 ? (G <= 3 ? 3 : 2) : (G <= 3 ? 5 : 4);  // waves; blocks in flight
    // floats per reduction row: 16-byte aligned, and the four row groups of a
    // store (4 rows apart) hit distinct banks
    constexpr int LD = 16 * CT + 4;
    __shared__ __attribute__((aligned(16))) float red[NW][G * 16][LD];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16 * CT;
    const int kb0 = blockIdx.y * kps, kb1 = min(KB, kb0 + kps);
    // this lane's row of each group and column of each tile (rows past M and
    // columns past N repeat the last; their sums are dropped)
    const unsigned short *xr[G];
#pragma unroll
    for (int q = 0; q < G; q++) xr[q] = X + (size_t)min(q * 16 + c, M - 1) * KBX * 64 + 8 * g;
    int n[CT];
#pragma unroll
    for (int t = 0; t < CT; t++) n[t] = min(n0 + 16 * t + c, N - 1);

    f32x4 acc[G][CT];
#pragma unroll
    for (int q = 0; q < G; q++)
#pragma unroll
        for (int t = 0; t < CT; t++) acc[q][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    // UU blocks kb, kb + NW, ...: every load first, then the MFMAs
    auto chunk = [&](int kb, auto UU) __attribute__((always_inline)) {
        constexpr int UV = decltype(UU)::value;
        WRaw<WF> b[UV][CT];
        float d[UV][CT];
        u32x4 a[UV][G][2];
#pragma unroll
        for (int u = 0; u < UV; u++) {
            const int k = kb + u * NW, ka = WF == WF_F16P && k >= KBX ? k - KBX : k;
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const size_t blk = (size_t)k * N + n[t];
                b[u][t].load(Wq, blk, g);
                d[u][t] = Wsc[blk];
            }
#pragma unroll
            for (int q = 0; q < G; q++)
#pragma unroll
                for (int l = 0; l < 2; l++)
                    a[u][q][l] = *reinterpret_cast<const u32x4 *>(xr[q] + (size_t)ka * 64 + l * 32);
        }
#pragma unroll
        for (int u = 0; u < UV; u++)
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const f16x8 wv = b[u][t].f16(g);
                f32x4 v[G];
#pragma unroll
                for (int q = 0; q < G; q++)
                    v[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[u][q][0]), wv, zero, 0, 0,
                                                                  0);
#pragma unroll
                for (int q = 0; q < G; q++)
                    v[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[u][q][1]), wv, v[q], 0, 0,
                                                                  0);
#pragma unroll
                for (int q = 0; q < G; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[q][t][e] = __builtin_fmaf(d[u][t], v[q][e], acc[q][t][e]);
            }
    };
    int kb = kb0 + w, left = (kb1 - kb + NW - 1) / NW;  // this wave's blocks
    for (; left >= U; left -= U, kb += NW * U) chunk(kb, std::integral_constant<int, U>{});
    switch (left) {
    case 4:
        if constexpr (U > 4) chunk(kb, std::integral_constant<int, 4>{});
        break;
    case 3:
        if constexpr (U > 3) chunk(kb, std::integral_constant<int, 3>{});
        break;
    case 2: chunk(kb, std::integral_constant<int, 2>{}); break;
    case 1: chunk(kb, std::integral_constant<int, 1>{}); break;
    default: break;
    }
    // lane holds rows 16 q + 4 g + e, columns 16 t + c
#pragma unroll
    for (int q = 0; q < G; q++)
#pragma unroll
        for (int t = 0; t < CT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) red[w][q * 16 + 4 * g + e][16 * t + c] = acc[q][t][e];
    __syncthreads();
    // one thread per row and four columns; the waves' sums in wave order
    for (int it = tid; it < M * 4 * CT; it += 64 * NW) {
        const int row = it / (4 * CT), c4 = 4 * (it % (4 * CT)), col = n0 + c4;
        if (col >= N) continue;
        f32x4 v = *reinterpret_cast<const f32x4 *>(&red[0][row][c4]);
#pragma unroll
        for (int s = 1; s < NW; s++) v += *reinterpret_cast<const f32x4 *>(&red[s][row][c4]);
        if (part) {
            *reinterpret_cast<f32x4 *>(part + ((size_t)blockIdx.y * M + row) * N + col) = v;
            continue;
        }
        if (bias) v += *reinterpret_cast<const f32x4 *>(bias + col);
        if (epi == EPI_GELU || epi == EPI_GELU_H2)
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = gelu_as(v[e]);
        if (epi == EPI_GELU_H2) {
            h2_store4(static_cast<unsigned short *>(Yv), row, col, N, make_float4(v.x, v.y, v.z, v.w));
        } else {
            f32x4 *dst = reinterpret_cast<f32x4 *>(static_cast<float *>(Yv) + (size_t)row * ldy + col);
            if (epi == EPI_RESIDUAL) v = *dst + v;
            *dst = v;
        }
    }
}

bool gemm_rows_applies(const DevMatrix &W, int a_fmt, int M, int epi) {
    if (a_fmt != AF_H2 || M < 1 || M > GEMM_ROWS_MAX || W.N <= 0 || W.N % 16 || W.K % 32 || W.K <= 0) return false;
    if (W.fmt != WF_Q8 && W.fmt != WF_Q4 && W.fmt != WF_F16P) return false;
    if (epi != EPI_NONE && epi != EPI_RESIDUAL && epi != EPI_GELU && epi != EPI_GELU_H2) return false;
    if (epi == EPI_GELU_H2 && W.N % 32) return false;
    // From 49 rows on the LDS GEMM's 64-row tiles take over, except where K is
    // short or the LayerNorm after the projection adds many splits anyway
    // (timed alone, us at 48 / 64 rows, this kernel against 64 x 64 tiles: 650M QKV 10.5 /
    // 12.5 against 10.6 / 10.7, FC1 11.5 / 13.5 against 12.6 / 12.7, FC2 with
    // its LayerNorm 12.0 / 13.6 against 14.7 / 15.0; 35M QKV 5.3 / 6.1 against
    // 6.0 / 5.7; 8M FC1 4.4 / 5.0 against 5.8 / 5.4; 3B FC2 21.8 / 28.6 against
    // 21.8 / 22.8).
    if (M > 48 && W.K > (epi == EPI_RESIDUAL ? 5120 : 512)) return false;
    // the k-sum is regrouped by wave: CIH_SPLITK=0 keeps whole-K sums; the
    // switches that choose among the other GEMMs turn this one off
    const char *re = getenv("CIH_GEMM_ROWS"), *ke = getenv("CIH_SPLITK"), *pe = getenv("CIH_GEMM_PLAN");
    return !(re && !strcmp(re, "0")) && !(ke && !strcmp(ke, "0")) && !(pe && !strcmp(pe, "0")) &&
           !getenv("CIH_GEMM_LDS") && !getenv("CIH_GEMM_TILE") && !getenv("CIH_GEMM_TILE_N") &&
           !getenv("CIH_GEMM_TILE_N_GELU") && !getenv("CIH_GEMM_KW");
}

template <int WF, int G>
static hipError_t launch_rows_g(const DevMatrix &W, int KB, int KBX, const unsigned short *X, const float *bias,
                                void *Y, int ldy, int M, int epi, float *part, int S, int kps, int ct,
                                hipStream_t st) {
    const unsigned char *q = static_cast<const unsigned char *>(W.q);
    const dim3 grid((W.N + 16 * ct - 1) / (16 * ct), S), block(512);
#define CIH_ROWS(CT)                                                                                               \
    hipLaunchKernelGGL((k_gemm_rows<WF, G, CT>), grid, block, 0, st, X, M, KB, KBX, q, W.sc, W.N, bias, Y, ldy,     \
                       epi, part, kps)
    if (ct == 1) CIH_ROWS(1);
    else if (ct == 2) CIH_ROWS(2);
    else if (ct == 4) CIH_ROWS(4);
    else return hipErrorInvalidValue;
#undef CIH_ROWS
    return hipGetLastError();
}

template <int WF>
static hipError_t launch_rows_w(const DevMatrix &W, int KB, int KBX, const unsigned short *X, const float *bias,
                                void *Y, int ldy, int M, int epi, float *part, int S, int kps, int ct,
                                hipStream_t st) {
    switch ((M + 15) / 16) {
    case 1: return launch_rows_g<WF, 1>(W, KB, KBX, X, bias, Y, ldy, M, epi, part, S, kps, ct, st);
    case 2: return launch_rows_g<WF, 2>(W, KB, KBX, X, bias, Y, ldy, M, epi, part, S, kps, ct, st);
    case 3: return launch_rows_g<WF, 3>(W, KB, KBX, X, bias, Y, ldy, M, epi, part, S, kps, ct, st);
    default: return launch_rows_g<WF, 4>(W, KB, KBX, X, bias, Y, ldy, M, epi, part, S, kps, ct, st);
    }
}

// Column tiles per workgroup and k-splits: the fewest bytes a CU takes (its
// workgroups' activations and weights, one after the other when there are
// more than CUs), at the 45 B/ns a CU gets from L2.  Splits add the partial
// sums' traffic (4 TB/s) and, unless the caller folds them into its next
// kernel, a fold launch of 4.6 us.  Within 5% of the best of CT x S timed alone
// on the ESM-2 projections at 9 to 48 rows; inside a forward, where the wide
// projections take 1 to 3 us more, the choices have not been compared.
static void rows_plan(int M, int N, int KB, bool deferred, size_t part_floats, double wbyte, int &ct, int &S) {
    const long cus = device_cus();
    const double rowb = (M + 15) / 16 * 16 * 128.0;
    double best = 0;
    for (int t = 1; t <= 4; t *= 2)
        for (int s = 1; s <= 16; s++) {
            const int kps = (KB + s - 1) / s;
            if ((KB + kps - 1) / kps != s || (s > 1 && (kps < 4 || (size_t)s * M * N > part_floats))) continue;
            const long wgs = (long)((N + 16 * t - 1) / (16 * t)) * s;
            double cost = (double)((wgs + cus - 1) / cus) * kps * (rowb + 16 * t * 32 * wbyte) / 45.0;
            if (s > 1) cost += 2.0 * 4.0 * s * M * N / 4000.0 + (deferred ? 0.0 : 4600.0);
            if (best == 0 || cost < best) {
                best = cost;
                ct = t;
                S = s;
            }
        }
}

hipError_t launch_gemm_rows(const DevMatrix &W, const unsigned short *X, const float *bias, void *Y, int ldy, int M,
                            int epi, const PartialBuf *pb, int *defer, hipStream_t st) {
    if (defer) *defer = 0;
    if (M <= 0) return hipSuccess;
    if (!gemm_rows_applies(W, AF_H2, M, epi) || !X || !W.q || !W.sc || (epi != EPI_GELU_H2 && (ldy < W.N || ldy % 4)))
        return hipErrorInvalidValue;
    const int KBX = W.K / 32, KB = WF_F16P == W.fmt ? 2 * KBX : KBX;
    int ct = 1, S = 1;
    const bool deferred = defer && epi == EPI_RESIDUAL;
    rows_plan(M, W.N, KB, deferred, pb && pb->part ? pb->floats : 0,
              W.fmt == WF_Q8 ? 1.125 : (W.fmt == WF_Q4 ? 0.625 : 2.125), ct, S);
    const int kps = (KB + S - 1) / S;
    float *pp = S > 1 ? pb->part : nullptr;
    hipError_t e;
    if (W.fmt == WF_Q8) e = launch_rows_w<WF_Q8>(W, KB, KBX, X, bias, Y, ldy, M, epi, pp, S, kps, ct, st);
    else if (W.fmt == WF_Q4) e = launch_rows_w<WF_Q4>(W, KB, KBX, X, bias, Y, ldy, M, epi, pp, S, kps, ct, st);
    else e = launch_rows_w<WF_F16P>(W, KB, KBX, X, bias, Y, ldy, M, epi, pp, S, kps, ct, st);
    if (S > 1 && e == hipSuccess) {
        if (deferred) *defer = S;
        else e = launch_splitk_reduce(pb->part, S, M, W.N, bias, Y, ldy, epi, st);
    }
    return e;
}

}  // namespace cih
