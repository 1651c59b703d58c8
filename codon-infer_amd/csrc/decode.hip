// Autoregressive decoding against a per-slot KV cache: rotary embedding of
// the new rows' Q and K with their K/V written into the cache, and causal
// attention of each new row over its slot's positions 0..pos.  Replaces the
// cache write and attention_head_avx1 of forward / forward_q8 / forward_q4
// (codon-infer src/lib.rs:3616-3663, 3438-3483).
#include <math.h>

#include <type_traits>

#include "head_wo.h"
#include "kernels.h"
#include "x3.h"

namespace cih {

namespace {

constexpr int DEC_THREADS = 256;

// apply_rope (lib.rs:3533-3552) on row r's Q (in place) and K (into the
// cache at the row's position); V is copied to the cache.  Products and sums
// are rounded one by one as the reference computes them (no fused multiply-add).
__global__ __launch_bounds__(DEC_THREADS) void k_rope_kv(float *__restrict__ qkv, int d, int hd,
                                                         const int *__restrict__ rows, const float *__restrict__ rc,
                                                         const float *__restrict__ rs, float *__restrict__ kc,
                                                         float *__restrict__ vc, int64_t slot_stride) {
    const int r = blockIdx.x;
    const int slot = rows[2 * r], pos = rows[2 * r + 1];
    const int half = hd / 2;
    float *q = qkv + (size_t)r * 3 * d;
    const float *k = q + d, *v = q + 2 * d;
    float *kd = kc + slot * slot_stride + (size_t)pos * d;
    float *vd = vc + slot * slot_stride + (size_t)pos * d;
    const float *c = rc + (size_t)pos * half, *s = rs + (size_t)pos * half;
    for (int i = threadIdx.x; i < d / 2; i += DEC_THREADS) {
        const int h = i / half, j = i - h * half;
        const int i0 = h * hd + j, i1 = i0 + half;
        const float cj = c[j], sj = s[j];
        const float q0 = q[i0], q1 = q[i1], k0 = k[i0], k1 = k[i1];
        q[i0] = __fsub_rn(__fmul_rn(q0, cj), __fmul_rn(q1, sj));
        q[i1] = __fadd_rn(__fmul_rn(q1, cj), __fmul_rn(q0, sj));
        kd[i0] = __fsub_rn(__fmul_rn(k0, cj), __fmul_rn(k1, sj));
        kd[i1] = __fadd_rn(__fmul_rn(k1, cj), __fmul_rn(k0, sj));
    }
    for (int i = threadIdx.x; i < d; i += DEC_THREADS) vd[i] = v[i];
}

constexpr int ATT_THREADS = 512;  // 8 waves per (row, head)

typedef float f32x4 __attribute__((ext_vector_type(4)));

// v of the lane that DPP control C names (all lanes read a valid one)
template <int C> __device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), C, 0xf, 0xf, true));
}

__device__ __forceinline__ float block_reduce(float v, float *scratch, bool is_max) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float u = __shfl_xor(v, o);
        v = is_max ? fmaxf(v, u) : v + u;
    }
    const int w = threadIdx.x >> 6;
    __syncthreads();  // scratch free from the previous reduction
    if ((threadIdx.x & 63) == 0) scratch[w] = v;
    __syncthreads();
    float r = scratch[0];
#pragma unroll
    for (int i = 1; i < ATT_THREADS / 64; i++) r = is_max ? fmaxf(r, scratch[i]) : r + scratch[i];
    return r;
}

// One workgroup per (row, head).  Scores s_t = (q . k_t) / sqrt(hd) for
// t = 0..pos, softmax as softmax() (lib.rs:3500-3504: max, exp(s - max),
// 1 / sum), then out = sum_t p_t v_t.  Bound by reading the slot's K and V
// (512 bytes a key at hd 64) at the 45 B/ns a CU takes: L = HD / 4 lanes read
// a row in 16-byte pieces, so a wave's load covers 64 / L whole rows, and
// each wave has U such loads in flight (eight, or 1, 2 or 4 that cover all
// keys), the first U of K and of V requested before anything else.  A key's score is added over its lanes, an output
// dim over a lane's keys, the wave's key groups and the waves, in that order.
// (A thread per key row, and V rows four at a time by 64 lanes, took 28.8 us
// per layer for 8 rows at position 700 of 650M and 13.9 us for one at 280;
// now 17.4 and 10.6; a prompt's rows 97 -> 61 us at 256 rows per call.
// Keeping V's second sweep in K's registers under the softmax changed neither
// and cost the prompt's rows their second workgroup per CU, 61 -> 101.)
//
// FUSED (each slot at most once in the launch): the workgroup also applies
// RoPE to its head's Q and K, writes K and V at pos into the cache for later
// steps, and takes key pos from LDS rather than from the cache, so no
// workgroup reads what another one writes.  Otherwise k_rope_kv has run.
//
// WOF (WF_Q8 / WF_Q4; 0: none): instead of storing the head's output, the
// workgroup multiplies it by the head's k-blocks of Wo (HeadWo) for columns
// [z 128 WP, (z + 1) 128 WP), z = blockIdx.z, into wo_part + (h n + r) N:
// the heads are the projection's splits.  Its weights are requested before
// the attention, which each column chunk repeats (only chunk 0 writes the
// cache).  WP = 1 for one row, 2 for two (650M Q4_0: one stream 929 -> 940
// tokens/s with 128 columns, two streams 1,728 with 256 against 1,532).
template <int HD, bool FUSED, int OF, int WOF = 0, int WP = 2>
__global__ __launch_bounds__(ATT_THREADS) void k_decode_attention(const float *__restrict__ qkv,
                                                                  const float *__restrict__ part, int splits,
                                                                  const float *__restrict__ bias, int d,
                                                                  const int *__restrict__ rows,
                                                                  const float *__restrict__ rc,
                                                                  const float *__restrict__ rs, float *__restrict__ kc,
                                                                  float *__restrict__ vc, int64_t slot_stride,
                                                                  float inv_scale, float *__restrict__ out,
                                                                  const unsigned char *__restrict__ wo_q = nullptr,
                                                                  const float *__restrict__ wo_sc = nullptr,
                                                                  int wo_n = 0) {
    constexpr int HALF = HD / 2, NWV = ATT_THREADS / 64;
    constexpr int LK = HD == 24 ? 8 : HD / 4;  // lanes per key (hd 24: lanes 6 and 7 of 8 idle)
    constexpr int KW = 64 / LK;                // keys per load of a wave
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *qs = sm;                        // [HD] rotated query
    float *kcur = qs + HD, *vcur = kcur + HD;  // [HD] key and value at pos (FUSED)
    float *gsum = vcur + HD;               // [NWV][HD] per-wave partial outputs
    float *red = gsum + ATT_THREADS;       // [8]
    float *p = red + 8;                    // [pos + 1]
    const int r = blockIdx.x, h = blockIdx.y;
    const int slot = rows[2 * r], pos = rows[2 * r + 1];
    float *K = kc + slot * slot_stride + h * HD;
    float *V = vc + slot * slot_stride + h * HD;
    const int t = threadIdx.x;
    const int n_cached = FUSED ? pos : pos + 1;  // keys read from the cache
    constexpr int NKB = HD / 32;
    HeadWo<WOF ? WOF : WF_Q8, WP> wo;
    const int wc0 = (int)blockIdx.z * 128 * WP, wc1 = min(wc0 + 128 * WP, wo_n);
    if constexpr (WOF != 0) wo.load(wo_q, wo_sc, wo_n, h * NKB, NKB, wc0, wc1);
    const bool cache_writer = WOF == 0 || blockIdx.z == 0;
    // key j of (sweep s0, load u): s0 + (u NWV + wave) KW + lane / LK; this
    // lane's quad of its dims
    const int lane = t & 63, wave = t >> 6, kq = lane / LK, dl = 4 * min(lane % LK, HD / 4 - 1);
    const bool live = lane % LK < HD / 4;
    const float *Kl = K + dl, *Vl = V + dl;
    auto key = [&](int s0, int u) __attribute__((always_inline)) { return s0 + (u * NWV + wave) * KW + kq; };
    f32x4 o4 = {0.0f, 0.0f, 0.0f, 0.0f};
    auto attend = [&](auto UU) __attribute__((always_inline)) {
        // keys past the cached ones re-read the last (their scores are not stored, their weights zero)
        constexpr int U = decltype(UU)::value, STEP = NWV * KW * U;  // loads in flight, keys per sweep of the workgroup
        auto fetch = [&](const float *base, int s0, f32x4 (&v)[U]) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; u++)
                v[u] = *reinterpret_cast<const f32x4 *>(base + (size_t)min(key(s0, u), n_cached - 1) * d);
        };
        // The first sweep of K and of V is requested before anything waits, so its
        // latency overlaps the gather, the rotation, the softmax and the barriers.
        f32x4 kv[U], vv[U];
        if (n_cached > 0) {
            fetch(Kl, 0, kv);
            fetch(Vl, 0, vv);
        }
        if constexpr (FUSED) {
            float c = 0.0f, s = 0.0f;
            if (t < HALF) {
                c = rc[(size_t)pos * HALF + t];
                s = rs[(size_t)pos * HALF + t];
            }
            // this head's q, k, v: the row of qkv, or the GEMV's partial sums
            // (eight interleaved sums over the splits) + bias
            if (t < 3 * HD) {
                const int which = t / HD, col = which * d + h * HD + (t - which * HD);
                float v;
                if (part) {
                    const size_t stride = (size_t)gridDim.x * 3 * d;
                    const float *pp = part + (size_t)r * 3 * d + col;
                    float a[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                    int y = 0;
                    for (; y + 8 <= splits; y += 8) {
#pragma unroll
                        for (int u = 0; u < 8; u++) a[u] += pp[(y + u) * stride];
                    }
                    for (int u = 0; y < splits; y++, u++) a[u] += pp[y * stride];
                    v = (((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]))) + bias[col];
                } else {
                    v = qkv[(size_t)r * 3 * d + col];
                }
                qs[t] = v;  // qs | kcur | vcur are contiguous
            }
            __syncthreads();
            // apply_rope (lib.rs:3533-3552) for this head, products rounded one by one
            if (t < HALF) {
                const float q0 = qs[t], q1 = qs[t + HALF], k0 = kcur[t], k1 = kcur[t + HALF];
                qs[t] = __fsub_rn(__fmul_rn(q0, c), __fmul_rn(q1, s));
                qs[t + HALF] = __fadd_rn(__fmul_rn(q1, c), __fmul_rn(q0, s));
                const float r0 = __fsub_rn(__fmul_rn(k0, c), __fmul_rn(k1, s));
                const float r1 = __fadd_rn(__fmul_rn(k1, c), __fmul_rn(k0, s));
                kcur[t] = r0;
                kcur[t + HALF] = r1;
                if (cache_writer) {
                    K[(size_t)pos * d + t] = r0;
                    K[(size_t)pos * d + t + HALF] = r1;
                }
            } else if (t >= 64 && t < 64 + HD && cache_writer) {
                V[(size_t)pos * d + t - 64] = vcur[t - 64];
            }
        } else {
            const float *q = qkv + (size_t)r * 3 * d + h * HD;
            if (t < HD) qs[t] = q[t];
        }
        __syncthreads();
        const f32x4 q4 = *reinterpret_cast<const f32x4 *>(qs + dl);
        // a key's products over its lanes: DPP adds within 16 lanes (quads, halves
        // of 8, mirrored: partners hold equal sums by then)
        auto key_sum = [&](f32x4 k) __attribute__((always_inline)) {
            float a = live ? fmaf(q4.w, k.w, fmaf(q4.z, k.z, fmaf(q4.y, k.y, q4.x * k.x))) : 0.0f;
            a += dpp<0xB1>(a);                            // lane ^ 1
            a += dpp<0x4E>(a);                            // lane ^ 2
            if constexpr (LK >= 8) a += dpp<0x141>(a);    // mirrored in 8
            if constexpr (LK >= 16) a += dpp<0x140>(a);   // mirrored in 16
            return a;
        };
        for (int s0 = 0; s0 < n_cached; s0 += STEP) {
            float a[U];
#pragma unroll
            for (int u = 0; u < U; u++) a[u] = key_sum(kv[u]);
            if (s0 + STEP < n_cached) fetch(Kl, s0 + STEP, kv);
#pragma unroll
            for (int u = 0; u < U; u++)
                if (lane % LK == 0 && key(s0, u) < n_cached) p[key(s0, u)] = a[u] * inv_scale;
        }
        if (FUSED && wave == 0) {
            const float a = key_sum(*reinterpret_cast<const f32x4 *>(kcur + dl));
            if (lane == 0) p[pos] = a * inv_scale;
        }
        __syncthreads();
        float mx = -INFINITY;
        for (int j = t; j <= pos; j += ATT_THREADS) mx = fmaxf(mx, p[j]);
        mx = block_reduce(mx, red, true);
        float sum = 0.0f;
        for (int j = t; j <= pos; j += ATT_THREADS) {
            const float e = expf(p[j] - mx);
            p[j] = e;
            sum += e;
        }
        sum = block_reduce(sum, red, false);
        const float inv = 1.0f / sum;
        __syncthreads();
        for (int s0 = 0; s0 < n_cached; s0 += STEP) {
            if (s0 > 0) fetch(Vl, s0, vv);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int j = key(s0, u);
                const float w = j < n_cached ? p[j] * inv : 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) o4[e] = fmaf(w, vv[u][e], o4[e]);
            }
        }
        if (FUSED && wave == 0 && kq == 0) {
            const float w = p[pos] * inv;
            const f32x4 v = *reinterpret_cast<const f32x4 *>(vcur + dl);
#pragma unroll
            for (int e = 0; e < 4; e++) o4[e] = fmaf(w, v[e], o4[e]);
        }
    };
    // As many loads in flight as the cached keys fill, up to eight: the ones past
    // the last key would still pass through the CU's load path (with eight
    // throughout: 8M Q4_0, a prompt of 439 rows 0.73 -> 0.62 ms; 650M Q4_0, one
    // stream at position 30 1.038 -> 0.989 ms per step)
    const int need = (n_cached + NWV * KW - 1) / (NWV * KW);
    if (need <= 1) attend(std::integral_constant<int, 1>{});
    else if (need <= 2) attend(std::integral_constant<int, 2>{});
    else if (need <= 4) attend(std::integral_constant<int, 4>{});
    else attend(std::integral_constant<int, 8>{});
    // the wave's key groups, then the waves
#pragma unroll
    for (int o = LK; o < 64; o <<= 1)
#pragma unroll
        for (int e = 0; e < 4; e++) o4[e] += __shfl_xor(o4[e], o);
    if (kq == 0 && live) *reinterpret_cast<f32x4 *>(gsum + wave * HD + dl) = o4;
    __syncthreads();
    if (t < HD) {
        float o = gsum[t];
#pragma unroll
        for (int k = 1; k < NWV; k++) o += gsum[k * HD + t];
        if constexpr (WOF != 0) qs[t] = o;  // the query is no longer read
        else if constexpr (OF == AF_H2) h2_store(reinterpret_cast<unsigned short *>(out), r, h * HD + t, d, o);
        else out[(size_t)r * d + h * HD + t] = o;
    }
    if constexpr (WOF != 0) {
        static_assert(HD % 32 == 0, "heads of whole 32-wide blocks");
        __syncthreads();
        wo.run(qs, HD, 1, NKB, wo_n, wc0, wc1, out + ((size_t)h * gridDim.x + r) * wo_n);
    }
}

}  // namespace

size_t decode_attention_lds(int hd, int max_len) {
    return sizeof(float) * (3 * (size_t)hd + ATT_THREADS + 8 + (size_t)max_len);
}

hipError_t launch_rope_kv(float *qkv, int d, int hd, const int *rows, int n, const float *rope_c, const float *rope_s,
                          float *kc, float *vc, int64_t slot_stride, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_rope_kv, dim3(n), dim3(DEC_THREADS), 0, st, qkv, d, hd, rows, rope_c, rope_s, kc, vc,
                       slot_stride);
    return hipGetLastError();
}

template <bool FUSED>
static hipError_t launch_att(const float *qkv, const float *part, int splits, const float *bias, int d, int H,
                             const int *rows, int n, int max_len, const float *rc, const float *rs, float *kc,
                             float *vc, int64_t slot_stride, float *out, int out_fmt, hipStream_t st) {
    const int hd = d / H;
    const float inv_scale = 1.0f / sqrtf((float)hd);
    const size_t lds = decode_attention_lds(hd, max_len);
    const dim3 grid(n, H), block(ATT_THREADS);
    if (out_fmt != AF_F32 && (out_fmt != AF_H2 || d % 32)) return hipErrorInvalidValue;
#define CIH_ATT_CASE(HDV)                                                                                           \
    case HDV:                                                                                                      \
        if (out_fmt == AF_H2)                                                                                      \
            hipLaunchKernelGGL((k_decode_attention<HDV, FUSED, AF_H2>), grid, block, lds, st, qkv, part, splits,   \
                               bias, d, rows, rc, rs, kc, vc, slot_stride, inv_scale, out);                        \
        else                                                                                                       \
            hipLaunchKernelGGL((k_decode_attention<HDV, FUSED, AF_F32>), grid, block, lds, st, qkv, part, splits,  \
                               bias, d, rows, rc, rs, kc, vc, slot_stride, inv_scale, out);                        \
        break;
    switch (hd) {
        CIH_ATT_CASE(16)
        CIH_ATT_CASE(24)
        CIH_ATT_CASE(32)
        CIH_ATT_CASE(64)
    default: return hipErrorInvalidValue;
    }
#undef CIH_ATT_CASE
    return hipGetLastError();
}

hipError_t launch_decode_attention(const float *qkv, int d, int H, const int *rows, int n, int max_len,
                                   const float *kc, const float *vc, int64_t slot_stride, float *out,
                                   hipStream_t st, int out_fmt) {
    if (n <= 0) return hipSuccess;
    return launch_att<false>(qkv, nullptr, 0, nullptr, d, H, rows, n, max_len, nullptr, nullptr,
                             const_cast<float *>(kc), const_cast<float *>(vc), slot_stride, out, out_fmt, st);
}

hipError_t launch_decode_attention_fused_wo(float *qkv, const float *part, int splits, const float *bias, int d, int H,
                                            const int *rows, int n, int max_len, const float *rope_c,
                                            const float *rope_s, float *kc, float *vc, int64_t slot_stride,
                                            const DevMatrix &Wo, float *wo_part, size_t wo_part_floats,
                                            hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int hd = H > 0 ? d / H : 0;
    if ((part && (!bias || splits < 1)) || hd * H != d || (hd != 32 && hd != 64) ||
        (Wo.fmt != WF_Q8 && Wo.fmt != WF_Q4) || Wo.K != d || Wo.N % 16 || !wo_part ||
        (size_t)H * n * Wo.N > wo_part_floats)
        return hipErrorInvalidValue;
    const float inv_scale = 1.0f / sqrtf((float)hd);
    const size_t lds = decode_attention_lds(hd, max_len);
    const int wp = n == 1 ? 1 : 2;  // Wo columns per workgroup: 128 wp
    const dim3 grid(n, H, (Wo.N + 128 * wp - 1) / (128 * wp)), block(ATT_THREADS);
    const unsigned char *wq = static_cast<const unsigned char *>(Wo.q);
#define CIH_ATT_WO(HDV, WFV)                                                                                          \
    if (wp == 1)                                                                                                      \
        hipLaunchKernelGGL((k_decode_attention<HDV, true, AF_F32, WFV, 1>), grid, block, lds, st, qkv, part, splits,  \
                           bias, d, rows, rope_c, rope_s, kc, vc, slot_stride, inv_scale, wo_part, wq, Wo.sc, Wo.N);  \
    else                                                                                                              \
        hipLaunchKernelGGL((k_decode_attention<HDV, true, AF_F32, WFV, 2>), grid, block, lds, st, qkv, part, splits,  \
                           bias, d, rows, rope_c, rope_s, kc, vc, slot_stride, inv_scale, wo_part, wq, Wo.sc, Wo.N)
    if (hd == 64 && Wo.fmt == WF_Q8) {
        CIH_ATT_WO(64, WF_Q8);
    } else if (hd == 64) {
        CIH_ATT_WO(64, WF_Q4);
    } else if (Wo.fmt == WF_Q8) {
        CIH_ATT_WO(32, WF_Q8);
    } else {
        CIH_ATT_WO(32, WF_Q4);
    }
#undef CIH_ATT_WO
    return hipGetLastError();
}

hipError_t launch_decode_attention_fused(float *qkv, const float *part, int splits, const float *bias, int d, int H,
                                         const int *rows, int n, int max_len, const float *rope_c,
                                         const float *rope_s, float *kc, float *vc, int64_t slot_stride, float *out,
                                         hipStream_t st, int out_fmt) {
    if (n <= 0) return hipSuccess;
    if (part && (!bias || splits < 1)) return hipErrorInvalidValue;
    return launch_att<true>(qkv, part, splits, bias, d, H, rows, n, max_len, rope_c, rope_s, kc, vc, slot_stride, out,
                            out_fmt, st);
}

}  // namespace cih
