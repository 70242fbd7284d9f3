// The offline Base/Ortho sieve on the device: what /root/reference/tools/sieve.py:13-95
// computes with torch ops, as four small kernels with the arithmetic of
// those ops on a GPU tensor (so that the results carry the same bits).
//
//  quantize_int4 (:13-23)   one workgroup per row: max|w| (NaN propagates),
//                            clamp at 1e-8 in w's dtype, s = max * fp32(1/7)
//                            (torch divides a GPU tensor by a host scalar
//                            through its reciprocal; a CPU tensor by IEEE
//                            division, the ieee_div mode), q = clamp(rint(w / s), -8, 7),
//                            w_base = q * s, non-finite results 0.  Every
//                            intermediate is rounded to w's dtype, as the
//                            torch ops round each result.
//  hessian_sieve (:25-76)   the same pass also writes the score residual^2 /
//                            (H_inv + 1e-6); with a sparsity target, the k-th
//                            largest score is found by a radix select over the
//                            order-preserving key of each FP32 score (NaN
//                            largest, as torch.topk): 11 bits counted in the
//                            first pass itself, 11 in a pass over the scores
//                            that also collects those of the found prefix, 10
//                            over the collected ones; then w_ortho = residual *
//                            (score > t), both formed again from w and w_base.
//  compute_hessian_diag_approx (:79-95)  diag(X^T X) / n + 1e-6: the
//                            diagonal only (column sums of squares, FP32
//                            partial sums over row slices added in slice
//                            order), not the K x K product.
//
// Off the forward path: these run once per weight matrix when a model is
// split, and are measured as load-time work.  The split is bound by memory:
// w read and w_base and the scores written, the scores read once, w and
// w_base read and w_ortho written, 28 bytes an FP32 weight.  4096 x 4096 FP32,
// 2 % kept: 106 us (40 + 16 + 5 + 36 in the passes, 5 TB/s), against 371 us with
// the residual stored, four 8-bit passes over all scores (58 us each, on a
// handful of histogram bins' LDS atomics) and a one-thread scan after each.
#include <atomic>
#include <type_traits>

#include "orth_common.h"

namespace orth {

constexpr int kSieveNT = 256;

__device__ __forceinline__ float sieve_max_nan(float a, float b) {
    // torch's max propagates NaN
    return (a != a || b != b) ? __builtin_nanf("") : fmaxf(a, b);
}

// Order-preserving key of an FP32 value, NaN above everything (the key
// torch.topk selects on).
__device__ __forceinline__ uint32_t sieve_key(float f) {
    const uint32_t x = __float_as_uint(f);
    if (f != f) return 0xffffffffu;
    return x ^ ((x & 0x80000000u) ? 0xffffffffu : 0x80000000u);
}

__device__ __forceinline__ float sieve_unkey(uint32_t k) {
    if (k == 0xffffffffu) return __builtin_nanf("");
    return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

struct SieveArgs {
    const void *w;
    int64_t N, K;
    void *w_base;
    void *w_ortho;      // or null: quantise only
    float *score;       // [N*K] score values (exact in FP32), or null
    const void *h;      // H_inv: element k at h[k * h_stride]
    int hdt;
    int64_t h_stride;
    int score_dt;       // dtype of the score (torch's promotion of w's and H's)
    int ieee_div;       // 1: division by a host scalar as IEEE division (CPU
                        // tensors), 0: as a product with its FP32 reciprocal
    int keep;           // the first pass stores the residual in w_ortho (else the
                        // last one forms it again from w and w_base)
    struct SieveSel *sel;  // radix select, or null: the threshold below
    uint32_t rank;
    float thresh;
};

// v / d for a host scalar d, as torch computes it on the tensor's device.
__device__ __forceinline__ float sieve_scalar_div(float v, float d, int ieee_div) {
    return ieee_div ? v / d : v * (1.0f / d);
}

constexpr int kSvNT = 512;                      // threads of the split's passes
constexpr int kSvLdsCols = 16384;               // columns of h + 1e-6 a workgroup keeps in LDS
constexpr int kSvCache = 4;                     // vectors of a row per thread kept in registers
constexpr int kSvLanes = 4;                     // LDS histograms, by lane

__global__ void __launch_bounds__(256) sieve_sel_init_kernel(SieveSel *st) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < 3 * kSelCopies * kSelBins) (&st->hist[0][0][0])[i] = 0u;
}

// The bin of level `lv` (from the top) that holds the k-th largest key, and
// the rank within it; every thread of the workgroup gets both.  Workgroup 0
// records them for the later passes.
__device__ void sieve_pick(SieveSel *st, int lv, uint32_t k, uint32_t &bin, uint32_t &left) {
    __shared__ uint32_t part[kSvNT / 64], found[2];
    constexpr int PER = kSelBins / kSvNT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        c[j] = 0;
#pragma unroll
        for (int i = 0; i < kSelCopies; i++) c[j] += st->hist[lv][i][tid * PER + j];
        sum += c[j];
    }
    uint32_t incl = sum;  // keys in this thread's bins and those of later lanes, then of later waves
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_down(incl, off);
        if (lane + off < 64) incl += v;
    }
    if (lane == 0) part[wave] = incl;
    __syncthreads();
    uint32_t above = incl - sum;
    for (int w = wave + 1; w < kSvNT / 64; w++) above += part[w];
#pragma unroll
    for (int j = PER - 1; j >= 0; j--) {
        if (k > above && k <= above + c[j]) {  // (one bin of one thread)
            found[0] = (uint32_t)(tid * PER + j);
            found[1] = k - above;
        }
        above += c[j];
    }
    __syncthreads();
    bin = found[0];
    left = found[1];
    if (blockIdx.x == 0 && tid == 0 && lv < 2) {
        st->bin[lv] = bin;
        st->left[lv] = left;
    }
}

// a * b as an FP32 product of its own: rounded to FP16 at once the compiler
// makes it a fused multiply-add with +0, which turns a product of -0 into +0.
__device__ __forceinline__ float sieve_mul(float a, float b) {
    float p = a * b;
    asm("" : "+v"(p));
    return p;
}

// V consecutive elements from i, as floats.
template <int DT, int V>
__device__ __forceinline__ void sieve_load(const void *p, int64_t i, float v[V]) {
    if constexpr (V == 1) {
        v[0] = load_as_f32(p, DT, i);
    } else if constexpr (DT == ORTH_DT_F32) {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(p) + i);
#pragma unroll
        for (int e = 0; e < V; e++) v[e] = a[e];
    } else {
        const uint2 a = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(p) + i);
        const uint32_t u[2] = {a.x, a.y};
#pragma unroll
        for (int e = 0; e < V; e++) {
            const uint16_t b = (uint16_t)(u[e >> 1] >> (16 * (e & 1)));
            v[e] = DT == ORTH_DT_F16 ? (float)__builtin_bit_cast(f16, b) : bf16_bits_to_f32(b);
        }
    }
}

template <int DT, int V>
__device__ __forceinline__ void sieve_store(void *p, int64_t i, const float v[V]) {
    if constexpr (V == 1) {
        store_from_f32(p, DT, i, v[0]);
    } else if constexpr (DT == ORTH_DT_F32) {
        *reinterpret_cast<f32x4 *>(static_cast<float *>(p) + i) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
        uint32_t u[V];
#pragma unroll
        for (int e = 0; e < V; e++)
            u[e] = DT == ORTH_DT_F16 ? (uint32_t)__builtin_bit_cast(uint16_t, (f16)v[e]) : (uint32_t)f32_to_bf16_bits(v[e]);
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(p) + i) = uint2{u[0] | (u[1] << 16), u[2] | (u[3] << 16)};
    }
}

// h + 1e-6 in h's dtype: in LDS for every column (HL), else of column k from
// memory.
template <bool HL>
__device__ __forceinline__ float sieve_h(const SieveArgs &a, const float *hs, int64_t k) {
    if constexpr (HL) return hs[k];
    else return round_as(a.hdt, load_as_f32(a.h, a.hdt, k * a.h_stride) + 1e-6f);
}

template <bool HL>
__device__ __forceinline__ void sieve_stage_h(const SieveArgs &a, float *hs) {
    if constexpr (HL)
        for (int64_t k = threadIdx.x; k < a.K; k += kSvNT)
            hs[k] = round_as(a.hdt, load_as_f32(a.h, a.hdt, k * a.h_stride) + 1e-6f);
}

// The residual and the score of an element, as the torch ops round them
// (S32: the score's dtype is FP32; else one of the two others, by a select).
template <int DT, bool S32>
__device__ __forceinline__ float sieve_score(float wv, float wb, float hs, bool s16, float &resid) {
    resid = round_as(DT, wv - wb);
    const float sc = round_as(DT, sieve_mul(resid, resid)) / hs;
    if constexpr (S32) return sc;
    const float f = (float)(f16)sc, b = bf16_bits_to_f32(f32_to_bf16_bits(sc));
    return s16 ? f : b;
}

// Rows blockIdx.x, + gridDim.x, ...: max|w|, w_base, and with a score buffer
// the scores, their top 11 key bits counted when a rank is selected.  V
// elements per load (4: aligned rows).  A row's first kSvCache vectors per
// thread stay in registers between the two sweeps.
// (4 waves per SIMD: two workgroups a CU, one's loads beside the other's
// divisions)
template <int DT, int V, bool HL, bool S32>
__global__ void __launch_bounds__(kSvNT) __attribute__((amdgpu_waves_per_eu(4))) sieve_quant_kernel(SieveArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    float *hs = reinterpret_cast<float *>(smem);
    uint32_t *hist = reinterpret_cast<uint32_t *>(smem + (HL ? a.K * 4 : 0));
    __shared__ float red[2][kSvNT / 64];
    const int tid = threadIdx.x;
    const bool count = a.score && a.sel, s16 = a.score_dt == ORTH_DT_F16;  // (uniform)
    if (a.score) sieve_stage_h<HL>(a, hs);
    if (count)
        for (int i = tid; i < kSvLanes * kSelBins; i += kSvNT) hist[i] = 0u;
    __syncthreads();
    uint32_t *mine = hist + (tid & (kSvLanes - 1)) * kSelBins;
    int par = 0;
    for (int64_t r = blockIdx.x; r < a.N; r += gridDim.x, par ^= 1) {
        const int64_t base = r * a.K;
        float w[kSvCache][V];
        float m = 0.f;
        for (int64_t b0 = 0; b0 < a.K; b0 += (int64_t)kSvCache * kSvNT * V) {
            // (vectors past the end: the row's last one again, which changes no
            // maximum; where a whole sweep's lie there, not read at all)
            auto sweep = [&](auto whole) {
                float t[kSvCache][V];
#pragma unroll
                for (int j = 0; j < kSvCache; j++) {
                    if (!decltype(whole)::value && b0 + (int64_t)j * kSvNT * V >= a.K) break;  // (uniform)
                    sieve_load<DT, V>(a.w, base + min(b0 + ((int64_t)j * kSvNT + tid) * V, a.K - V), t[j]);
                }
#pragma unroll
                for (int j = 0; j < kSvCache; j++) {
                    if (!decltype(whole)::value && b0 + (int64_t)j * kSvNT * V >= a.K) break;
#pragma unroll
                    for (int e = 0; e < V; e++) {
                        m = sieve_max_nan(m, fabsf(t[j][e]));
                        if (b0 == 0) w[j][e] = t[j][e];
                    }
                }
            };
            if (b0 + (int64_t)(kSvCache - 1) * kSvNT * V < a.K) sweep(std::true_type{});
            else sweep(std::false_type{});
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = sieve_max_nan(m, __shfl_xor(m, off, 64));
        if ((tid & 63) == 0) red[par][tid >> 6] = m;
        __syncthreads();  // (the other copy is written next, after every wave has read this one)
        m = red[par][0];
#pragma unroll
        for (int i = 1; i < kSvNT / 64; i++) m = sieve_max_nan(m, red[par][i]);
        // clamp(min=1e-8): the bound in w's dtype (0 in FP16), NaN kept
        const float lo = round_as(DT, 1e-8f);
        const float mc = (m != m) ? m : fmaxf(m, lo);
        const float s = round_as(DT, sieve_scalar_div(mc, 7.0f, a.ieee_div));
        for (int64_t b0 = 0; b0 < a.K; b0 += (int64_t)kSvCache * kSvNT * V) {
#pragma unroll
            for (int j = 0; j < kSvCache; j++) {
                const int64_t k = b0 + ((int64_t)j * kSvNT + tid) * V;
                if (k >= a.K) continue;
                if (b0 > 0) sieve_load<DT, V>(a.w, base + k, w[j]);
                float wb[V], sc[V];
#pragma unroll
                for (int e = 0; e < V; e++) {
                    float t = rintf(round_as(DT, w[j][e] / s));
                    t = (t != t) ? t : fminf(fmaxf(t, -8.f), 7.f);
                    wb[e] = round_as(DT, sieve_mul(t, s));
                    if (!__builtin_isfinite(wb[e])) wb[e] = 0.f;
                }
                sieve_store<DT, V>(a.w_base, base + k, wb);
                if (a.score) {
                    float rr[V];
#pragma unroll
                    for (int e = 0; e < V; e++) {
                        sc[e] = sieve_score<DT, S32>(w[j][e], wb[e], sieve_h<HL>(a, hs, k + e), s16, rr[e]);
                        if (count) atomicAdd(&mine[sieve_key(sc[e]) >> 21], 1u);
                    }
                    if (a.keep) sieve_store<DT, V>(a.w_ortho, base + k, rr);
                    sieve_store<ORTH_DT_F32, V>(a.score, base + k, sc);
                }
                __builtin_amdgcn_sched_barrier(0);  // one vector's divisions at a time: registers
            }
        }
    }
    if (count) {
        __syncthreads();
        for (int i = tid; i < kSelBins; i += kSvNT) {
            uint32_t c = 0;
#pragma unroll
            for (int l = 0; l < kSvLanes; l++) c += hist[l * kSelBins + i];
            if (c) atomicAdd(&a.sel->hist[0][blockIdx.x % kSelCopies][i], c);
        }
    }
}

// Workgroup b takes scores [b seg, b seg + seg): counts the next 11 key bits
// of those of the found prefix and lists their keys in its part of `list`
// (cap keys; more: the last pass reads the scores again).
template <int V>
__global__ void __launch_bounds__(kSvNT) sieve_collect_kernel(const float *score, int64_t n, int64_t seg,
                                                              SieveSel *st, uint32_t rank, uint32_t *list,
                                                              int64_t cap) {
    __shared__ uint32_t h[kSelBins];
    __shared__ int32_t cnt;
    const int tid = threadIdx.x, lane = tid & 63;
    for (int i = tid; i < kSelBins; i += kSvNT) h[i] = 0u;
    if (tid == 0) cnt = 0;
    uint32_t bin, left;
    sieve_pick(st, 0, rank, bin, left);
    const int64_t i0 = (int64_t)blockIdx.x * seg, i1 = min(n, i0 + seg);
    uint32_t *out = list + (int64_t)blockIdx.x * cap;
    constexpr int U = 4;
    for (int64_t ib = i0 + (int64_t)tid * V; ib < i1; ib += (int64_t)U * kSvNT * V) {
        float v[U][V];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = ib + (int64_t)u * kSvNT * V;
            if (i < i1) sieve_load<ORTH_DT_F32, V>(score, i, v[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (ib + (int64_t)u * kSvNT * V >= i1) continue;
#pragma unroll
            for (int e = 0; e < V; e++) {
                const uint32_t key = sieve_key(v[u][e]);
                if ((key >> 21) == bin) {
                    atomicAdd(&h[(key >> 10) & (kSelBins - 1)], 1u);
                    const int32_t at = atomicAdd(&cnt, 1);
                    if (at < cap) out[at] = key;
                }
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < kSelBins; i += kSvNT)
        if (h[i]) atomicAdd(&st->hist[1][blockIdx.x % kSelCopies][i], h[i]);
    if (tid == 0) st->count[blockIdx.x] = cnt <= cap ? cnt : -1;
}

// The last 10 key bits of the scores that share the 22 found.
__global__ void __launch_bounds__(kSvNT) sieve_refine_kernel(const float *score, int64_t n, int64_t seg, SieveSel *st,
                                                             const uint32_t *list, int64_t cap) {
    __shared__ uint32_t h[1024];
    const int tid = threadIdx.x;
    for (int i = tid; i < 1024; i += kSvNT) h[i] = 0u;
    uint32_t bin, left;
    sieve_pick(st, 1, st->left[0], bin, left);
    const uint32_t prefix = (st->bin[0] << 11) | bin;
    const int32_t cnt = st->count[blockIdx.x];
    if (cnt >= 0) {
        const uint32_t *in = list + (int64_t)blockIdx.x * cap;
        for (int i = tid; i < cnt; i += kSvNT) {
            const uint32_t key = in[i];
            if ((key >> 10) == prefix) atomicAdd(&h[key & 1023u], 1u);
        }
    } else {
        const int64_t i0 = (int64_t)blockIdx.x * seg, i1 = min(n, i0 + seg);
        for (int64_t i = i0 + tid; i < i1; i += kSvNT) {
            const uint32_t key = sieve_key(score[i]);
            if ((key >> 10) == prefix) atomicAdd(&h[key & 1023u], 1u);
        }
    }
    __syncthreads();
    for (int i = tid; i < 1024; i += kSvNT)
        if (h[i]) atomicAdd(&st->hist[2][blockIdx.x % kSelCopies][i], h[i]);
}

// The threshold: the selected k-th largest score, or the caller's rounded to
// the score's dtype (torch compares a tensor with a host scalar in the
// tensor's dtype).
__device__ __forceinline__ float sieve_threshold(const SieveArgs &a) {
    if (!a.sel) return round_as(a.score_dt, a.thresh);
    uint32_t bin, left;
    sieve_pick(a.sel, 2, a.sel->left[1], bin, left);
    return sieve_unkey((a.sel->bin[0] << 21) | (a.sel->bin[1] << 10) | bin);
}

// w_ortho = residual * (score > t); NaN compares false.  Both are formed again
// from w and w_base: the residual is not stored in between.
template <int DT, int V, bool HL, bool S32>
__global__ void __launch_bounds__(kSvNT) __attribute__((amdgpu_waves_per_eu(4))) sieve_mask_kernel(SieveArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    float *hs = reinterpret_cast<float *>(smem);
    const int tid = threadIdx.x;
    sieve_stage_h<HL>(a, hs);
    const bool s16 = a.score_dt == ORTH_DT_F16;
    const float t = sieve_threshold(a);
    __syncthreads();
    for (int64_t r = blockIdx.x; r < a.N; r += gridDim.x) {
        const int64_t base = r * a.K;
        for (int64_t b0 = 0; b0 < a.K; b0 += (int64_t)kSvCache * kSvNT * V) {
            float w[kSvCache][V], wb[kSvCache][V];
#pragma unroll
            for (int j = 0; j < kSvCache; j++) {
                const int64_t k = min(b0 + ((int64_t)j * kSvNT + tid) * V, a.K - V);
                sieve_load<DT, V>(a.w, base + k, w[j]);
                sieve_load<DT, V>(a.w_base, base + k, wb[j]);
            }
#pragma unroll
            for (int j = 0; j < kSvCache; j++) {
                const int64_t k = b0 + ((int64_t)j * kSvNT + tid) * V;
                if (k >= a.K) continue;
                float o[V];
#pragma unroll
                for (int e = 0; e < V; e++) {
                    float rr;
                    const float sc = sieve_score<DT, S32>(w[j][e], wb[j][e], sieve_h<HL>(a, hs, k + e), s16, rr);
                    o[e] = sieve_mul(rr, sc > t ? 1.f : 0.f);
                }
                sieve_store<DT, V>(a.w_ortho, base + k, o);
                __builtin_amdgcn_sched_barrier(0);  // (as above)
            }
        }
    }
}

// The same from the residual stored in w_ortho and the scores (a.keep).
template <int DT, int V>
__global__ void __launch_bounds__(kSvNT) sieve_apply_kernel(SieveArgs a) {
    const float t = sieve_threshold(a);
    const int64_t n = a.N * a.K, step = (int64_t)gridDim.x * kSvNT * V;
    for (int64_t i = ((int64_t)blockIdx.x * kSvNT + threadIdx.x) * V; i < n; i += step) {
        float r[V], sc[V];
        sieve_load<DT, V>(a.w_ortho, i, r);
        sieve_load<ORTH_DT_F32, V>(a.score, i, sc);
#pragma unroll
        for (int e = 0; e < V; e++) r[e] = sieve_mul(r[e], sc[e] > t ? 1.f : 0.f);
        sieve_store<DT, V>(a.w_ortho, i, r);
    }
}

// Column sums of squares of x [n, K] over row slice blockIdx.y (slices of
// `rows` rows), in FP32: partial[y][k].
__global__ void __launch_bounds__(kSieveNT) sieve_hdiag_partial_kernel(const void *x, int dt, int64_t n, int64_t K,
                                                                       int64_t rows, float *partial) {
    const int64_t k = (int64_t)blockIdx.x * kSieveNT + threadIdx.x;
    if (k >= K) return;
    const int64_t r0 = (int64_t)blockIdx.y * rows, r1 = min(n, r0 + rows);
    float s = 0.f;
    for (int64_t r = r0; r < r1; r++) {
        const float v = load_as_f32(x, dt, r * K + k);
        s = __builtin_fmaf(v, v, s);
    }
    partial[(int64_t)blockIdx.y * K + k] = s;
}

// diag / n + 1e-6 with torch's steps: the diagonal rounded to x's dtype,
// divided by n (a host scalar: times its FP32 reciprocal, or IEEE division
// in the ieee_div mode), rounded, plus 1e-6, rounded.
__global__ void __launch_bounds__(kSieveNT) sieve_hdiag_final_kernel(const float *partial, int slices, int64_t n,
                                                                     int64_t K, int dt, void *out, int ieee_div) {
    const int64_t k = (int64_t)blockIdx.x * kSieveNT + threadIdx.x;
    if (k >= K) return;
    float s = 0.f;
    for (int i = 0; i < slices; i++) s += partial[(int64_t)i * K + k];
    const float d = round_as(dt, s);
    const float q = round_as(dt, sieve_scalar_div(d, (float)n, ieee_div));
    store_from_f32(out, dt, k, round_as(dt, q + 1e-6f));
}

// 4 elements per load where every row of the four arrays starts aligned.
static bool sieve_vec(const SieveArgs &a, int dt) {
    const int64_t al = dt == ORTH_DT_F32 ? 16 : 8;
    const uintptr_t p = reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.w_base) |
                        reinterpret_cast<uintptr_t>(a.w_ortho);
    return a.K % 4 == 0 && p % al == 0 && reinterpret_cast<uintptr_t>(a.score) % 16 == 0;
}

template <int DT, int V, bool HL, bool S32>
static hipError_t sieve_launch_t(const SieveArgs &a, hipStream_t stream) {
    const int64_t n = a.N * a.K;
    const unsigned rows = (unsigned)(a.N < kSelWgs ? a.N : kSelWgs);
    const uint32_t hb = HL ? (uint32_t)a.K * 4 : 0;
    // more than 64 KB of dynamic LDS must be allowed once per device (the
    // attribute call is idempotent, so two threads racing to set it is harmless)
    static std::atomic<int> allowed[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && !allowed[dev].load(std::memory_order_acquire)) {
        const int most = kSvLdsCols * 4 + kSvLanes * kSelBins * 4;
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(sieve_quant_kernel<DT, V, HL, S32>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, most);
        if (e == hipSuccess)
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(sieve_mask_kernel<DT, V, HL, S32>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, most);
        if (e != hipSuccess) return e;
        allowed[dev].store(1, std::memory_order_release);
    }
    if (a.sel)
        hipLaunchKernelGGL(sieve_sel_init_kernel, dim3(3 * kSelCopies * kSelBins / 256), dim3(256), 0, stream, a.sel);
    hipLaunchKernelGGL((sieve_quant_kernel<DT, V, HL, S32>), dim3(rows), dim3(kSvNT),
                       hb + (a.sel ? kSvLanes * kSelBins * 4 : 0), stream, a);
    if (!a.w_ortho) return hipGetLastError();
    if (a.sel) {
        // segments of whole vectors; their keys' list is the w_ortho buffer,
        // which the last pass overwrites (none where it holds the residual)
        const int64_t seg = ((n + kSelWgs - 1) / kSelWgs + 3) & ~int64_t(3);
        const unsigned wgs = (unsigned)((n + seg - 1) / seg);
        uint32_t *list = static_cast<uint32_t *>(a.w_ortho);
        const int64_t cap = !a.keep && reinterpret_cast<uintptr_t>(a.w_ortho) % 4 == 0
                                ? n * (DT == ORTH_DT_F32 ? 4 : 2) / 4 / kSelWgs : 0;
        if (n % 4 == 0 && reinterpret_cast<uintptr_t>(a.score) % 16 == 0)
            hipLaunchKernelGGL((sieve_collect_kernel<4>), dim3(wgs), dim3(kSvNT), 0, stream, a.score, n, seg, a.sel,
                               a.rank, list, cap);
        else
            hipLaunchKernelGGL((sieve_collect_kernel<1>), dim3(wgs), dim3(kSvNT), 0, stream, a.score, n, seg, a.sel,
                               a.rank, list, cap);
        hipLaunchKernelGGL(sieve_refine_kernel, dim3(wgs), dim3(kSvNT), 0, stream, a.score, n, seg, a.sel, list, cap);
    }
    if (a.keep) {
        const int64_t wgs = (n + (int64_t)kSvNT * V - 1) / ((int64_t)kSvNT * V);
        hipLaunchKernelGGL((sieve_apply_kernel<DT, V>), dim3((unsigned)(wgs < 4096 ? wgs : 4096)), dim3(kSvNT), 0,
                           stream, a);
    } else {
        hipLaunchKernelGGL((sieve_mask_kernel<DT, V, HL, S32>), dim3(rows), dim3(kSvNT), hb, stream, a);
    }
    return hipGetLastError();
}

// Whether two of the four buffers of a split share memory.
static bool sieve_overlap(const SieveArgs &a, int dt) {
    const int64_t n = a.N * a.K, e = dt == ORTH_DT_F32 ? 4 : 2;
    const void *p[4] = {a.w, a.w_base, a.w_ortho, a.score};
    const int64_t bytes[4] = {n * e, n * e, n * e, n * 4};
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < i; j++) {
            const char *b0 = static_cast<const char *>(p[i]), *b1 = static_cast<const char *>(p[j]);
            if (b0 < b1 + bytes[j] && b1 < b0 + bytes[i]) return true;
        }
    return false;
}

template <int DT, bool S32>
static hipError_t sieve_launch_s(const SieveArgs &a, hipStream_t stream) {
    if (a.K > kSvLdsCols) return sieve_launch_t<DT, 1, false, S32>(a, stream);
    return sieve_vec(a, DT) ? sieve_launch_t<DT, 4, true, S32>(a, stream) : sieve_launch_t<DT, 1, true, S32>(a, stream);
}

template <int DT>
static hipError_t sieve_launch_d(const SieveArgs &a, hipStream_t stream) {
    return a.score_dt == ORTH_DT_F32 ? sieve_launch_s<DT, true>(a, stream) : sieve_launch_s<DT, false>(a, stream);
}

static hipError_t sieve_launch(const SieveArgs &a, int dt, hipStream_t stream) {
    if (dt == ORTH_DT_F32) return sieve_launch_d<ORTH_DT_F32>(a, stream);
    if (dt == ORTH_DT_F16) return sieve_launch_d<ORTH_DT_F16>(a, stream);
    return sieve_launch_d<ORTH_DT_BF16>(a, stream);
}

hipError_t launch_sieve_quantize(const void *w, int dt, int64_t N, int64_t K, void *w_base, int ieee_div,
                                 hipStream_t stream) {
    SieveArgs a{};
    a.ieee_div = ieee_div;
    a.w = w;
    a.N = N;
    a.K = K;
    a.w_base = w_base;
    a.score_dt = ORTH_DT_F32;  // (no score is formed)
    return sieve_launch(a, dt, stream);
}

hipError_t launch_sieve_split(const void *w, int dt, int64_t N, int64_t K, const void *h, int hdt, int64_t h_stride,
                              int score_dt, int use_rank, int64_t rank, float thresh, void *w_base, void *w_ortho,
                              float *score, void *sel, int ieee_div, hipStream_t stream) {
    SieveArgs a{};
    a.ieee_div = ieee_div;
    a.w = w;
    a.N = N;
    a.K = K;
    a.w_base = w_base;
    a.w_ortho = w_ortho;
    a.score = score;
    a.h = h;
    a.hdt = hdt;
    a.h_stride = h_stride;
    a.score_dt = score_dt;
    a.sel = use_rank && rank > 0 ? static_cast<SieveSel *>(sel) : nullptr;
    a.rank = (uint32_t)rank;
    // rank 0: the reference keeps nothing (threshold max + 1)
    a.thresh = use_rank ? __builtin_nanf("") : thresh;
    // in place (w_base or w_ortho is w): w is read in the first pass only,
    // each element before it is written.  Also with a given threshold and a
    // strided h (a matrix's diagonal: a cache line a column), so that h is
    // gathered once: us, residual formed again / stored, 1024 x 1024 FP32 20.0 /
    // 17.0, 2048 x 20480 561 / 394.
    a.keep = sieve_overlap(a, dt) || (!a.sel && h_stride > 1);
    return sieve_launch(a, dt, stream);
}

int64_t sieve_hdiag_slices(int64_t n) {
    const int64_t s = (n + 255) / 256;
    return s < 64 ? (s > 0 ? s : 1) : 64;
}

hipError_t launch_sieve_hdiag(const void *x, int dt, int64_t n, int64_t K, float *partial, void *out, int ieee_div,
                              hipStream_t stream) {
    const int64_t slices = sieve_hdiag_slices(n);
    const int64_t rows = (n + slices - 1) / slices;
    const unsigned cb = (unsigned)((K + kSieveNT - 1) / kSieveNT);
    hipLaunchKernelGGL(sieve_hdiag_partial_kernel, dim3(cb, (unsigned)slices), dim3(kSieveNT), 0, stream, x, dt, n, K,
                       rows, partial);
    hipLaunchKernelGGL(sieve_hdiag_final_kernel, dim3(cb), dim3(kSieveNT), 0, stream, partial, (int)slices, n, K, dt,
                       out, ieee_div);
    return hipGetLastError();
}

}  // namespace orth
