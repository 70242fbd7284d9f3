// FP32 activations, batches from a few dozen tokens (general_variant): the dual GEMM on the
// matrix cores without giving up an FP32 bit of the activations.
//
// Same formula as /root/reference/src/dual_gemm.cu:176-225, whose
// activations are FP32.  Two launches:
//
//  * float_kernel, the dense term.  An FP32 value is the exact sum of three
//    bfloat16 values (its significand cut in three runs of 8 bits, by
//    truncation, so nothing rounds or overflows), and an INT4 weight / 1024
//    is an exact bfloat16 value, so three v_mfma_f32_16x16x32_bf16 passes form
//    x * q with exact products and FP32 sums; the group scale multiplies the
//    group's FP32 partial.  That is three passes at the bfloat16 matrix rate
//    (2.5 PFLOP/s dense) against one at the FP32 matrix rate (157 TFLOP/s).
//    Tile 64 tokens x 128 rows per workgroup of 8 waves: two K halves of each
//    64-column step x (2 x 2) waves of 32 tokens x 64 rows, so that 512
//    tokens of a 4096-row layer make 256 workgroups; the halves' sums meet in
//    LDS.  x is split and the weights are converted while they are staged
//    (once per tile, not per wave), two stages, loads two steps ahead; the
//    tile's scales are staged once.  What bounds a step is its vector ALU
//    work (the split, the conversion, the scaling: ~150 instructions a wave
//    beside 24 MFMAs): the two K halves, which share each SIMD, therefore
//    take the MFMAs and the staging in opposite order (77 -> 74 us at 512
//    tokens of 4096 -> 4096, alpha = 0, with the byte conversions written
//    out; 1,203 us on the wave-per-row kernel).
//  * float_ortho_kernel, the sparse term (alpha > 0): y += alpha * sum v x.
//    A workgroup keeps all columns of up to 8 tokens in LDS, [column][token],
//    so that an entry costs one 16-byte LDS read per 4 tokens, and walks the
//    CSR of a range of rows, 16 lanes a row, a lane its own entries (two lanes
//    sharing each, with a branch around an empty slot: 28 us against 23 at 512
//    tokens of 4096 -> 4096 at 1 %).  y is FP32, so adding to it in a second
//    launch rounds as adding in registers would.  Bound by its LDS reads (4
//    bytes a product) and vector ALU work.  (Folding the values into the
//    weight tile, as the 16-bit prefill does, would need two more bfloat16
//    parts per weight.)
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "orth_common.h"
#include "orth_general_shape.h"

namespace orth {

constexpr int kFlNT = 512;
constexpr int kFlPlane = kFlBM * kFlBK * 2;           // one bfloat16 part of the activations' stage
constexpr int kFlW = kFlBN * kFlBK * 2;               // the weights' stage
constexpr int kFlStage = 3 * kFlPlane + kFlW;         // 40 KB

struct FloatArgs {
    const uint8_t *q;
    const void *scales;
    int scale_dtype;
    int ngroups;
    int spg;            // 64-column steps per scale group
    const float *x;
    float *y;
    int64_t M, K, N;
    int ntm;            // token tiles
    const void *bias;   // added here when there is no sparse launch
    int bias_dtype;
};

// SPF: steps per flush of the partials into the scaled sums, 1 or 2 (2 needs
// an even number of steps per scale group).
template <int SPF>
__global__ void __launch_bounds__(kFlNT) float_kernel(FloatArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    float *sl = reinterpret_cast<float *>(smem + 2 * kFlStage);  // scales [group][128 rows]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nl = lane & 15, g = lane >> 4;
    const int kh = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const int64_t m0 = (int64_t)(blockIdx.x % (unsigned)a.ntm) * kFlBM;
    const int64_t n0 = (int64_t)(blockIdx.x / (unsigned)a.ntm) * kFlBN;
    const int64_t K = a.K;
    const int nsteps = (int)(K / kFlBK);

    // staging: token tid / 8, columns 8 (tid % 8) ..; row tid / 4, columns 16 (tid % 4) ..
    const int xt = tid >> 3, xc = tid & 7;
    const int wr = tid >> 2, wc = tid & 3;
    const float *xp = a.x + min(m0 + xt, a.M - 1) * K + 8 * xc;
    const uint8_t *wp = a.q + min(n0 + wr, a.N - 1) * (K >> 1) + 8 * wc;
    struct Regs {
        f32x4 xa, xb;
        uint2 w;
    };
    auto load = [&](int t, Regs &r) {
        const int64_t k0 = (int64_t)min(t, nsteps - 1) * kFlBK;
        r.xa = *reinterpret_cast<const f32x4 *>(xp + k0);
        r.xb = *reinterpret_cast<const f32x4 *>(xp + k0 + 4);
        r.w = *reinterpret_cast<const uint2 *>(wp + (k0 >> 1));
    };
    // a stage's rows are 128 bytes, their eight 16-byte chunks XOR-ed by the row
    auto at = [](int row, int chunk) { return row * (kFlBK * 2) + ((chunk ^ (row & 7)) << 4); };
    auto store = [&](int s, const Regs &r) {
        unsigned char *st = smem + s * kFlStage;
        u32x4 p[3];
        split_bf16x3(r.xa, r.xb, p);
#pragma unroll
        for (int i = 0; i < 3; i++) *reinterpret_cast<u32x4 *>(st + i * kFlPlane + at(xt, xc)) = p[i];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t o[4];
            int4x8_to_bf16_exact(h ? r.w.y : r.w.x, o);
            *reinterpret_cast<u32x4 *>(st + 3 * kFlPlane + at(wr, 2 * wc + h)) = u32x4{o[0], o[1], o[2], o[3]};
        }
    };

    Regs r0, r1;
    load(0, r0);
    load(1, r1);
    // the weights' divisor goes into the scales, or (FP32 scales too large for
    // that somewhere in the tile) multiplies the finished sums
    auto scales = [&](float f) -> int {
        int over = 0;
        for (int i = tid; i < kFlBN * a.ngroups; i += kFlNT) {
            const int row = i / a.ngroups, gi = i - row * a.ngroups;
            const float v = load_as_f32(a.scales, a.scale_dtype, min(n0 + row, a.N - 1) * a.ngroups + gi);
            sl[gi * kFlBN + row] = f * v;
            over |= !__builtin_isfinite(f * v) && __builtin_isfinite(v) ? 1 : 0;
        }
        return over;
    };
    const int over = scales(kBf16Q);
    store(0, r0);
    load(2, r0);
    const bool late = __syncthreads_or(over) != 0;  // (uniform)
    if (late) {
        scales(1.0f);
        __syncthreads();
    }

    f32x4 acc[2][4], part[2][4];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    int in_group = 0, grp = 0;
    auto flush = [&]() {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float s = sl[grp * kFlBN + wn * 64 + 16 * j + nl];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][j][i] = __builtin_fmaf(s, part[t][j][i], acc[t][j][i]);
        }
        in_group += SPF;
        const bool last = in_group == a.spg;  // (uniform)
        grp += last ? 1 : 0;
        in_group = last ? 0 : in_group;
    };
    // stage s; FIRST: the partials start here, FLUSH: and are flushed here
    auto compute = [&](int s, auto first_c, auto flush_c) {
        constexpr bool FIRST = decltype(first_c)::value, FLUSH = decltype(flush_c)::value;
        const unsigned char *st = smem + s * kFlStage;
        bf16x8 bw[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            bw[j] = *reinterpret_cast<const bf16x8 *>(st + 3 * kFlPlane + at(wn * 64 + 16 * j + nl, 4 * kh + g));
#pragma unroll
        for (int i = 2; i >= 0; i--) {  // the smallest parts first
            bf16x8 av[2];
#pragma unroll
            for (int t = 0; t < 2; t++)
                av[t] = *reinterpret_cast<const bf16x8 *>(st + i * kFlPlane + at(wm * 32 + 16 * t + nl, 4 * kh + g));
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    part[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t], bw[j],
                                                                         FIRST && i == 2 ? zero : part[t][j], 0, 0, 0);
        }
        if (FLUSH) flush();
    };
    constexpr auto kYes = std::integral_constant<bool, true>{};
    constexpr auto kFirst1 = std::integral_constant<bool, SPF == 1>{};
    // step t: the MFMAs of its stage, and the next step's data into the other
    // stage (last read before the previous barrier), its loads three steps
    // ahead.  The two K halves, which share each SIMD, do the two in opposite
    // order, so that one's MFMAs run beside the other's conversion.  (Two
    // loops, not a branch around the loads, which would make every wait a
    // full one; each wave meets one barrier a step.)
    auto barrier = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    int t = 0;
    if (kh == 0) {
        for (; t + 1 < nsteps; t += 2) {
            compute(0, kYes, kFirst1);
            __builtin_amdgcn_sched_barrier(0);
            store(1, r1);
            load(t + 3, r1);
            barrier();
            compute(1, kFirst1, kYes);
            __builtin_amdgcn_sched_barrier(0);
            store(0, r0);
            load(t + 4, r0);
            barrier();
        }
    } else {
        for (; t + 1 < nsteps; t += 2) {
            store(1, r1);
            load(t + 3, r1);
            __builtin_amdgcn_sched_barrier(0);
            compute(0, kYes, kFirst1);
            barrier();
            store(0, r0);
            load(t + 4, r0);
            __builtin_amdgcn_sched_barrier(0);
            compute(1, kFirst1, kYes);
            barrier();
        }
    }
    if (t < nsteps) compute(0, kYes, kYes);

    // the two K halves meet in LDS: half 1 hands its sums to half 0
    __syncthreads();
    float *red = reinterpret_cast<float *>(smem);  // [4 waves][8 tiles][64 lanes][4]
    f32x4 *mine = reinterpret_cast<f32x4 *>(red) + (wave & 3) * 8 * 64 + lane;
    if (kh == 1) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < 4; j++) mine[(u * 4 + j) * 64] = acc[u][j];
    }
    __syncthreads();
    if (kh == 1) return;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t n = n0 + wn * 64 + 16 * j + nl;
        if (n >= a.N) continue;
        const float b = a.bias ? load_as_f32(a.bias, a.bias_dtype, n) : 0.f;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const f32x4 v = (acc[u][j] + mine[(u * 4 + j) * 64]) * (late ? kBf16Q : 1.0f);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t m = m0 + wm * 32 + 16 * u + 4 * g + i;
                if (m < a.M) a.y[m * a.N + n] = a.bias ? v[i] + b : v[i];
            }
        }
    }
}

// ------------------------------------------------------------- sparse term

struct FloatOrthoArgs {
    const int32_t *row_ptr;
    const int32_t *col;
    const void *vals;
    int64_t nnz;
    const float *x;
    float *y;
    int64_t M, K, N;
    float alpha;
    int ntm;            // token tiles
    int wgs;            // workgroups per token tile
    const void *bias;
    int bias_dtype;
};

// TT tokens per workgroup (8, 4, 2 or 1); VH: FP16 values, else FP32.
// Every wave takes units of 16 rows (no barrier after the staging, so the
// waves' CSR loads overlap): four passes of 4 rows, 16 lanes a row, the first
// U batches of entries of all four loaded before the first is used.
template <int TT, bool VH>
__global__ void __launch_bounds__(kFoNT) float_ortho_kernel(FloatOrthoArgs a) {
    constexpr int U = 3;                 // batches of 16 entries of a row in flight
    constexpr int PL = (TT * kFoRows + 63) / 64;  // outputs per lane of a unit
    extern __shared__ __align__(16) unsigned char smem[];
    float *xs = reinterpret_cast<float *>(smem);          // [K + 1][TT], the last column zero (for empty entries)

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    float *sums = xs + (a.K + 1) * TT + wave * (TT * kFoRows);  // the wave's [TT][16]
    if (tid < TT) xs[a.K * TT + tid] = 0.f;
    const int64_t m0 = (int64_t)(blockIdx.x % (unsigned)a.ntm) * TT;
    const int wg = (int)(blockIdx.x / (unsigned)a.ntm);

    // columns k, k + 1024 per round, every token's loads issued together
    for (int64_t k = tid; k < a.K; k += 2 * kFoNT) {
        const int64_t k2 = min(k + kFoNT, a.K - 1);
        float v[2][TT];
#pragma unroll
        for (int t = 0; t < TT; t++) {
            const float *xp = a.x + min(m0 + t, a.M - 1) * a.K;
            v[0][t] = xp[k];
            v[1][t] = xp[k2];
        }
#pragma unroll
        for (int t = 0; t < TT; t++) xs[k * TT + t] = v[0][t];
        if (k + kFoNT < a.K) {
#pragma unroll
            for (int t = 0; t < TT; t++) xs[k2 * TT + t] = v[1][t];
        }
    }
    __syncthreads();

    auto value = [&](int32_t j) -> float {
        if constexpr (VH) return (float)static_cast<const f16 *>(a.vals)[j];
        else return static_cast<const float *>(a.vals)[j];
    };
    const int sub = lane >> 4, l16 = lane & 15;           // row of a pass, lane of the row
    const int64_t units = (a.N + kFoRows - 1) / kFoRows;
    for (int64_t un = (int64_t)wg * kFoW + wave; un < units; un += (int64_t)a.wgs * kFoW) {
        const int64_t r0 = un * kFoRows;
        // the unit's outputs so far: lane's tokens lane / 16 + 4 i, row l16
        float old[PL];
#pragma unroll
        for (int i = 0; i < PL; i++)
            old[i] = a.y[min(m0 + min(sub + 4 * i, TT - 1), a.M - 1) * a.N + min(r0 + l16, a.N - 1)];
        const int32_t rp = a.row_ptr[min(r0 + min(lane, 16), a.N)];
        int32_t js[4], je[4], c[4][U];
        float v[4][U];
#pragma unroll
        for (int p = 0; p < 4; p++) {  // (clamped as csr_row_range does)
            const int32_t nnz = (int32_t)a.nnz;
            js[p] = min(max(__shfl(rp, 4 * p + sub), 0), nnz);
            je[p] = min(max(__shfl(rp, 4 * p + sub + 1), js[p]), nnz);
            if (r0 + 4 * p + sub >= a.N) je[p] = js[p];
        }
        // batch u of a row at jb: lane l16 loads entry jb + 16 u + l16, clamped (nnz > 0)
        auto load = [&](int p, int32_t jb, int32_t (&cc)[U], float (&vv)[U]) {
            const int32_t last = (int32_t)min((int64_t)max(je[p] - 1, 0), a.nnz - 1);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int32_t ju = min(jb + 16 * u + l16, last);
                cc[u] = a.col[ju];
                vv[u] = value(ju);
            }
        };
#pragma unroll
        for (int p = 0; p < 4; p++) load(p, js[p], c[p], v[p]);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            float acc[TT];
#pragma unroll
            for (int t = 0; t < TT; t++) acc[t] = 0.f;
            // a lane takes its own entries, all tokens of each
            auto use = [&](int32_t jb, const int32_t (&cc)[U], const float (&vv)[U]) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const bool ok = jb + 16 * u + l16 < je[p] && cc[u] >= 0 && cc[u] < a.K;
                    if (u > 0 && !__any(ok)) continue;  // (uniform)
                    const float val = ok ? vv[u] : 0.f;
                    const float *xc = xs + (ok ? (int64_t)cc[u] : a.K) * TT;
                    float x[TT];
                    if constexpr (TT >= 4) {
#pragma unroll
                        for (int i = 0; i < TT / 4; i++) {
                            const f32x4 q = reinterpret_cast<const f32x4 *>(xc)[i];
#pragma unroll
                            for (int e = 0; e < 4; e++) x[4 * i + e] = q[e];
                        }
                    } else {
#pragma unroll
                        for (int t = 0; t < TT; t++) x[t] = xc[t];
                    }
#pragma unroll
                    for (int t = 0; t < TT; t++) acc[t] = __builtin_fmaf(val, x[t], acc[t]);
                }
            };
            use(js[p], c[p], v[p]);
            for (int32_t jb = js[p] + 16 * U; jb < je[p]; jb += 16 * U) {
                int32_t c2[U];
                float v2[U];
                load(p, jb, c2, v2);
                use(jb, c2, v2);
            }
            // sums over the row's 16 lanes, halving the tokens a lane keeps as
            // it goes (partners: lane ^ 8, 7 - lane of each 8, lane ^ 2, lane ^ 1)
            auto fold = [&](auto ctrl_c, int bit, auto n_c) {
                constexpr int CTRL = decltype(ctrl_c)::value, NV = decltype(n_c)::value;  // NV values: halve, 0: keep all
                if constexpr (NV > 0) {
#pragma unroll
                    for (int t = 0; t < NV / 2; t++) {
                        const float keep = (l16 & bit) ? acc[t + NV / 2] : acc[t], give = (l16 & bit) ? acc[t] : acc[t + NV / 2];
                        acc[t] = keep + dpp_f32<CTRL>(give);
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < TT; t++) acc[t] += dpp_f32<CTRL>(acc[t]);
                }
            };
            fold(std::integral_constant<int, 0x128>{}, 8, std::integral_constant<int, TT == 8 ? 8 : 0>{});
            fold(std::integral_constant<int, 0x141>{}, 4, std::integral_constant<int, TT >= 4 ? 4 : 0>{});
            fold(std::integral_constant<int, 0x4E>{}, 2, std::integral_constant<int, TT >= 2 ? 2 : 0>{});
            const float one = acc[0] + dpp_f32<0xB1>(acc[0]);
            const int tok = (TT == 8 ? (l16 >> 3) * 4 : 0) + (TT >= 4 ? ((l16 >> 2) & 1) * 2 : 0) + (TT >= 2 ? (l16 >> 1) & 1 : 0);
            // (the lanes of one token hold the same bits: partners add the same two values)
            if ((l16 & 1) == 0) sums[tok * kFoRows + 4 * p + sub] = one;
        }
        __builtin_amdgcn_wave_barrier();  // (same wave: LDS keeps the order)
        const int64_t n = r0 + l16;
#pragma unroll
        for (int i = 0; i < PL; i++) {
            const int t = sub + 4 * i;
            if (t < TT && m0 + t < a.M && n < a.N) {
                float o = old[i] + a.alpha * sums[t * kFoRows + l16];
                if (a.bias) o += load_as_f32(a.bias, a.bias_dtype, n);
                a.y[(m0 + t) * a.N + n] = o;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------ host

// More than 64 KB of dynamic LDS must be allowed once per device and kernel
// (the attribute call is idempotent, so two threads racing is harmless).
static hipError_t float_allow_lds(const void *fn, int bytes, std::atomic<int> *allowed) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64 || allowed[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) allowed[dev].store(1, std::memory_order_release);
    return e;
}

template <int SPF>
static hipError_t launch_float_dense(const FloatArgs &d, int64_t N, hipStream_t stream) {
    static std::atomic<int> allowed[64];
    hipError_t e = float_allow_lds(reinterpret_cast<const void *>(float_kernel<SPF>), 2 * kFlStage + kFlMaxGroups * kFlBN * 4, allowed);
    if (e != hipSuccess) return e;
    const uint32_t lds = 2 * kFlStage + (uint32_t)d.ngroups * kFlBN * 4;
    const unsigned blocks = (unsigned)(d.ntm * ((N + kFlBN - 1) / kFlBN));
    hipLaunchKernelGGL((float_kernel<SPF>), dim3(blocks), dim3(kFlNT), lds, stream, d);
    return hipGetLastError();
}

template <int TT, bool VH>
static hipError_t launch_float_ortho(FloatOrthoArgs o, int cus, hipStream_t stream) {
    static std::atomic<int> allowed[64];
    hipError_t e = float_allow_lds(reinterpret_cast<const void *>(float_ortho_kernel<TT, VH>), (int)kFoLdsMax, allowed);
    if (e != hipSuccess) return e;
    const int64_t ntm = (o.M + TT - 1) / TT;
    o.ntm = (int)ntm;
    o.wgs = (int)float_ortho_wgs(o.N, ntm, cus);
    const uint32_t lds = (uint32_t)((o.K + 1 + kFoRows * kFoW) * TT * 4);
    hipLaunchKernelGGL((float_ortho_kernel<TT, VH>), dim3((unsigned)(ntm * o.wgs)), dim3(kFoNT), lds, stream, o);
    return hipGetLastError();
}

template <bool VH>
static hipError_t launch_float_ortho_v(const FloatOrthoArgs &o, int cus, hipStream_t stream) {
    const int tt = float_ortho_tile(o.K, o.M);
    if (tt == 8) return launch_float_ortho<8, VH>(o, cus, stream);
    if (tt == 4) return launch_float_ortho<4, VH>(o, cus, stream);
    if (tt == 2) return launch_float_ortho<2, VH>(o, cus, stream);
    return launch_float_ortho<1, VH>(o, cus, stream);
}

hipError_t launch_float(const ForwardArgs &a, int cus, hipStream_t stream) {
    FloatArgs d;
    d.q = a.q;
    d.scales = a.scales;
    d.scale_dtype = a.scale_dtype;
    d.ngroups = (int)a.ngroups;
    d.spg = (int)(a.G / kFlBK);
    d.x = static_cast<const float *>(a.x);
    d.y = static_cast<float *>(a.y);
    d.M = a.M;
    d.K = a.K;
    d.N = a.N;
    d.ntm = (int)((a.M + kFlBM - 1) / kFlBM);
    d.bias = a.has_ortho ? nullptr : a.bias;
    d.bias_dtype = a.bias_dtype;
    // The partials are summed into the scaled sums every two steps, also
    // inside a longer group: one chain over all of K would lose more than the
    // wave-per-row kernel's lanes do (4096 columns, one scale per row: relative
    // error against FP64 4.2e-7; flushed every two steps 1.3e-7, those
    // lanes 1.6e-7).
    hipError_t e = d.spg % 2 ? launch_float_dense<1>(d, a.N, stream) : launch_float_dense<2>(d, a.N, stream);
    if (e != hipSuccess || !a.has_ortho) return e;
    FloatOrthoArgs o;
    o.row_ptr = a.row_ptr;
    o.col = a.col;
    o.vals = a.vals;
    o.nnz = a.nnz;
    o.x = d.x;
    o.y = d.y;
    o.M = a.M;
    o.K = a.K;
    o.N = a.N;
    o.alpha = a.alpha;
    o.bias = a.bias;
    o.bias_dtype = a.bias_dtype;
    return a.val_dtype == ORTH_DT_F16 ? launch_float_ortho_v<true>(o, cus, stream)
                                      : launch_float_ortho_v<false>(o, cus, stream);
}

}  // namespace orth
