// The dual GEMM for the layouts the other kernels do not take: FP32
// activations in small batches, in_features that no 128-column chunk divides,
// scale groups of 32, 64, 96, ... columns.
//
// Same formula as /root/reference/src/dual_gemm.cu:176-225.  A wave of the
// wave-per-row kernel owns one output row and reads every activation for it (4
// tokens of 4096 FP32 columns: 64 KB a row, 268 MB over a 4096-row layer); here
// a workgroup stages the activations of up to 16 tokens in LDS once and takes
// RB blocks of 16 rows per pass, and the products run on the matrix cores:
//
//  * 8 waves, each a run of the 128-column chunks (K is padded to whole chunks
//    with zero activations, against which a weight read past the row's end
//    counts nothing).  A lane holds 32 weights of its row per chunk: one
//    16-byte load (WIDE), or four words 16 columns apart so that each MFMA
//    covers 32 consecutive columns and takes its own group's scale (groups
//    that are multiples of 32, rows of any multiple of 4 bytes).  Four chunks
//    of loads are in flight, issued before the staging waits for its own.
//  * The weights become exact FP16 integers or bfloat16 q / 1024; FP32 activations
//    are cut into three bfloat16 parts without rounding (split_bf16x3), so
//    every product is exact and every sum FP32; the scale multiplies a
//    chunk's (or 32 columns') partial.
//  * Sparse term: each wave takes 2 RB rows; a row's entries are loaded 64 at
//    a time, one per lane, before the staging's barrier, with the place of the
//    activation in a staged row (empty slots: a zero past its end), and handed
//    to the lanes (entry, token) in turn, which gather there.  This follows
//    the dense term, whose weights were asked for first: 4000 -> 11008, 16
//    FP16 tokens at 1 %, weights in cache, 21.7 -> 18.9 us against taking it first with a test
//    per entry; the dense term alone 12.2.
//  * The waves' partials meet in LDS (deterministic) and are rounded once.
//
// What bounds it: the latency chain (staging, the weights' first bytes, the
// reduction) at few tokens, the LDS reads of the sparse term at 16 (4000 ->
// 11008, 16 FP16 tokens at 1 %, weights from HBM: 149.8 us on the wave-per-row
// kernel, 21.8 here; 1 token 26.3 and 18.4).
#include <algorithm>
#include <atomic>

#include "orth_common.h"
#include "orth_general_shape.h"

namespace orth {

constexpr int kRwNT = 64 * kRwW;
constexpr int kRwD = 4;            // chunks of weights in flight
constexpr int kRwXB = 8;           // 16-byte activation loads in flight per thread

struct RowsArgs {
    const uint8_t *q;
    const f16 *scales;
    int ngroups;
    int g32;             // 32-column runs per scale group
    const int32_t *row_ptr;
    const int32_t *col;
    const f16 *vals;
    int32_t nnz;
    int sparse;
    float alpha;
    const void *x;
    void *y;
    int64_t M, N;
    int K;
    int nch;             // chunks, the last one padded
    int cpw;             // chunks per wave
    int mt;              // tokens per workgroup
    int tl;              // lanes per entry in the sparse term: a power of two >= mt
    int npass;           // RB-block passes over the rows
    const void *bias;
    int bias_dtype;
};

// IO: the activations' type.  RB: 16-row blocks per pass.  WIDE: see above.
template <int IO, int RB, bool WIDE>
__global__ void __launch_bounds__(kRwNT) rows_kernel(RowsArgs a) {
    constexpr bool F32 = IO == ORTH_DT_F32, F16 = IO == ORTH_DT_F16;
    constexpr int NP = F32 ? 3 : 1;            // parts of an activation
    constexpr int EV = F32 ? 4 : 8;            // activations per 16 bytes
    constexpr int NS = WIDE ? 1 : 4;           // scales per chunk and row
    constexpr int NR = 2 * RB;                 // rows per wave in the sparse term
    typedef typename std::conditional<F32, float, uint16_t>::type X;

    extern __shared__ __align__(16) unsigned char smem[];
    const int xst = a.nch * 128 + EV;          // token stride of the staged activations
    X *xs = reinterpret_cast<X *>(smem);       // [mt][xst]
    float *red = reinterpret_cast<float *>(smem + (((size_t)a.mt * xst * sizeof(X) + 15) & ~size_t(15)));  // [4][RB * 16][RS]
    float *sp = red + 4 * RB * 16 * kRwRS;     // [RB * 16][RS]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nl = lane & 15, g = lane >> 4;
    const int K = a.K;
    const int64_t m0 = (int64_t)blockIdx.y * a.mt;
    const int live = (int)min((int64_t)a.mt, a.M - m0);
    const int c0 = wave * a.cpw, c1 = min(c0 + a.cpw, a.nch);  // the wave's chunks (maybe none)

    // ---- weights and scales of chunk c, rows of pass ps
    struct Buf {
        u32x4 w[RB];
        f16 s[RB][NS];
    };
    auto issue = [&](int ps, int c, Buf &b) {
        c = min(c, a.nch - 1);
#pragma unroll
        for (int r = 0; r < RB; r++) {
            const int64_t row = min(((int64_t)ps * RB + r) * 16 + nl, a.N - 1);
            const uint8_t *qr = a.q + row * (int64_t)(K >> 1);
            const f16 *sr = a.scales + row * a.ngroups;
            if constexpr (WIDE) {
                b.w[r] = *reinterpret_cast<const u32x4 *>(qr + min(c * 64 + 16 * g, (K >> 1) - 16));
                b.s[r][0] = sr[min(4 * c / a.g32, a.ngroups - 1)];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    b.w[r][j] = *reinterpret_cast<const uint32_t *>(qr + min(c * 64 + 16 * j + 4 * g, (K >> 1) - 4));
                    b.s[r][j] = sr[min((4 * c + j) / a.g32, a.ngroups - 1)];
                }
            }
        }
    };
    // ---- entries of the wave's rows: row i's bounds and its first 64
    //      entries, one per lane (place of its activation in a token's row |
    //      value bits << 16; none: the zero place past the last column, 0)
    auto row_of = [&](int ps, int i) -> int64_t { return (int64_t)ps * RB * 16 + wave * NR + i; };
    int32_t js[NR], je[NR];
    uint32_t ent[NR];
    auto entries = [&](int64_t jb, int32_t end) -> uint32_t {
        const int32_t j = (int32_t)min(jb + lane, (int64_t)max(end - 1, 0));
        const uint32_t c = (uint32_t)a.col[j];
        const uint32_t v = __builtin_bit_cast(uint16_t, a.vals[j]);
        const uint32_t at = F16 ? (c & ~7u) | (uint32_t)interleaved_pos(c & 7) : c;
        return (c < (uint32_t)K && jb + lane < end) ? (at | (v << 16)) : (uint32_t)(a.nch * 128);
    };
    auto bounds = [&](int ps) {
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const int64_t n = row_of(ps, i);
            csr_row_range(a.row_ptr, min(n, a.N - 1), a.nnz, js[i], je[i]);
            if (n >= a.N) je[i] = js[i];
        }
    };

    // ---- staging: 16-byte pieces, columns past K zero; FP16 in the
    //      interleaved order of its weight conversion
    const int vpt = a.nch * 128 / EV;          // pieces per token
    const int total = live * vpt;
    auto load_x = [&](int p) -> u32x4 {
        const int t = min(p, total - 1) / vpt, k = (min(p, total - 1) - t * vpt) * EV;
        return *reinterpret_cast<const u32x4 *>(static_cast<const X *>(a.x) + (m0 + t) * K + min(k, K - EV));
    };
    auto store_x = [&](int p, u32x4 v) {
        if (p >= total) return;
        const int t = p / vpt, k = (p - t * vpt) * EV;
        if (k >= K) v = u32x4{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4 *>(xs + t * xst + k) = F16 ? permute_x8(v) : v;
    };
    for (int t = tid; t < live; t += kRwNT)  // the zero place (and its row's padding)
        *reinterpret_cast<u32x4 *>(xs + t * xst + a.nch * 128) = u32x4{0u, 0u, 0u, 0u};
    const int span = kRwNT * kRwXB;
    int p0 = tid;
    u32x4 xr[kRwXB];
    for (; p0 + span < tid + total; p0 += span) {  // all but the last round (uniform)
#pragma unroll
        for (int i = 0; i < kRwXB; i++) xr[i] = load_x(p0 + kRwNT * i);
#pragma unroll
        for (int i = 0; i < kRwXB; i++) store_x(p0 + kRwNT * i, xr[i]);
    }
    int ps = blockIdx.x;
    Buf buf[kRwD];
#pragma unroll
    for (int i = 0; i < kRwXB; i++) xr[i] = load_x(p0 + kRwNT * i);
    if (a.sparse) bounds(ps);
#pragma unroll
    for (int d = 0; d < kRwD; d++) issue(ps, c0 + d, buf[d]);
    if (a.sparse) {
#pragma unroll
        for (int i = 0; i < NR; i++) ent[i] = entries(js[i], je[i]);
    }
#pragma unroll
    for (int i = 0; i < kRwXB; i++) store_x(p0 + kRwNT * i, xr[i]);
    __syncthreads();

    const X *xa = xs + min(nl, live - 1) * xst;  // the lane's token (padding tokens repeat the last one)
    for (;;) {
        // ---- dense term
        f32x4 acc[RB];
#pragma unroll
        for (int r = 0; r < RB; r++) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto mfma = [](const u32x4 &av, const u32x4 &bv, const f32x4 &c) -> f32x4 {
            if constexpr (F16)
                return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, bv),
                                                              c, 0, 0, 0);
            else
                return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av),
                                                               __builtin_bit_cast(bf16x8, bv), c, 0, 0, 0);
        };
        auto chunk = [&](int c, const Buf &b) {
            const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
            // F32: the two lower parts in a chain of their own, so that the
            // sum of the high parts rounds a third as often
            f32x4 part[RB], low[F32 ? RB : 1];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const X *xp = xa + c * 128 + (WIDE ? 32 * g + 8 * j : 32 * j + 8 * g);
                u32x4 av[NP];
                if constexpr (F32)
                    split_bf16x3(*reinterpret_cast<const f32x4 *>(xp), *reinterpret_cast<const f32x4 *>(xp + 4), av);
                else
                    av[0] = *reinterpret_cast<const u32x4 *>(xp);
#pragma unroll
                for (int r = 0; r < RB; r++) {
                    uint32_t bw[4];
                    if constexpr (F16) int4x8_to_f16_interleaved(b.w[r][j], bw);
                    else int4x8_to_bf16_exact(b.w[r][j], bw);
                    const u32x4 bv = u32x4{bw[0], bw[1], bw[2], bw[3]};
                    const bool first = !WIDE || j == 0;
                    part[r] = mfma(av[0], bv, first ? zero : part[r]);
                    if constexpr (F32) low[r] = mfma(av[1], bv, mfma(av[2], bv, first ? zero : low[r]));
                    if (!WIDE || j == 3) {
                        const float s = (float)b.s[r][WIDE ? 0 : j] * (F16 ? 1.0f : kBf16Q);
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            acc[r][i] = __builtin_fmaf(s, F32 ? part[r][i] + low[F32 ? r : 0][i] : part[r][i], acc[r][i]);
                    }
                }
            }
        };
        for (int c = c0; c < c1; c += kRwD) {
#pragma unroll
            for (int d = 0; d < kRwD; d++) {
                if (c + d < c1) chunk(c + d, buf[d]);  // (uniform)
                issue(ps, c + d + kRwD, buf[d]);
            }
        }

        // ---- sparse sums: lane (entry lane / tl of a round, token lane % tl).
        //      After the dense term: the entries' loads were issued after the
        //      weights'
        if (a.sparse) {
            const int tl = a.tl, tok = min(lane & (tl - 1), live - 1), e0 = lane / tl, epi = 64 / tl;
            const X *xt = xs + tok * xst;
            auto product = [&](uint32_t w, float s) -> float {
                const float v = (float)__builtin_bit_cast(f16, (uint16_t)(w >> 16));
                const X x = xt[w & 0xffffu];
                float xv;
                if constexpr (F32) xv = x;
                else if constexpr (F16) xv = (float)__builtin_bit_cast(f16, x);
                else xv = bf16_bits_to_f32(x);
                return __builtin_fmaf(v, xv, s);
            };
            // every row's first 64 entries in step (a row that ends earlier
            // holds empty ones): the rows' LDS round trips overlap
            float s[NR];
            int32_t top = 0;
#pragma unroll
            for (int i = 0; i < NR; i++) {
                s[i] = 0.f;
                top = max(top, je[i] - js[i]);
            }
            top = min(top, 64);
            for (int r = 0; r < top; r += epi) {
                uint32_t w[NR];
#pragma unroll
                for (int i = 0; i < NR; i++) w[i] = __shfl(ent[i], r + e0);  // (r + e0 < 64)
#pragma unroll
                for (int i = 0; i < NR; i++) s[i] = product(w[i], s[i]);
            }
#pragma unroll
            for (int i = 0; i < NR; i++) {  // longer rows
                for (int64_t jb = (int64_t)js[i] + 64; jb < je[i]; jb += 64) {
                    const uint32_t en = entries(jb, je[i]);
                    for (int r = 0; r < 64; r += epi) s[i] = product(__shfl(en, r + e0), s[i]);
                }
            }
            for (int off = 32; off >= tl; off >>= 1)
#pragma unroll
                for (int i = 0; i < NR; i++) s[i] += __shfl_xor(s[i], off, 64);
            if (lane < live) {
#pragma unroll
                for (int i = 0; i < NR; i++) sp[(wave * NR + i) * kRwRS + lane] = s[i];
            }
        }

        // ---- the waves' partials: waves 4 .. 7 hand theirs to 0 .. 3, whose
        //      four sums are added below (token 4 g + i of row nl in a lane)
        float *mine = red + (wave & 3) * RB * 16 * kRwRS;
        if (wave >= 4) {
#pragma unroll
            for (int r = 0; r < RB; r++) *reinterpret_cast<f32x4 *>(mine + (16 * r + nl) * kRwRS + 4 * g) = acc[r];
        }
        __syncthreads();
        if (wave < 4) {
#pragma unroll
            for (int r = 0; r < RB; r++) {
                f32x4 *p = reinterpret_cast<f32x4 *>(mine + (16 * r + nl) * kRwRS + 4 * g);
                *p = acc[r] + *p;
            }
        }
        const int next = ps + (int)gridDim.x;
        const bool more = next < a.npass;  // (uniform)
        if (more) {
            if (a.sparse) {
                bounds(next);
#pragma unroll
                for (int i = 0; i < NR; i++) ent[i] = entries(js[i], je[i]);
            }
#pragma unroll
            for (int d = 0; d < kRwD; d++) issue(next, c0 + d, buf[d]);
        }
        __syncthreads();
        for (int o = tid; o < RB * 16 * live; o += kRwNT) {
            const int t = o / (RB * 16), row = o - t * (RB * 16);
            const int64_t n = (int64_t)ps * RB * 16 + row;
            if (n >= a.N) continue;
            const float *p = red + row * kRwRS + t;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < 4; w++) v += p[w * RB * 16 * kRwRS];
            if (a.sparse) v += a.alpha * sp[row * kRwRS + t];
            if (a.bias) v = round_as(IO, v) + load_as_f32(a.bias, a.bias_dtype, n);
            store_from_f32(a.y, IO, (m0 + t) * a.N + n, v);
        }
        if (!more) break;
        ps = next;
        __syncthreads();  // the buffers are read before the next pass writes them
    }
}

// ------------------------------------------------------------------ host

template <int IO, int RB, bool WIDE>
static hipError_t rows_launch_t(const RowsArgs &d, const RowsShape &sh, hipStream_t stream) {
    // more than 64 KB of dynamic LDS must be allowed once per device (the
    // attribute call is idempotent, so two threads racing to set it is harmless)
    static std::atomic<int> allowed[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && !allowed[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(rows_kernel<IO, RB, WIDE>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kRwLdsMax);
        if (e != hipSuccess) return e;
        allowed[dev].store(1, std::memory_order_release);
    }
    hipLaunchKernelGGL((rows_kernel<IO, RB, WIDE>), dim3((unsigned)sh.gx, (unsigned)sh.tiles), dim3(kRwNT),
                       (uint32_t)sh.lds, stream, d);
    return hipGetLastError();
}

template <int IO, bool WIDE>
static hipError_t rows_launch_rb(const RowsArgs &d, const RowsShape &sh, hipStream_t stream) {
    switch (sh.rb) {
        case 1: return rows_launch_t<IO, 1, WIDE>(d, sh, stream);
        case 2: return rows_launch_t<IO, 2, WIDE>(d, sh, stream);
        case 3:
            if constexpr (WIDE || IO != ORTH_DT_F32) return rows_launch_t<IO, 3, WIDE>(d, sh, stream);
            return hipErrorInvalidValue;
        default:
            if constexpr (WIDE) return rows_launch_t<IO, 4, WIDE>(d, sh, stream);
            return hipErrorInvalidValue;
    }
}

template <int IO>
static hipError_t rows_launch_io(const RowsArgs &d, const RowsShape &sh, hipStream_t stream) {
    return sh.wide ? rows_launch_rb<IO, true>(d, sh, stream) : rows_launch_rb<IO, false>(d, sh, stream);
}

hipError_t launch_rows(const ForwardArgs &a, int cus, hipStream_t stream) {
    RowsShape sh;
    if (!rows_shape(a, cus, sh)) return hipErrorInvalidValue;
    RowsArgs d;
    d.q = a.q;
    d.scales = static_cast<const f16 *>(a.scales);
    d.ngroups = (int)a.ngroups;
    d.g32 = a.ngroups == 1 ? (1 << 20) : (int)(a.G / 32);
    d.row_ptr = a.row_ptr;
    d.col = a.col;
    d.vals = static_cast<const f16 *>(a.vals);
    d.nnz = (int32_t)a.nnz;
    d.sparse = a.has_ortho;
    d.alpha = a.alpha;
    d.x = a.x;
    d.y = a.y;
    d.M = a.M;
    d.N = a.N;
    d.K = (int)a.K;
    d.nch = (int)((a.K + 127) / 128);
    d.cpw = (d.nch + kRwW - 1) / kRwW;
    d.mt = sh.mt;
    d.tl = sh.tl;
    d.npass = sh.npass;
    d.bias = a.bias;
    d.bias_dtype = a.bias_dtype;
    if (a.io_dtype == ORTH_DT_F32) return rows_launch_io<ORTH_DT_F32>(d, sh, stream);
    if (a.io_dtype == ORTH_DT_BF16) return rows_launch_io<ORTH_DT_BF16>(d, sh, stream);
    return rows_launch_io<ORTH_DT_F16>(d, sh, stream);
}

}  // namespace orth
