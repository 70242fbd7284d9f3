// Which of the general kernels takes a call, and how the rows and the tile
// kernel lay it out: host arithmetic that the dispatcher needs too.
#pragma once
#include <algorithm>
#include <cmath>

#include "orth_common.h"

namespace orth {

// The kernels behind KERNEL_GENERAL (orth_hip_last_variant()).
enum GeneralVariant {
    GENERAL_WAVE = 1,   // a wave per output row (orth_general.hip): every call
    GENERAL_ROWS = 2,   // activations staged once, 16-row blocks (orth_rows.hip)
    GENERAL_TILES = 3   // FP32 batches, 64 x 128 tiles (orth_float.hip)
};

// ------------------------------------------------------------ rows kernel

constexpr int kRwW = 8;            // waves
constexpr int kRwRS = 20;          // row stride of the partials in LDS, in floats
constexpr int kRwMaxRB = 4;
constexpr int64_t kRwLdsMax = 160 * 1024;

struct RowsShape {
    int rb, mt, tl, tiles, lds, gx, npass;
    bool wide;
};

inline bool rows_shape(const ForwardArgs &a, int cus, RowsShape &sh) {
    if (a.K % 8 != 0 || a.K < 32 || a.N >= ((int64_t)1 << 31)) return false;
    if (a.K > 65408) return false;  // an entry holds its activation's place, at most K rounded up to 128, in 16 bits
    if (a.scale_dtype != ORTH_DT_F16 || (a.has_ortho && a.val_dtype != ORTH_DT_F16)) return false;
    if (a.ngroups != 1 && a.G % 32 != 0) return false;
    if ((reinterpret_cast<uintptr_t>(a.x) & 15) || (reinterpret_cast<uintptr_t>(a.q) & 3)) return false;
    sh.wide = a.K % 32 == 0 && (reinterpret_cast<uintptr_t>(a.q) & 15) == 0 && (a.ngroups == 1 || a.G % 128 == 0);
    const int64_t kp = (a.K + 127) / 128 * 128;
    const int64_t tok = a.io_dtype == ORTH_DT_F32 ? (kp + 4) * 4 : (kp + 8) * 2;  // LDS bytes of a token
    const int64_t nblk = (a.N + 15) / 16;
    // one workgroup per CU where the rows allow it, each looping over its
    // passes with the activations staged once.  More blocks per pass share
    // the reading (and cutting) of the activations and the pass's barriers:
    // a pass costs about 1.5 blocks beside its own (narrow rows: registers
    // for 3 blocks, with FP32 activations 2)
    int64_t best = 0;
    const int max_rb = sh.wide ? kRwMaxRB : a.io_dtype == ORTH_DT_F32 ? 2 : 3;
    for (int rb = 1; rb <= max_rb; rb++) {
        const int64_t red = (int64_t)5 * rb * 16 * kRwRS * 4 + 16;
        const int64_t fit = std::min<int64_t>(16, (kRwLdsMax - red) / tok);
        if (fit < 1) break;
        const int64_t tiles = (a.M + fit - 1) / fit;
        if (tiles > 65535) break;
        const int64_t npass = (nblk + rb - 1) / rb;
        const int64_t gx = std::min<int64_t>(npass, std::max<int64_t>(1, cus / tiles));
        const int64_t rounds = (tiles * gx + cus - 1) / cus;
        const int64_t cost = rounds * ((npass + gx - 1) / gx) * (2 * rb + 3);
        if (best && cost >= best) continue;
        best = cost;
        sh.rb = rb;
        sh.tiles = (int)tiles;
        sh.mt = (int)((a.M + tiles - 1) / tiles);
        sh.lds = (int)(((sh.mt * tok + 15) & ~int64_t(15)) + red);
        sh.npass = (int)npass;
        sh.gx = (int)gx;
    }
    if (!best) return false;
    sh.tl = 1;
    while (sh.tl < sh.mt) sh.tl *= 2;
    return true;
}

// ----------------------------------------------------------- tile kernel

constexpr int kFlBM = 64, kFlBN = 128, kFlBK = 64;
constexpr int kFlMaxGroups = 128;          // scale groups the tile's LDS holds (64 KB)

// Its sparse term: threads and waves of a workgroup, rows per unit (one wave's).
constexpr int kFoNT = 1024;
constexpr int kFoW = kFoNT / 64;
constexpr int kFoRows = 16;
constexpr int64_t kFoLdsMax = 160 * 1024;

// Tokens a sparse-term workgroup keeps in LDS (0: K is too large).
inline int float_ortho_tokens(int64_t K) {
    for (int tt = 8; tt >= 1; tt /= 2)
        if ((K + 1 + kFoRows * kFoW) * tt * 4 <= kFoLdsMax) return tt;
    return 0;
}

// The same for a call of M tokens, and its workgroups per token tile: about
// one workgroup per CU (its LDS holds one), each wave with work.
inline int float_ortho_tile(int64_t K, int64_t M) {
    const int64_t tt = std::min<int64_t>(float_ortho_tokens(K), M);
    return tt >= 8 ? 8 : tt >= 4 ? 4 : tt >= 2 ? 2 : 1;
}
inline int64_t float_ortho_wgs(int64_t N, int64_t ntm, int cus) {
    const int64_t units = (N + kFoRows - 1) / kFoRows;
    return std::max<int64_t>(1, std::min<int64_t>((units + kFoW - 1) / kFoW, cus / ntm));
}

inline bool float_supported(const ForwardArgs &a) {
    if (a.io_dtype != ORTH_DT_F32 || a.K % kFlBK != 0) return false;
    if (a.ngroups != 1 && (a.G % kFlBK != 0 || a.ngroups > kFlMaxGroups)) return false;
    if (reinterpret_cast<uintptr_t>(a.x) & 15 || reinterpret_cast<uintptr_t>(a.q) & 7) return false;
    if (a.has_ortho && float_ortho_tokens(a.K) == 0) return false;
    const int64_t tiles = ((a.M + kFlBM - 1) / kFlBM) * ((a.N + kFlBN - 1) / kFlBN);
    return a.M + a.N < ((int64_t)1 << 31) && tiles < ((int64_t)1 << 31);
}

// ----------------------------------------------------------------- choice
//
// The kernels' times in microseconds, from the shapes of their loops.  The
// constants are a least-squares fit to MI355X times of calls whose weights
// come from HBM: 14,255 wave-per-row, 13,934 rows and 4,761 tile calls over K
// 256 .. 30000, N 512 .. 28672, 1 .. 256 tokens, 0 .. 20 % ortho, FP16 and
// FP32 activations; they are off by 10, 8 and 6 % (rms).

inline double ceil_div(double a, double b) { return std::ceil(a / b); }

// A wave per row and token tile: its own steps (512 columns, 64 entries) one
// after the other, beside those of all waves.
inline double wave_us(const ForwardArgs &a, int cus) {
    static const double step[3] = {0.55, 0.78, 1.0}, steps[3] = {1.1, 1.9, 2.9}, row[3] = {0.43, 0.64, 1.9},
                        ent[3] = {0.49, 1.2, 2.4};
    const int k = a.M <= 1 ? 0 : a.M == 2 ? 1 : 2;  // tiles of 1, 2 and 4 tokens
    const double waves = (double)a.N * ceil_div((double)a.M, 1 << k) * 1e-4, rows = a.N * 1e-4;
    const double it = ceil_div((double)a.K, 512), se = a.has_ortho ? ceil_div((double)a.nnz, 64.0 * a.N) : 0;
    const double one = it * step[k] + 0.9 * se;
    const double all = (waves * (it * steps[k] + row[k] + se * ent[k]) + rows * (0.9 * it + 1.8 * se)) * 256 / cus;
    return 2.8 + std::sqrt(one * one + all * all);
}

// Staging once per workgroup, then its passes: chunks (wide rows' loads go four
// at a time, also where a wave has fewer; narrow rows of several groups load
// and place four scales a chunk) and entries.
inline double rows_us(const ForwardArgs &a, const RowsShape &sh, int cus) {
    const bool f32 = a.io_dtype == ORTH_DT_F32;
    const double rounds = ceil_div((double)sh.tiles * sh.gx, cus), passes = ceil_div(sh.npass, sh.gx);
    const double nch = ceil_div((double)a.K, 128), cpw = ceil_div(nch, kRwW);
    const double busy = ceil_div(nch, cpw) / kRwW;  // waves with chunks
    const double chunks = sh.wide ? 0.074 * cpw + 1.4 * ceil_div(cpw, 4) * busy : (a.ngroups > 1 ? 1.6 : 0.59) * cpw;
    const double dense = sh.rb * chunks + (f32 ? 0.65 * cpw : 0);
    const double sparse = !a.has_ortho ? 0 : sh.rb * (0.0023 * (double)a.nnz / a.N * sh.tl + 1.3 * ceil_div((double)a.nnz, 64.0 * a.N));
    const double start = 3.0 + sh.rb * (sh.wide ? 1.1 : 3.8) + 1.5 * sh.mt * (double)a.K * (f32 ? 4 : 2) / 65536;
    const double pass = 3.0 + (sh.wide ? 0 : 2.3 * sh.rb);
    return rounds * (start + passes * (dense + sparse) + (passes - 1) * pass) +
           0.058e-6 * sh.tiles * (double)a.N * a.K / 2;
}

// Rounds of the tile grid, and of the sparse launch: its staging, then a
// wave's units of 16 rows, 48 entries of a row at a time.
inline double tiles_us(const ForwardArgs &a, int cus) {
    const double tiles = ceil_div((double)a.M, kFlBM) * ceil_div((double)a.N, kFlBN);
    double t = ceil_div(tiles, cus) * (6.1 + 0.89 * (double)(a.K / kFlBK));
    if (!a.has_ortho) return t;
    const int tt = float_ortho_tile(a.K, a.M);
    const int64_t ntm = (a.M + tt - 1) / tt, wgs = float_ortho_wgs(a.N, ntm, cus);
    const double units = ceil_div(ceil_div((double)a.N, kFoRows), (double)wgs * kFoW);
    const double unit = 0.0023 * (double)a.nnz / a.N * tt + 2.2 * ceil_div((double)a.nnz, 48.0 * a.N) + 2.0;
    return t + ceil_div((double)ntm * wgs, cus) * (3.5 * (double)a.K * tt * 4 / 65536 + units * unit);
}

// The general kernel a call takes: the one with the smallest of these times
// (the wave-per-row one within 3 %, at one token 20 %: it gains more from
// weights in cache, FP32 4096 -> 4096 at 1 token 10.9 / 12.1 then).
// us, wave / rows / tiles, at 1 % unless said: FP32 4096 -> 4096, 1 token 12.8 /
// 12.5 / 67, 4 tokens 20.5 / 13.4 / 70, 64 tokens 173 / 57 / 73, 128 tokens 348 /
// 106 / 74; FP32 4096 -> 11008, 1 token 24.8 / 24.3; FP32 8192 -> 1024, 128
// tokens 194 / 88 / 133, 256 tokens 355 / 165 / 133; FP32 28672 -> 1024 without
// ortho, 24 tokens 101 / 155; FP32 1024 -> 1024 at 20 %, 16 tokens 11.7 / 20.3;
// FP16 4000 -> 11008, 1 token 25.2 / 17.6, 16 tokens 140 / 20.7; FP16 1344 ->
// 11008 in groups of 96 without ortho, 4 tokens 22.6 / 25.8, 16 tokens 54 / 26.
// (Lines at a fixed M * N sent calls with more entries, more columns or
// narrower rows than the ones they were drawn from to a kernel up to 4.8 times
// slower; by these times the chosen one is 0.5 % off the best on average, and
// in 0.5 % of the calls above more than 10 % slower than the wave-per-row one.)
inline int general_variant(const ForwardArgs &a, int cus) {
    int v = GENERAL_WAVE;
    double best = wave_us(a, cus) / (a.M == 1 ? 1.2 : 1.03);
    RowsShape sh;
    if (rows_shape(a, cus, sh)) {
        const double t = rows_us(a, sh, cus);
        if (t < best) best = t, v = GENERAL_ROWS;
    }
    if (float_supported(a) && tiles_us(a, cus) < 1.03 * best) v = GENERAL_TILES;  // (the surer estimate)
    return v;
}

}  // namespace orth
