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

// The general kernel a call takes.  FP32 activations, large batches: the tile
// kernel takes the same time for any batch of one round of its grid (~1 us per
// 64 columns), the rows kernel's grows with M * N.  us, rows / tiles, alpha = 1:
// 4096 -> 4096 at 64 tokens 52 / 74, at 80 81 / 76, at 128 100 / 76; 4096 ->
// 11008 at 32 78 / 76; 1024 -> 4096 at 64 20 / 28, at 128 37 / 29; where
// only 4 tokens' columns fit the rows kernel's LDS, 8192 -> 1024 at 128
// 83 / 132, at 256 159 / 133, 11008 -> 4096 at 32 150 / 175, at 48 186 / 180.
// Without the rows kernel (FP32 scales or values) they cross the wave-per-row
// kernel near 2^17: 4096 -> 4096 at 24 tokens 61 (wave) / 72, at 32 80 / 72.
// The rows kernel needs enough outputs to pay for the staging and its barrier:
// the wave-per-row kernel's time grows with M * N, its hardly below 16 tokens
// (us, wave / rows): FP32 4096 -> 4096 at 2 tokens 10.2 / 11.4, at 4 14.6 /
// 12.3, 4096 -> 11008 at 1 18.8 / 22.3, at 2 25.0 / 22.0, at 8 66 / 24.9; FP16
// 4000 -> 4096 at 1 10.8 / 11.2, 4000 -> 11008 at 1 20.3 / 13.5, at 16 139 /
// 18.5; narrow rows (2720 -> 4096, group 32) at 4 12.9 / 12.4, at 16 37.8 /
// 16.4.
inline int general_variant(const ForwardArgs &a, int cus) {
    RowsShape sh;
    const bool rows = rows_shape(a, cus, sh) &&
                      a.M * a.N >= (!sh.wide ? 24576 : a.io_dtype == ORTH_DT_F32 ? 16384 : 8192);
    const int64_t from = !rows ? 1 << 17 : a.K >= 8192 ? 200000 : 300000;
    if (a.M * a.N >= from && float_supported(a)) return GENERAL_TILES;
    return rows ? GENERAL_ROWS : GENERAL_WAVE;
}

}  // namespace orth
