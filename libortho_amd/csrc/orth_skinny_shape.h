// How the split-K mid-batch kernel (orth_skinny.hip) lays out a call: host
// arithmetic that the dispatcher needs too.
#pragma once
#include <algorithm>
#include <cmath>

#include "orth_common.h"

namespace orth {

constexpr int kSkNT = 512;            // 8 waves
constexpr int kSkRows = 128;          // rows per workgroup (= ortho plan block)
constexpr int kSkMaxCPS = 8;          // chunks per slice (compile-time bound)

// Chunks per slice the kernel of ntt token tiles is built for: even (group
// scales are read in pairs) and with at most 8 activation pieces per thread.
constexpr int sk_cps_bound(int ntt) { return ntt * kSkMaxCPS > 16 ? ((16 / ntt) & ~1) : kSkMaxCPS; }

constexpr int kSsRows = 16;                // rows per unit (one wave's)
constexpr int kSsLdsMax = 150 * 1024;
constexpr int kSsLdsCu = 160 * 1024;       // of a compute unit

inline int ss_lds(int64_t K, int tt) {
    return (int)(K * 2 * tt + K / 8 * 16 + 16 + (kSkNT / 64) * kSsRows * tt * 4);
}

// Tokens per workgroup (0: K is too large).  As many as fit: every token tile
// reads all of the CSR, which costs more than the second workgroup per CU
// that a smaller tile would leave room for (8192 -> 4096 at 48 tokens: 24.7 us
// with 8 tokens, 26.1 with 4).
inline int ss_tokens(int64_t K) {
    for (int tt = 8; tt >= 2; tt /= 2)
        if (K <= 65536 && ss_lds(K, tt) <= kSsLdsMax) return tt;
    return 0;
}

struct SkinnyShape {
    int ntt, cps, S, nblocks, xstride;
    int lds_cr, lds_xs, lds_sp, lds_xt, lds_bytes;
    int sp_wgs, sp_tt, sp_tiles;  // the ortho term's own workgroups (0: none)
    bool sp_own;  // they take the entries only where the plan does not locate them
};

inline bool skinny_shape(const ForwardArgs &a, int cus, SkinnyShape &sh) {
    const int ntt = (int)((a.M + 15) / 16);
    const int nchunks = (int)(a.K / 128);
    sh.ntt = ntt;
    sh.nblocks = (int)((a.N + kSkRows - 1) / kSkRows);
    const int mp = ntt * 16;
    const int cps_max = sk_cps_bound(ntt);
    // enough workgroups to keep every CU streaming: about 1.3 per CU
    int S = (int)std::min<int64_t>(nchunks, std::max<int64_t>(1, (cus * 13 / 10 + sh.nblocks - 1) / sh.nblocks));
    int cps = (nchunks + S - 1) / S;
    cps = std::min(cps + (cps & 1), cps_max);              // even: group scales read as pairs
    S = (nchunks + cps - 1) / cps;
    sh.cps = cps;
    sh.S = S;
    sh.xstride = cps * 128 + 8;
    int off = 0;
    sh.lds_cr = off;
    off += cps * mp * 4;
    sh.lds_xs = off;
    off += ((mp * sh.xstride * 2) + 15) & ~15;
    sh.lds_sp = off;
    off += a.has_ortho && ntt == 1 ? kSkRows * mp * 4 : 0;  // the kernel's QUAD exchange
    sh.lds_xt = off;  // the transposed activations: 8 or 16 tokens a column, a zero column after the last
    if (a.has_ortho && ntt == 1) off += (kSkMaxCPS * 128 + 1) * (a.M <= 8 ? 16 : 32) + (kSkMaxCPS * 128 / 8) * 16;
    sh.lds_bytes = off;
    sh.sp_wgs = sh.sp_tt = sh.sp_tiles = 0;
    sh.sp_own = false;
    if (a.has_ortho && ntt > 1 && S > 1 && ss_tokens(a.K) > 0 &&
        (int64_t)(S + 1) * a.M * a.N * 4 <= (int64_t)ORTH_NOALLOC_SCRATCH_BYTES) {
        int tt = ss_tokens(a.K), tiles = (int)((a.M + tt - 1) / tt);
        // three workgroups to four CUs, beside the dense ones (4096 -> 11008 at
        // 48 tokens, 1 %: 128 workgroups 30.3 us, 192 26.8, 256 28.8), each
        // wave with at least one unit of rows; whole rows of the XCD map
        const int64_t units = (a.N + kSsRows - 1) / kSsRows;
        auto count = [&] {
            const int64_t per = std::max<int64_t>(1, std::min<int64_t>((units + 7) / 8, cus * 3 / 4 / tiles));
            return (int)((per * tiles + 7) / 8 * 8);
        };
        int wgs = count();
        // With a plan each lane can find its own entries of the slice instead.
        // That is the faster one for many entries in rows of like length, which
        // the estimates below (us; fitted to 3,048 planned calls, off by 6 and
        // 12 %) tell well enough.  Own workgroups / own entries, 1 %, 5 % and 20 %:
        // 4096 -> 1024 at 33 tokens 12.3 / 12.6, 20.6 / 16.1, 55.9 / 38.9; 4096 ->
        // 4096 at 64 tokens 22 / 24, 37.8 / 29.1, 109 / 66.  Rows of very unlike
        // length favour the workgroups (4096 -> 14336 at 49 tokens, 1 %, lognormal
        // rows: 57 / 144), also where few entries make the extra partial the
        // larger part (1024 -> 14336 at 48 tokens, 0.5 %: 17.7 / 14.4 with like
        // rows, 18.9 / 37.8 with lognormal ones: up to 8 entries of a row and slice
        // stay with the workgroups).  (33 tokens and more at K > 4096:
        // the prefill kernel takes the calls with many entries.)
        const double e = (double)a.nnz / a.N, es = e / S;
        const double run = std::ceil((double)units / std::max(1, wgs / tiles * 8));  // units of a wave
        const double own_wgs = 4.9 + 0.6 * cps * std::max(1.0, (double)sh.nblocks * S / (2 * cus)) +
                               run * (0.003 * e * tt + 1.6 * std::ceil(e / 48)) + 0.28e-4 * a.K * tt +
                               1.5e-6 * (S + 1) * a.M * a.N + 0.39e-6 * tiles * a.nnz;
        const double rounds = std::ceil((double)sh.nblocks * S / ((ntt == 2 ? 2 : 1) * cus));
        const double own_entries = 9.6 + rounds * (0.98 * cps + 0.36 * ntt * std::sqrt(es)) + ntt * (0.12 * es + 2.2e-6 * a.nnz);
        sh.sp_own = a.planned && (a.M <= 32 || a.K <= 4096) && es > 8 && own_wgs >= 1.05 * own_entries;
        if (sh.sp_own) {
            // (workgroups that mostly end at once: no more LDS than leaves room
            // for all to start, or for as many dense ones to a CU)
            const int all = (sh.nblocks * S + wgs + cus - 1) / cus;
            const int room = kSsLdsCu / std::max(1, std::min(all, kSsLdsCu / off));
            while (tt > 2 && ss_lds(a.K, tt) > room) tt /= 2;
            tiles = (int)((a.M + tt - 1) / tt);
            wgs = count();
        }
        sh.sp_tt = tt;
        sh.sp_tiles = tiles;
        sh.sp_wgs = wgs;
        sh.lds_bytes = std::max(off, ss_lds(a.K, tt));
    }
    return off <= 150 * 1024;
}

// Workspace bytes of a call of that shape (0 when K is not split).
inline int64_t skinny_shape_workspace(const ForwardArgs &a, const SkinnyShape &sh) {
    return sh.S > 1 ? (int64_t)(sh.S + (sh.sp_wgs > 0 ? 1 : 0)) * a.M * a.N * 4 : 0;
}

// 33 .. 64 tokens at K > 4096 (the dispatcher's choice between this kernel and
// the prefill kernel with K split).  us, this / prefill: without an ortho term
// 11008 -> 4096 at 33 tokens 16.6 / 29.7, at 64 22.1 / 31.5, 8192 -> 2048 at 64
// 11.6 / 22.9; with one, where a workgroup of its own keeps 8 tokens (18 K +
// 4112 bytes of LDS within 150 KB: K up to 8192) and it is neither too large
// (entries x tokens) nor its rows too long: 5120 -> 5120 at 64, 1 % (17 million)
// 25.0 / 27.7, 2 % (34) 31.3 / 28.2, 8192 -> 4096 at 40, 2 % (26.8) 25.6 / 30.6,
// 5120 -> 8192 at 64, 1 % (26.8) 35.2 / 33.1, 8192 -> 2048 at 64, 2 % (21) 21.1 /
// 26.7; 8192 -> 1024 at 33, 3 % 24.5 / 25.3, 4 % 31 / 25.5, 5 % 33.6 / 25.3, 5120
// -> 512 at 33, 3 % 18 / 19.1, 5 % 23.5 / 19.2; 11008 -> 4096 at 64, 2 % 56.7 /
// 35.7.  Its partials must fit the no-allocation scratch array, as the prefill
// kernel's always do.
inline bool skinny_wide_k_preferred(const ForwardArgs &a, int cus) {
    SkinnyShape sh;
    if (!skinny_shape(a, cus, sh) || skinny_shape_workspace(a, sh) > (int64_t)ORTH_NOALLOC_SCRATCH_BYTES) return false;
    return !a.has_ortho || (sh.sp_tt == 8 && a.nnz * a.M <= 27000000 && a.nnz * 32 <= a.N * a.K);
}

}  // namespace orth
