// How the split-K mid-batch kernel (orth_skinny.hip) lays out a call: host
// arithmetic that the dispatcher needs too.
#pragma once
#include <algorithm>

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
    if (a.has_ortho && ntt > 1 && S > 1 && ss_tokens(a.K) > 0 &&
        (int64_t)(S + 1) * a.M * a.N * 4 <= (int64_t)ORTH_NOALLOC_SCRATCH_BYTES) {
        sh.sp_tt = ss_tokens(a.K);
        sh.sp_tiles = (int)((a.M + sh.sp_tt - 1) / sh.sp_tt);
        // three workgroups to four CUs, beside the dense ones (4096 -> 11008 at
        // 48 tokens, 1 %: 128 workgroups 30.3 us, 192 26.8, 256 28.8), each
        // wave with at least one unit of rows; whole rows of the XCD map
        const int64_t units = (a.N + kSsRows - 1) / kSsRows;
        const int64_t per = std::max<int64_t>(1, std::min<int64_t>((units + 7) / 8, cus * 3 / 4 / sh.sp_tiles));
        sh.sp_wgs = (int)((per * sh.sp_tiles + 7) / 8 * 8);
        sh.lds_bytes = std::max(off, ss_lds(a.K, sh.sp_tt));
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
// 11.6 / 22.9; with one, where a workgroup of its own keeps 8 tokens (K up to
// 8250) and it is not too large (entries x tokens): 5120 -> 5120 at 64, 1 % (17
// million) 25.0 / 27.7, 2 % (34) 31.3 / 28.2, 8192 -> 2048 at 64, 2 % (21)
// 21.1 / 26.7, 8192 -> 8192 at 40, 1 % (27) 43.3 / 45.7; 11008 -> 4096 at 64, 2 %
// 56.7 / 35.7.  Its partials must fit the no-allocation scratch array, as the
// prefill kernel's always do.
inline bool skinny_wide_k_preferred(const ForwardArgs &a, int cus) {
    SkinnyShape sh;
    if (!skinny_shape(a, cus, sh) || skinny_shape_workspace(a, sh) > (int64_t)ORTH_NOALLOC_SCRATCH_BYTES) return false;
    return !a.has_ortho || (sh.sp_tt == 8 && a.nnz * a.M <= 27000000);
}

}  // namespace orth
