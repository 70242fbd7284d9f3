"""The load path's kernels byte by byte: the ortho plan against a plain numpy
form of its layout (orth_prefill.hip), the CSR against torch's nonzero and the
INT4 nibbles against the divisions they round (orth_pack.hip)."""
import ctypes
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from libortho_amd import _lib  # noqa: E402

pytestmark = pytest.mark.gpu


def layer(K, N, density, seed, heavy=None):
    """CSR arrays, columns ascending; heavy: rows with many more entries."""
    g = np.random.Generator(np.random.PCG64(seed))
    p = np.full(N, density)
    if heavy is not None:
        p[heavy] = 0.6
    mask = g.random((N, K)) < p[:, None]
    rows, col = np.nonzero(mask)
    row_ptr = np.zeros(N + 1, np.int32)
    row_ptr[1:] = np.cumsum(np.bincount(rows, minlength=N))
    return row_ptr, col.astype(np.int32), g.normal(0, 0.1, col.size).astype(np.float16)


def tag(kind, N, K, nnz, words, g, c):
    m = 0xffffffff
    return (kind ^ (nnz & m) ^ (N * 0x9E3779B1 & m) ^ (K << 13 & m) ^ (words * 0xC2B2AE3D & m) ^ (g * 0x85EBCA77 & m)
            ^ (c * 0x27D4EB2F & m))


def cell_words(N, K, nnz, cols, most):
    mean = -(-16 * cols * nnz // (N * K))
    w = -(-(20 + mean + 4 * (math.isqrt(mean) + 1)) // 256) * 256
    return w if w <= most else 0


def reference(K, N, row_ptr, col, vals):
    """[(byte offset, bytes)] of the plan's parts, and its size."""
    nnz, nk, nb, nch = col.size, K // 64, -(-N // 128), K // 128
    vbits = vals.astype(np.float16).view(np.uint16).astype(np.uint32)
    flags = 0
    for n in range(N):
        c = col[row_ptr[n]:row_ptr[n + 1]].astype(np.int64)
        inr = c[(c >= 0) & (c < K)]
        flags |= 4 * bool((np.diff(c) <= 0).any()) | bool((np.diff(inr) <= 0).any())
    qcols = ((nch + 3) // 4 + 1 & ~1) * 128
    qw = cell_words(N, K, nnz, qcols, 2048) if K % 128 == 0 else 0
    sw = cell_words(N, K, nnz, 1024, 512) if K % 128 == 0 else 0
    head = np.array([0x504f5254, 5, 128, 64, nb, nk, N & 0xffffffff, N >> 32, K, 0, nnz, 0, flags, qw, sw, 0], np.uint32)
    parts, at = [(0, head)], 64
    offs, ents = np.zeros((nb, nk + 1), np.int32), []
    row_of = np.repeat(np.arange(N), np.diff(row_ptr))
    for b in range(nb):
        lo, hi = row_ptr[b * 128], row_ptr[min(N, (b + 1) * 128)]
        j = np.arange(lo, hi)
        j = j[(col[lo:hi] >= 0) & (col[lo:hi] < K)]
        j = j[np.lexsort((j, row_of[j], col[j] // 64))]
        offs[b] = lo + np.searchsorted(col[j] // 64, np.arange(nk + 1))
        ents.append((lo, ((row_of[j] - b * 128).astype(np.uint32) << 24) | ((col[j].astype(np.uint32) & 63) << 16) | vbits[j]))
    parts.append((at, offs))
    at += (offs.nbytes + 15) // 16 * 16
    parts += [(at + 4 * int(lo), e) for lo, e in ents]
    at = (at + 4 * nnz + 15) // 16 * 16
    if K % 128:
        return parts, at
    table = np.zeros((N, nch + 1), np.uint16)
    for n in range(N):  # the first entry at or past each boundary, in CSR order
        top = np.maximum.accumulate(col[row_ptr[n]:row_ptr[n + 1]]) if row_ptr[n + 1] > row_ptr[n] else np.zeros(0)
        table[n] = np.searchsorted(top, 128 * np.arange(nch + 1), side="left")
    parts.append((at, table))
    at += (table.nbytes + 15) // 16 * 16
    for kind, words, cols, ncells in ((0x51524543, qw, qcols, 4), (0x53524543, sw, 1024, -(-K // 1024))):
        if not words:
            continue
        rec = np.full((-(-N // 16), ncells, words), 0xffff, np.uint32)
        for g in range(rec.shape[0]):
            for c in range(ncells):
                c0, c1, run, cap, r = c * cols, min((c + 1) * cols, K), 0, words - 20, rec[g, c]
                for i in range(16):
                    n, b = 16 * g + i, run
                    if n < N:
                        j = np.arange(row_ptr[n], row_ptr[n + 1])
                        j = j[(col[j] >= c0) & (col[j] < c1)]
                        w = (col[j] - c0).astype(np.uint32) | (vbits[j] << 16)
                        r[20 + min(run, cap):20 + min(run + j.size, cap)] = w[:max(0, cap - run)]
                        run += j.size
                    r[2 + i] = min(b, cap) | (min(run, cap) << 16)
                r[0], r[1], r[18:20] = tag(kind, N, K, nnz, words, g, c), max(0, run - cap), 0
        parts.append((at, rec))
        at += rec.nbytes
    return parts, at


def build(K, N, row_ptr, col, vals):
    dev = [torch.from_numpy(a).cuda() for a in (row_ptr, col, vals)]
    L = _lib.lib()
    d = _lib.OrthHipLayer()
    d.base.q_weight, d.base.q_scales, d.base.q_bits, d.base.scale_groups = 16, 16, 4, 1  # (not read)
    d.base.in_features, d.base.out_features = K, N
    d.ortho.row_ptr, d.ortho.col_indices, d.ortho.values = (t.data_ptr() for t in dev)
    d.ortho.value_dtype = _lib.DT_F16 if vals.dtype == np.float16 else _lib.DT_F32
    d.ortho.count, d.alpha = col.size, 1.0
    n = L.orth_ortho_plan_bytes(ctypes.byref(d))
    plan = torch.zeros(n, dtype=torch.uint8, device="cuda")
    _lib.check(L.orth_ortho_plan_build(ctypes.byref(d), plan.data_ptr(), n, torch.cuda.current_stream().cuda_stream))
    return plan.cpu().numpy()


def check(K, N, row_ptr, col, vals):
    got = build(K, N, row_ptr, col, vals)
    parts, size = reference(K, N, row_ptr, col, vals)
    assert got.size == size
    for at, want in parts:
        assert np.array_equal(got[at:at + want.nbytes], np.ascontiguousarray(want).view(np.uint8).reshape(-1)), at


# ragged rows and K not a multiple of 1024; K without tables; a heavy row (its
# group's records overflow, a row of several 64-entry batches); groups of more
# entries than are staged; records of 512 words, and none
@pytest.mark.parametrize("K,N,density,heavy", [
    (1152, 1000, 0.02, None), (4160, 300, 0.01, None), (64, 200, 0.1, None), (2048, 200, 0.004, [5, 6, 150]),
    (4096, 40, 0.3, None), (4096, 150, 0.02, [3]), (11008, 33, 0.03, [0, 32]), (12288, 17, 0.002, None)])
@pytest.mark.parametrize("order", ["sorted", "some", "reversed"])
def test_plan_bytes(gpu, K, N, density, heavy, order):
    """order: columns ascending; some rows not, among rows that are, with
    duplicates and columns out of range; every row descending."""
    row_ptr, col, vals = layer(K, N, density, 100 + K + N, heavy)
    g = np.random.Generator(np.random.PCG64(7))
    for n in range(N):
        c = col[row_ptr[n]:row_ptr[n + 1]]
        if order == "reversed":
            c[:] = c[::-1].copy()
        elif order == "some" and n % 5 == 1 and c.size:
            g.shuffle(c)
            c[g.integers(0, c.size)] = c[0]
        elif order == "some" and n % 7 == 3 and c.size:
            c[-1], c[0] = K + 3, -2
    check(K, N, row_ptr, col, vals if N % 2 else vals.astype(np.float32))


# rows of one and of several 4096-column chunks; sparse and dense chunks, both
# in one row, a lane's 64 columns full; more rows than one pass of the scan
@pytest.mark.parametrize("K,N,density,block", [
    (4096, 70, 0.01, None), (4096, 70, 0.1, None), (8320, 33, 0.5, None), (12288, 20, 0.003, (4100, 4164)),
    (12288, 20, 0.003, (4096, 8192)), (64, 20000, 0.02, None), (128, 8193, 0.3, None), (4100, 30, 0.03, (0, 90))])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_pack_csr_entries(gpu, K, N, density, block, dtype):
    from libortho_amd import _C_ops
    g = torch.Generator().manual_seed(K + N)
    mask = torch.rand(N, K, generator=g) < density
    if block:
        mask[::2, block[0]:block[1]] = True
    w = torch.where(mask, torch.randn(N, K, generator=g).to(dtype), torch.zeros((), dtype=dtype))
    row_ptr, col, vals = (t.cpu() for t in _C_ops.pack_csr(w.cuda()))
    at = torch.nonzero(w)
    assert torch.equal(row_ptr[1:].long(), torch.bincount(at[:, 0], minlength=N).cumsum(0)) and row_ptr[0] == 0
    assert torch.equal(col.long(), at[:, 1]) and torch.equal(vals, w[at[:, 0], at[:, 1]])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("group", [None, 128])
def test_pack_nibbles_at_the_halves(gpu, dtype, group):
    """Weights at and beside half steps of their scale, where the quotient's
    last bit decides; scales from the clamp to near the top of the range."""
    from libortho_amd import _C_ops
    K, N = 1024, 600
    g = torch.Generator().manual_seed(3)
    top = {torch.float16: 12.0, torch.bfloat16: 120.0, torch.float32: 120.0}[dtype]
    mx = torch.exp2(torch.rand(N, 1, generator=g) * (top + 18) - 18) * (1 + torch.rand(N, 1, generator=g))
    mx[:7] = torch.tensor([1e-9, 6.9e-6, 7e-6, 7.1e-6, 1.0, 7.0, 14.0])[:, None]
    mx = mx.to(dtype)
    s = (mx.float() * torch.tensor(1.0) / 7).to(dtype)
    w = (s.float() * (torch.randint(-14, 15, (N, K), generator=g) / 2)).to(dtype)
    step = torch.randint(-2, 3, (N, K), generator=g)
    bits = w.view(torch.int32 if dtype == torch.float32 else torch.int16)
    w = torch.where(w != 0, (bits + step.to(bits.dtype)).view(dtype), w)
    w[:, ::128] = mx
    wd = w.cuda()
    cells = wd.float().view(N, -1, group or K)
    amax = cells.abs().amax(-1, keepdim=True)
    scale = torch.clamp((amax * torch.tensor(1.0 / 7, device="cuda")).to(dtype), min=1e-6)
    want = torch.clamp(torch.round((cells / scale.float()).to(dtype).float()), -8, 7).view(N, K).to(torch.int8)
    q, scales = _C_ops.pack_base(wd, group)
    got = torch.stack((q & 15, q >> 4), -1).reshape(N, K).to(torch.int8)
    assert torch.equal((got ^ 8) - 8, want)
    assert torch.equal(scales.view(N, -1), scale.view(N, -1).half())
