"""The rows kernel (orth_rows.hip): FP32 activations in small batches and the
layouts no 128-column chunk or group divides, against the FP64 oracle at the
edges of its tiles, within the rounding of its output plus its FP32 sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from libortho_amd import _C_ops  # noqa: E402
from libortho_amd import workloads as W  # noqa: E402
from tests.test_gpu_float import bound, dense64, rms_error  # noqa: E402

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
EPS = {F16: 2.0 ** -11, BF16: 2.0 ** -8, F32: 0.0}  # half a step of the output, relative
TINY = {F16: 2.0 ** -25, BF16: 0.0, F32: 0.0}  # half of FP16's smallest step (its subnormals')


def within(y, ref, sums, dtype):
    """The FP32 sums' error, then one rounding to dtype."""
    return (np.abs(y - ref) <= sums + np.maximum(EPS[dtype] * (np.abs(ref) + sums), TINY[dtype])).all()


def run(lay, x, alpha, dtype, bias=None, variant="rows"):
    d = W.to_device(lay)
    xd = torch.from_numpy(x).cuda().to(dtype)
    y = torch.empty(x.shape[0], lay.N, dtype=dtype, device="cuda")
    _C_ops.forward_planned(d["q"], d["scales"], d["vals"], d["col"], d["row_ptr"], xd, y, alpha, None, bias=bias)
    assert (_C_ops.last_kernel(), _C_ops.last_variant()) == ("general", variant)
    return y


# 16-byte weight loads with a partial last chunk (K = 4000, 160, 32), words
# (K = 1000, groups of 32, 64 and 96), 1 .. 4 row blocks per pass and several
# passes per workgroup, ragged rows, 1, 2, 15 .. 17 and 40 tokens, fewer
# tokens per LDS tile at large K, waves without a chunk, rows of more than 64
# entries, no ortho term
@pytest.mark.parametrize("K,N,group,M,density,dtype", [
    (4000, 4096, None, 2, 0.01, F16), (4000, 4099, None, 16, 0.01, F16), (4000, 8200, None, 17, 0.01, BF16),
    (4000, 11008, None, 1, 0.01, F16), (4000, 3000, None, 15, 0.05, BF16), (4000, 16500, None, 3, 0.005, F16),
    (160, 33000, None, 40, 0.0, F16), (32, 9001, None, 5, 0.3, BF16), (1000, 4096, None, 16, 0.02, F16),
    (1000, 12000, None, 40, 0.1, BF16), (2720, 1700, 32, 16, 0.01, F16), (2720, 9000, 32, 4, 0.01, BF16),
    (960, 2048, 96, 15, 0.02, F16), (448, 13000, 64, 2, 0.02, BF16), (4096, 4096, 128, 4, 0.01, F32),
    (4096, 2100, 128, 16, 0.02, F32), (4096, 8191, None, 17, 0.01, F32), (11008, 4096, 128, 7, 0.01, F32),
    (4000, 4100, None, 9, 0.02, F32), (2720, 4100, 32, 9, 0.02, F32), (1000, 13000, None, 2, 0.02, F32),
    (2720, 9000, 32, 17, 0.01, BF16), (448, 13000, 64, 16, 0.02, BF16), (1000, 13000, None, 16, 0.02, F32),
    (16384, 1030, 256, 16, 0.005, F32)])
def test_rows_parity(gpu, oracle_mod, K, N, group, M, density, dtype):
    lay = W.make_layer(K, N, group, density, 7500 + K + M)
    x = torch.from_numpy(W.make_x(M, K, 7501 + M)).to(dtype).float().numpy()
    if dtype == F32:
        x = np.random.Generator(np.random.PCG64(M)).normal(0, 1, (M, K)).astype(np.float32)
    small = (K, M) in ((448, 2), (1000, 2), (2720, 4))  # (left to the wave-per-row kernel)
    for alpha in (1.0, 0.0):
        y = run(lay, x, alpha, dtype, variant="wave" if small else "rows").float().cpu().numpy()
        ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, alpha)
        sums = bound(lay, x, alpha)
        assert within(y, ref, sums, dtype)
        if dtype == F32:
            assert rms_error(y, ref) <= 5e-7


# either side of the choice's lines, in calls whose times are well apart:
# few and many tokens, entries and columns, wide and narrow rows, FP32 scales
@pytest.mark.parametrize("K,N,group,M,density,dtype,variant", [
    (4096, 4096, 128, 4, 0.01, F32, "rows"), (4096, 4096, 128, 64, 0.01, F32, "rows"),
    (4096, 4096, 128, 128, 0.01, F32, "tiles"), (8192, 1024, 128, 128, 0.01, F32, "rows"),
    (1024, 1024, 128, 4, 0.01, F32, "wave"), (1024, 1024, 128, 16, 0.2, F32, "wave"),
    (28672, 1024, 128, 24, 0.0, F32, "wave"), (1344, 11008, 96, 4, 0.0, F16, "wave"),
    (1344, 11008, 96, 16, 0.0, F16, "rows"), (4000, 11008, None, 1, 0.01, BF16, "rows"),
    (30000, 1024, None, 48, 0.02, F16, "wave")])
def test_general_choice(gpu, oracle_mod, K, N, group, M, density, dtype, variant):
    lay = W.make_layer(K, N, group, density, 7900 + K)
    x = torch.from_numpy(W.make_x(M, K, 7901)).to(dtype).float().numpy()
    y = run(lay, x, 1.0, dtype, variant=variant).float().cpu().numpy()
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    assert within(y, ref, bound(lay, x, 1.0), dtype)


@pytest.mark.parametrize("dtype", [F16, BF16, F32])
def test_rows_odd_csr_bias_and_infinities(gpu, oracle_mod, dtype):
    """Duplicate, unsorted and out-of-range columns as given; the bias added
    to the rounded output; an infinity or a NaN stays with its token."""
    K, N, M = 480, 5000, 12
    lay = W.make_layer(K, N, None, 0.05, 7600)
    lay.col[:] = lay.col[::-1].copy()
    lay.col[::7] = lay.col[3]
    x = torch.from_numpy(W.make_x(M, K, 7601)).to(dtype).float().numpy()
    y = run(lay, x, 1.0, dtype)
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    sums = bound(lay, x, 1.0)
    assert within(y.float().cpu().numpy(), ref, sums, dtype)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(5)).cuda()
    want = (y.double() + bias.double()).float().to(dtype)  # (exact in FP64, one rounding through FP32 as the store's)
    got = run(lay, x, 1.0, dtype, bias=bias)
    assert torch.equal(got, (y.float() + bias).to(dtype)) or torch.equal(got, want)
    bad = x.copy()
    bad[1, 5], bad[4, 479] = np.inf, np.nan
    z = run(lay, bad, 1.0, dtype)
    keep = [m for m in range(M) if m not in (1, 4)]
    assert torch.equal(z[keep], y[keep]) and torch.isnan(z[4]).all() and not torch.isfinite(z[1]).any()
    lay.col[::11] = K + 5
    lay.col[1::11] = -3
    ok = (lay.col >= 0) & (lay.col < K)
    w = dense64(lay)
    np.add.at(w, (np.repeat(np.arange(N), np.diff(lay.row_ptr))[ok], lay.col[ok]), lay.vals[ok].astype(np.float64))
    y = run(lay, x, 1.0, dtype).float().cpu().numpy()
    lay.col[~ok] = 0
    ref, sums = x.astype(np.float64) @ w.T, bound(lay, x, 1.0)
    assert within(y, ref, sums, dtype)
