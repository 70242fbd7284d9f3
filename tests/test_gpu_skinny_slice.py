"""The split-K mid-batch kernel's ortho term as a slice of its own (17 .. 64
tokens): against the FP64 oracle where its token tiles, units of rows, batches
of entries and dispatch end, with and without a plan."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from libortho_amd import _C_ops, _lib  # noqa: E402
from libortho_amd import workloads as W  # noqa: E402
from tests.test_gpu_float import bound  # noqa: E402

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}  # half a step of the output, relative
TINY = {torch.float16: 2.0 ** -25, torch.bfloat16: 0.0}       # half of FP16's smallest step


def run(lay, x, alpha, dtype, plan=False, bias=None, policy="skinny"):
    d = W.to_device(lay)
    xd = torch.from_numpy(x).cuda().to(dtype)
    y = torch.empty(x.shape[0], lay.N, dtype=dtype, device="cuda")
    p = _C_ops.build_plan(d["q"], d["scales"], d["vals"], d["col"], d["row_ptr"], lay.K) if plan else None
    _lib.set_kernel_policy(policy)
    try:
        _C_ops.forward_planned(d["q"], d["scales"], d["vals"], d["col"], d["row_ptr"], xd, y, alpha, p, bias=bias)
    finally:
        _lib.set_kernel_policy("auto")
    return y, _C_ops.last_kernel()


def check(oracle_mod, lay, x, alpha, dtype, y):
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, alpha)
    # (the weights' bias, up to 136 q + 136 q for a weight q, is formed and
    # removed in FP32: sums of up to 18 times the magnitudes counted here)
    sums = 18 * bound(lay, x, alpha)
    err = np.abs(y.float().cpu().numpy() - ref)
    assert (err <= sums + np.maximum(EPS[dtype] * (np.abs(ref) + sums), TINY[dtype])).all()


def check_ortho(oracle_mod, lay, x, alpha, dtype, **kw):
    """With scales of zero the output is the ortho term alone (the dense sums
    are multiplied by 0), its bound that of its own few sums: one entry of a
    row left out or taken twice is far outside it."""
    scales = lay.scales.copy()
    lay.scales[:] = 0
    y, _ = run(lay, x, alpha, dtype, **kw)
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, alpha)
    sums = bound(lay, x, alpha)
    one = alpha * np.sqrt(np.mean(lay.vals.astype(np.float64) ** 2) * np.mean(x.astype(np.float64) ** 2))
    assert np.median(sums + EPS[dtype] * np.abs(ref)) < 0.2 * one  # (what one entry adds, rms)
    err = np.abs(y.float().cpu().numpy() - ref)
    assert (err <= sums + np.maximum(EPS[dtype] * (np.abs(ref) + sums), TINY[dtype])).all()
    lay.scales[:] = scales


# two, three and four token tiles, the last 8 (4, 2) tokens ragged, rows that
# end inside a unit, rows with more entries than one batch of loads, tiles of 8
# tokens (K <= 8192), 4 and 2, one scale per row
@pytest.mark.parametrize("K,N,group,M,density,dtype", [
    (4096, 1000, 128, 17, 0.01, torch.float16), (4096, 3001, 128, 33, 0.02, torch.bfloat16),
    (2048, 2000, None, 48, 0.05, torch.float16), (4096, 1040, 256, 64, 0.005, torch.float16),
    (8192, 500, 128, 41, 0.01, torch.bfloat16), (11008, 700, 128, 20, 0.02, torch.float16),
    (16768, 130, 128, 35, 0.01, torch.float16), (256, 5000, 128, 64, 0.3, torch.bfloat16)])
def test_skinny_slice_parity(gpu, oracle_mod, K, N, group, M, density, dtype):
    lay = W.make_layer(K, N, group, density, 8900 + K + M)
    x = torch.from_numpy(W.make_x(M, K, 8901 + M)).to(dtype).float().numpy()
    y, k = run(lay, x, 0.5, dtype)
    assert k == "skinny"
    check(oracle_mod, lay, x, 0.5, dtype, y)
    z, _ = run(lay, x, 0.5, dtype, plan=K <= 12288)
    if K == 11008:  # (with a plan each lane finds its own entries)
        check(oracle_mod, lay, x, 0.5, dtype, z)
        check_ortho(oracle_mod, lay, x, 0.5, dtype, plan=True)
    else:
        assert torch.equal(y, z)  # (it reads no plan)
    check_ortho(oracle_mod, lay, x, 0.5, dtype)


@pytest.mark.parametrize("K,N,M,density,dtype", [
    (4096, 1000, 33, 0.2, torch.float16), (4096, 2100, 64, 0.1, torch.bfloat16), (1152, 9000, 49, 0.2, torch.float16)])
def test_many_planned_entries(gpu, oracle_mod, K, N, M, density, dtype):
    """17 .. 64 tokens with a plan and so many entries that each lane finds its
    own: the same results as from the workgroups that take them without one,
    to the rounding of sums in another order."""
    lay = W.make_layer(K, N, 128, density, 9300 + K)
    x = torch.from_numpy(W.make_x(M, K, 9301 + M)).to(dtype).float().numpy()
    for plan in (True, False):
        y, k = run(lay, x, 1.0, dtype, plan=plan)
        assert k == "skinny"
        check(oracle_mod, lay, x, 1.0, dtype, y)
        check_ortho(oracle_mod, lay, x, 1.0, dtype, plan=plan)


@pytest.mark.parametrize("K,N,M,density,dtype", [
    (4096, 1000, 33, 0.2, torch.float16), (4096, 2100, 64, 0.1, torch.bfloat16), (1152, 9000, 49, 0.2, torch.float16),
    (8192, 1000, 17, 0.05, torch.bfloat16)])
def test_many_planned_entries_out_of_order(gpu, oracle_mod, K, N, M, density, dtype):
    """The same with columns that do not ascend, which the plan does not locate:
    the workgroups take them as without a plan (bit for bit where they hold the
    same 8 tokens), not each lane its whole row."""
    lay = W.make_layer(K, N, 128, density, 9400 + K)
    lay.col[:] = lay.col[::-1].copy()
    x = torch.from_numpy(W.make_x(M, K, 9401 + M)).to(dtype).float().numpy()
    y, k = run(lay, x, 1.0, dtype, plan=True)
    z, _ = run(lay, x, 1.0, dtype)
    assert k == "skinny"
    check(oracle_mod, lay, x, 1.0, dtype, y)
    check_ortho(oracle_mod, lay, x, 1.0, dtype, plan=True)
    if M >= 49:
        assert torch.equal(y, z)


def test_skinny_slice_odd_csr_infinities_and_bias(gpu, oracle_mod):
    K, N, M = 1024, 777, 50
    lay = W.make_layer(K, N, 128, 0.05, 9000)
    lay.col[:] = lay.col[::-1].copy()
    lay.col[::7] = lay.col[3]
    x = W.make_x(M, K, 9001).astype(np.float32)
    y, _ = run(lay, x, 1.0, torch.float16)
    check(oracle_mod, lay, x, 1.0, torch.float16, y)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)).cuda()
    b, _ = run(lay, x, 1.0, torch.float16, bias=bias)
    assert torch.equal(b, (y.float() + bias).half())
    bad = x.copy()
    bad[7, 5], bad[20, 1023] = np.inf, np.nan
    z, _ = run(lay, bad, 1.0, torch.float16)
    keep = [m for m in range(M) if m not in (7, 20)]
    assert torch.equal(z[keep], y[keep])
    lay.col[::11], lay.col[1::13] = K + 5, -3
    ok = (lay.col >= 0) & (lay.col < K)
    y, _ = run(lay, x, 1.0, torch.float16)
    lay.col[~ok], lay.vals[~ok] = 0, 0
    check(oracle_mod, lay, x, 1.0, torch.float16, y)


@pytest.mark.parametrize("K,N,M,density,dtype,plan", [
    (2048, 600, 5, 0.02, torch.float16, True), (1152, 600, 8, 0.1, torch.bfloat16, False),
    (11008, 300, 9, 0.02, torch.bfloat16, True), (2048, 600, 16, 0.05, torch.float16, False)])
def test_one_token_tile_transposed_copy(gpu, oracle_mod, K, N, M, density, dtype, plan):
    """5 .. 16 tokens, 8 or 16 a column, slices of fewer than 8 chunks and a
    narrower last one, from the records and from the CSR: parity, and an
    infinity or a NaN (also under an empty entry's column) stays with its token."""
    lay = W.make_layer(K, N, 128, density, 9200 + K)
    x = torch.from_numpy(W.make_x(M, K, 9201 + M)).to(dtype).float().numpy()
    y, k = run(lay, x, 1.0, dtype, plan=plan)
    assert k == "skinny"
    check(oracle_mod, lay, x, 1.0, dtype, y)
    check_ortho(oracle_mod, lay, x, 1.0, dtype, plan=plan)
    bad = x.copy()
    bad[1, 0], bad[M - 1, K - 1] = np.inf, np.nan
    z, _ = run(lay, bad, 1.0, dtype, plan=plan)
    keep = [m for m in range(M) if m not in (1, M - 1)]
    assert torch.equal(z[keep], y[keep]) and torch.isnan(z[M - 1]).all()


@pytest.mark.parametrize("K,N,M,density,alpha,kernel", [
    (8192, 1024, 33, 0.01, 1.0, "skinny"), (8320, 1024, 33, 0.01, 1.0, "prefill"),
    (8192, 2048, 64, 0.03, 1.0, "prefill"),          # entries x tokens past 27 million
    (5120, 512, 33, 0.03, 1.0, "skinny"), (5120, 512, 33, 0.04, 1.0, "prefill"),  # 1 entry in 32
    (11008, 1024, 64, 0.01, 0.0, "skinny"), (11008, 1024, 64, 0.01, 1.0, "prefill")])
def test_wide_k_dispatch(gpu, oracle_mod, K, N, M, density, alpha, kernel):
    lay = W.make_layer(K, N, 128, density, 9100 + K)
    x = W.make_x(M, K, 9101).astype(np.float32)
    y, k = run(lay, x, alpha, torch.float16, plan=True, policy="auto")
    assert k == kernel
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, alpha)
    assert np.abs(y.float().cpu().numpy() - ref).max() <= 2e-3 * np.abs(ref).max()
