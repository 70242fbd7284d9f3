"""FP32 activations on the matrix cores (orth_float.hip): parity with the FP64
oracle at the edges of its tiles and of its dispatch, against a bound derived
from the FP32 sums it forms."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from libortho_amd import _C_ops, _lib  # noqa: E402
from libortho_amd import workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu


def run(lay, x, alpha, bias=None, wide=False, variant="tiles", policy="auto"):
    d = W.to_device(lay)
    if wide:  # FP32 scales and values
        d["scales"], d["vals"] = d["scales"].float(), d["vals"].float()
    xd = torch.from_numpy(x).cuda()
    y = torch.empty(x.shape[0], lay.N, dtype=torch.float32, device="cuda")
    _lib.set_kernel_policy(policy)
    try:
        _C_ops.forward_planned(d["q"], d["scales"], d["vals"], d["col"], d["row_ptr"], xd, y, alpha, None, bias=bias)
    finally:
        _lib.set_kernel_policy("auto")
    assert (_C_ops.last_kernel(), _C_ops.last_variant()) == ("general", variant)
    return y.cpu().numpy()


def dense64(lay):
    nib = np.stack((lay.q & 15, lay.q >> 4), -1).reshape(lay.N, lay.K).astype(np.int16)
    s = lay.scales.astype(np.float64).reshape(lay.N, -1)
    return ((nib ^ 8) - 8).astype(np.float64) * np.repeat(s, lay.K // s.shape[1], axis=1)


def bound(lay, x, alpha):
    """Each output is a sum of exact products (the activations are split
    without rounding): at most K / 32 * 3 matrix-core additions and K / 64
    scaled ones for the dense part and the row's entries for the sparse part,
    each rounding by at most 2^-23 of the sum of magnitudes so far."""
    w = np.abs(dense64(lay))
    rows = np.repeat(np.arange(lay.N), np.diff(lay.row_ptr))
    np.add.at(w, (rows, lay.col), abs(alpha) * np.abs(lay.vals.astype(np.float64)))
    adds = lay.K / 32 * 3 + lay.K / 64 + max(1, int(np.diff(lay.row_ptr).max())) + 8
    return adds * 2.0 ** -23 * (np.abs(x).astype(np.float64) @ w.T) + 1e-30


def rms_error(y, ref):
    """Against FP64, of the outputs' rms: 1 to 2e-7 for FP32 sums of exact
    products in these kernels' order; activations of two bfloat16 parts in place
    of three would give 3e-6."""
    return np.sqrt(np.mean((y - ref) ** 2) / np.mean(ref ** 2))


# ragged token and row tiles, one K step, odd and even steps per
# scale group, one scale per row over an odd number of steps, 8 / 4 / 2 tokens
# per sparse workgroup (K = 4096, 9216, 11008), more entries per row than one
# batch of loads holds, FP32 scales and values
@pytest.mark.parametrize("K,N,group,M,density,alpha,wide", [
    (4096, 1024, 128, 127, 0.01, 1.0, True), (4096, 1024, 128, 128, 0.01, 1.0, True),
    (4096, 1200, 128, 378, 0.01, 1.0, False), (64, 4650, 64, 65, 0.05, 1.0, False),
    (192, 2333, 192, 129, 0.05, 0.5, False), (320, 1111, None, 130, 0.2, 1.0, True),
    (1024, 1600, 256, 319, 0.0, 1.0, False), (9216, 1000, 128, 253, 0.01, 1.0, False),
    (11008, 1010, 128, 200, 0.02, 1.0, False), (8192, 460, 64, 440, 0.01, 0.0, False)])
def test_float_parity(oracle_mod, K, N, group, M, density, alpha, wide):
    lay = W.make_layer(K, N, group, density, 7000 + K + M)
    x = np.random.Generator(np.random.PCG64(M)).normal(0, 1, (M, K)).astype(np.float32)
    y = run(lay, x, alpha, wide=wide)
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, alpha)
    assert np.isfinite(y).all()
    assert (np.abs(y - ref) <= bound(lay, x, alpha)).all()


def test_float_small_and_large_activations_keep_their_bits(oracle_mod):
    """Magnitudes over 40 binades, values whose 24 bits are all ones."""
    K, N, M = 512, 2400, 130
    lay = W.make_layer(K, N, 128, 0.02, 7100)
    g = np.random.Generator(np.random.PCG64(1))
    x = np.ldexp(np.float32(2) - np.float32(2 ** -23), g.integers(-20, 20, (M, K))).astype(np.float32)
    x *= g.choice([-1.0, 1.0], (M, K)).astype(np.float32)
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    assert (np.abs(run(lay, x, 1.0) - ref) <= bound(lay, x, 1.0)).all()


@pytest.mark.parametrize("M,K,N,G,variant", [(130, 512, 2400, 128, "tiles"), (3, 512, 8200, None, "wave"),
                                             (20, 480, 2400, 32, "wave"), (12, 2048, 4096, 128, "rows"),
                                             (64, 480, 4800, 32, "rows")])
def test_float_products_past_the_range_times_a_scale_within_it(oracle_mod, M, K, N, G, variant):
    """|q x| up to 4.8e38 overflows FP32, scale * q * x does not (tile kernel,
    rows kernel with wide and narrow rows, wave-per-row kernel)."""
    lay = W.make_layer(K, N, G, 0.02, 7300)
    x = np.zeros((M, K), np.float32)
    x[:, ::32] = np.random.Generator(np.random.PCG64(2)).uniform(-6e37, 6e37, (M, K // 32))
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 0.0)
    assert np.abs(ref).max() < 3e38
    y = run(lay, x, 0.0, variant=variant)
    assert np.isfinite(y).all() and (np.abs(y - ref) <= bound(lay, x, 0.0)).all()


@pytest.mark.parametrize("K,N,M,G", [(256, 4400, 70, 128), (64, 2100, 130, None)])
def test_float_scales_near_the_top_of_the_range(oracle_mod, K, N, M, G):
    """FP32 scales past FLT_MAX / 1024 beside ordinary ones, in
    some of the row tiles."""
    lay = W.make_layer(K, N, G, 0.0, 7400)
    x = W.make_x(M, K, 7401).astype(np.float32)
    d = W.to_device(lay)
    s = d["scales"].float()
    big = torch.arange(0, N - 300, 37)
    s[big.cuda()] *= 2.0 ** 123
    y = torch.empty(M, N, dtype=torch.float32, device="cuda")
    _C_ops.forward_planned(d["q"], s, d["vals"].float(), d["col"], d["row_ptr"], torch.from_numpy(x).cuda(), y, 1.0, None)
    assert _C_ops.last_variant() == "tiles"
    y = y.cpu().numpy()
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    err = bound(lay, x, 1.0)
    f = np.ones(N)
    f[big] = 2.0 ** 123
    assert np.abs(s.cpu().numpy()).max() > 3.4e35 and np.abs(ref * f).max() < 3.4e38
    assert np.isfinite(y).all() and (np.abs(y - ref * f) <= err * f).all()


def test_float_infinities_and_nan_stay_with_their_token():
    K, N, M = 256, 4400, 70
    lay = W.make_layer(K, N, 128, 0.02, 7200)
    x = W.make_x(M, K, 7201).astype(np.float32)
    clean = run(lay, x, 1.0)
    x[3, 17], x[5, 40], x[66, 255] = np.inf, np.nan, -np.inf
    x[9, 8] = np.float32(np.frombuffer(np.uint32(0x7f800001).tobytes(), np.float32)[0])  # a NaN of low bits only
    y = run(lay, x, 1.0)
    w = dense64(lay)
    np.add.at(w, (np.repeat(np.arange(N), np.diff(lay.row_ptr)), lay.col), lay.vals.astype(np.float64))
    q = np.stack((lay.q & 15, lay.q >> 4), -1).reshape(N, K)
    for m, k in ((3, 17), (66, 255)):
        plain = (q[:, k] != 0) & (lay.scales.reshape(N, -1)[:, k // 128] != 0)
        plain &= ~np.isin(np.arange(N), np.repeat(np.arange(N), np.diff(lay.row_ptr))[lay.col == k])
        assert np.array_equal(y[m][plain], np.copysign(np.inf, (x[m, k] * w[plain, k])).astype(np.float32))
        assert not np.isfinite(y[m]).any()
    assert np.isnan(y[5]).all() and np.isnan(y[9]).all()
    rest = [m for m in range(M) if m not in (3, 5, 9, 66)]
    assert np.array_equal(y[rest], clean[rest])


def test_float_odd_csr_and_bias(oracle_mod):
    """Duplicate and unsorted columns and columns out of range, as given; the
    bias is added to the finished output."""
    K, N, M = 256, 2150, 140
    lay = W.make_layer(K, N, 128, 0.05, 7300)
    lay.col[:] = lay.col[::-1].copy()
    lay.col[::7] = lay.col[3]
    x = W.make_x(M, K, 7301).astype(np.float32)
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    y = run(lay, x, 1.0)
    assert (np.abs(y - ref) <= bound(lay, x, 1.0)).all()
    bias = torch.randn(N, generator=torch.Generator().manual_seed(5))
    for alpha in (1.0, 0.0):
        got = run(lay, x, alpha, bias=bias.cuda())
        assert np.array_equal(got, run(lay, x, alpha) + bias.numpy()[None, :])
    lay.col[::11] = K + 5
    lay.col[1::11] = -3
    keep = (lay.col >= 0) & (lay.col < K)
    rows = np.repeat(np.arange(N), np.diff(lay.row_ptr))[keep]
    w = dense64(lay)
    np.add.at(w, (rows, lay.col[keep]), lay.vals[keep].astype(np.float64))
    y = run(lay, x, 1.0)
    lay.col[~keep] = 0
    assert (np.abs(y - x.astype(np.float64) @ w.T) <= bound(lay, x, 1.0)).all()


@pytest.mark.parametrize("K,N,M,variant", [(512, 2400, 130, "tiles"), (2048, 4096, 12, "rows")])
def test_the_general_policy_forces_the_wave_per_row_kernel(oracle_mod, K, N, M, variant):
    """Policy "general" takes the kernel that takes every call, also where the
    automatic choice is another of those reported as general."""
    lay = W.make_layer(K, N, 128, 0.02, 7500)
    x = W.make_x(M, K, 7501).astype(np.float32)
    a = run(lay, x, 1.0, variant=variant)
    b = run(lay, x, 1.0, variant="wave", policy="general")
    ref = oracle_mod.forward_f64(lay.q, lay.scales, lay.row_ptr, lay.col, lay.vals, x, 1.0)
    for y in (a, b):
        assert (np.abs(y - ref) <= bound(lay, x, 1.0)).all()
