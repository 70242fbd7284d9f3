"""Timed cases of the library's public entry points, on one GPU.

``listed()`` holds the fixed cases and ``draw(rng)`` makes one more of the
same ranges.  A case is a dict of plain values; its ``kind`` says which entry
points a pass goes through:

  linear  OrthoLinear.forward, the layer loaded from a packed state_dict
  group   OrthoLinear.forward_group over layers that read one input
  load    OrthoLinear.load_from_weights (packing on the GPU) and the first
          one-token forward after it, which lays the ortho entries out
  sieve   hessian_sieve with a sparsity target: the offline Base/Ortho split

Shapes are the layer shapes of ``libortho_amd.workloads`` (4096 -> 4096,
4096 -> 11008, 4096 -> 14336, 11008 -> 4096), the odd 4000 -> 11008 of the
benchmark's report, and generic powers and multiples between 1024 and 8192;
``group`` is the number of input columns per scale (0: one scale per row, the
layout of checkpoints that know no groups).
"""
import math

import torch

from libortho_amd.tools.sieve import hessian_sieve
from libortho_amd.torch_bind.ortho_linear import OrthoLinear

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# the most work a drawn case may have: that of the largest listed case of its
# path (16-bit activations with in_features a multiple of 64; all others)
_MAX_MNK = 2048 * 4096 * 11008
_MAX_MNK_OTHER = 512 * 4096 * 4096


def _linear(name, K, N, tokens, dtype, group, density, alpha=1.0, bias=False, skewed=False):
    return {"name": name, "kind": "linear", "K": K, "N": N, "tokens": tokens, "dtype": dtype, "group": group,
            "density": density, "alpha": alpha, "bias": bias, "skewed": skewed}


def listed():
    return [
        # one user's token through the widest projection: the smallest call,
        # launch and latency count
        _linear("decode-1", 4096, 11008, 1, "fp16", 128, 0.01),
        # q, k and v of a block for four concurrent users in BF16
        {"name": "qkv-bf16-4", "kind": "group", "K": 4096, "N": 4096, "layers": 3, "tokens": 4, "dtype": "bf16",
         "group": 128, "density": 0.02, "alpha": 1.0},
        # the down projection of a small serving batch in BF16
        _linear("down-bf16-8", 11008, 4096, 8, "bf16", 128, 0.02),
        # gate and up of a block for a serving batch of 32
        {"name": "gate-up-32", "kind": "group", "K": 4096, "N": 11008, "layers": 2, "tokens": 32, "dtype": "fp16",
         "group": 128, "density": 0.02, "alpha": 1.0},
        # a batch of 48 through a sieved layer: the ortho entries in a few
        # outlier columns
        _linear("skewed-48", 4096, 14336, 48, "fp16", 128, 0.005, skewed=True),
        # a short prompt of odd length in BF16, with a bias
        _linear("prompt-bf16-333", 4096, 4096, 333, "bf16", 128, 0.01, bias=True),
        # a long prompt: the largest ordinary call
        _linear("prompt-2048", 4096, 11008, 2048, "fp16", 128, 0.01),
        # FP32 activations (torch's default dtype), a few tokens, per-row scales
        _linear("float-4", 4096, 4096, 4, "fp32", 0, 0.01),
        # an FP32 prompt: evaluation of a packed layer inside an FP32 model
        _linear("float-512", 4096, 4096, 512, "fp32", 128, 0.01),
        # an in_features that no tile divides, per-row scales
        _linear("odd-k-16", 4000, 11008, 16, "fp16", 0, 0.01),
        # packing a split layer at load time, up to its first token
        {"name": "load", "kind": "load", "K": 4096, "N": 11008, "dtype": "fp16", "group": 128, "density": 0.01},
        # splitting one weight matrix offline, 2 % kept in the ortho part
        {"name": "sieve", "kind": "sieve", "K": 4096, "N": 4096, "dtype": "fp32", "target": 0.02},
    ]


_SHAPES = [(4096, 4096), (4096, 11008), (4096, 14336), (11008, 4096), (2048, 2048), (2048, 8192), (8192, 2048),
           (1024, 4096), (5120, 5120), (8192, 1024)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choices(["linear", "group", "load", "sieve"], [16, 3, 2, 2])[0]
    K, N = rng.choice(_SHAPES)
    if rng.random() < 0.25:
        N -= rng.randrange(1, 128)  # an odd number of rows (a shard, a trimmed head)
    dtype = rng.choices(["fp16", "bf16", "fp32"], [5, 4, 2])[0]
    density = rng.choice([0.005, 0.01, 0.02])
    group = rng.choice([128, 128, 128, 0])
    if kind == "load":
        return {"kind": kind, "K": K, "N": N, "dtype": dtype, "group": group, "density": density}
    if kind == "sieve":
        return {"kind": kind, "K": K, "N": N, "dtype": dtype, "target": rng.choice([0.005, 0.01, 0.02, 0.05])}
    alpha = rng.choice([1.0, 1.0, 1.0, 0.5, 0.0])
    if kind == "group":
        return {"kind": kind, "K": K, "N": N, "layers": rng.choice([2, 3]), "tokens": _log_int(rng, 1, 48),
                "dtype": rng.choice(["fp16", "bf16"]), "group": group, "density": density, "alpha": alpha}
    if rng.random() < 0.12:
        K, group = rng.choice([(4000, 0), (1000, 0), (2720, 32)])
    most = _MAX_MNK if dtype != "fp32" and K % 64 == 0 else _MAX_MNK_OTHER
    tokens = _log_int(rng, 1, min(2048, most // (K * N)))
    return {"kind": kind, "K": K, "N": N, "tokens": tokens, "dtype": dtype, "group": group, "density": density,
            "alpha": alpha, "bias": rng.random() < 0.2, "skewed": rng.random() < 0.2}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, sigma=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device="cuda") * sigma).to(dtype)


def _nnz(N, K, density):
    return int(round(density * N * K))


def _ortho_positions(g, N, K, density, skewed):
    """Flat positions of the ortho entries, ascending: as many as the density
    gives (a sieve keeps a fixed number), uniform or all in 1 % of the
    columns."""
    if not skewed:
        return torch.randperm(N * K, generator=g, device="cuda")[:_nnz(N, K, density)].sort().values
    cols = torch.randperm(K, generator=g, device="cuda")[:max(1, int(round(0.01 * K)))].sort().values
    n = cols.numel()
    at = torch.randperm(N * n, generator=g, device="cuda")[:min(N * n, _nnz(N, K, density))].sort().values
    return at // n * K + cols[at % n]


def _packed(g, K, N, group, density, skewed=False):
    """A packed layer's buffers, as a checkpoint holds them."""
    q = torch.randint(0, 256, (N, K // 2), generator=g, device="cuda", dtype=torch.uint8)
    sshape = (N, K // group) if group else (N,)
    scales = _randn(g, sshape, 0.02).abs().clamp(min=1e-6).to(torch.float16)
    at = _ortho_positions(g, N, K, density, skewed)
    rows, cols = at // K, at % K
    vals = _randn(g, (rows.numel(),), 0.2 if skewed else 0.05, torch.float16)
    row_ptr = torch.zeros(N + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=N), 0).to(torch.int32)
    return {"base_weight": q, "base_scales": scales, "ortho_values": vals, "ortho_col_indices": cols.to(torch.int32),
            "ortho_row_ptr": row_ptr}


def _inputs(case, seed):
    """The tensors a case starts from, from the seed alone."""
    g = _gen(seed)
    K, N, kind = case["K"], case["N"], case["kind"]
    dt = _DTYPES[case["dtype"]]
    if kind == "sieve":
        return {"w": _randn(g, (N, K), 0.02, dt),
                "h_inv": (1.0 / (torch.rand(K, generator=g, device="cuda") + 0.05)).to(dt)}
    if kind == "load":
        at = _ortho_positions(g, N, K, case["density"], False)
        w_ortho = torch.zeros(N * K, dtype=dt, device="cuda")
        # away from zero, so that every position is an entry
        w_ortho[at] = _randn(g, (at.numel(),), 0.05).abs().clamp(min=1e-3).to(dt)
        return {"w_base": _randn(g, (N, K), 0.02, dt), "w_ortho": w_ortho.view(N, K),
                "x": _randn(g, (1, K), 1.0, torch.float16)}
    layers = [_packed(g, K, N, case["group"], case["density"], case.get("skewed", False))
              for _ in range(case.get("layers", 1))]
    out = {"layers": layers, "x": _randn(g, (case["tokens"], K), 1.0, dt)}
    if case.get("bias"):
        out["bias"] = _randn(g, (N,), 1.0, dt)
    return out


def prepare(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "sieve":
        return {"kind": kind, "w": inp["w"], "h_inv": inp["h_inv"], "target": case["target"]}
    K, N = case["K"], case["N"]
    group = case["group"] or None
    if kind == "load":
        return {"kind": kind, "layer": OrthoLinear(K, N, group_size=group, device="cuda"), "w_base": inp["w_base"],
                "w_ortho": inp["w_ortho"], "x": inp["x"]}
    mods = []
    for sd in inp["layers"]:
        m = OrthoLinear(K, N, bias=bool(case.get("bias")), dtype=inp["x"].dtype, group_size=group, device="cuda")
        if case.get("bias"):
            sd = dict(sd, bias=inp["bias"])
        m.load_state_dict(sd)
        m.set_alpha(case["alpha"])
        mods.append(m)
    with torch.no_grad():
        for m in mods:  # a loaded model's warm-up token: the ortho layout is made once here
            m(inp["x"][:1])
    return {"kind": kind, "mods": mods, "x": inp["x"]}


def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind == "linear":
            return state["mods"][0](state["x"])
        if kind == "group":
            return OrthoLinear.forward_group(state["mods"], state["x"])
        if kind == "load":
            m = state["layer"]
            m.load_from_weights(state["w_base"], state["w_ortho"])
            y = m(state["x"])
            return {"q": m.base_weight, "scales": m.base_scales, "row_ptr": m.ortho_row_ptr,
                    "col": m.ortho_col_indices, "vals": m.ortho_values, "y": y}
        w_base, w_ortho = hessian_sieve(state["w"], state["h_inv"], sparsity_target=state["target"])
        return {"w_base": w_base, "w_ortho": w_ortho}


# -------------------------------------------------------------- references

def work(case):
    K, N, kind = case["K"], case["N"], case["kind"]
    e = 4 if case["dtype"] == "fp32" else 2
    if kind == "sieve":
        return {"bytes": 3 * e * N * K + e * K, "flops": 8 * N * K}
    groups = K // case["group"] if case["group"] else 1
    weights = N * K // 2 + 2 * N * groups
    nnz = _nnz(N, K, case["density"])
    if kind == "load":
        # both matrices in; the packed weights, the CSR and one token out
        return {"bytes": 2 * e * N * K + weights + 6 * nnz + 4 * (N + 1) + 2 * K + 2 * N,
                "flops": 4 * N * K + 2 * N * K + 2 * nnz}
    M, n = case["tokens"], case.get("layers", 1)
    if case["alpha"] <= 0:
        nnz = 0
    ortho = 6 * nnz + 4 * (N + 1) if nnz else 0
    return {"bytes": n * (weights + ortho + e * M * N) + e * M * K, "flops": n * 2 * M * (N * K + nnz)}


def tolerance(case):
    """Four times the relative error measured against ``exact`` over the
    ranges: the 16-bit output's rounding, and where the weights themselves
    are rounded to the activations' type (batches above 32 tokens) that too;
    32-bit sums in another order for FP32."""
    kind = case["kind"]
    if kind == "sieve":
        return "exact"
    if case["dtype"] == "bf16":  # (the scales of a BF16 weight matrix, for load)
        return {"rel": 7e-3 if kind == "load" else 1e-2}
    if kind == "load":
        return {"rel": 1e-3}
    if case["dtype"] == "fp32":
        return {"rel": 1e-6}
    return {"rel": 1.2e-3 if case["tokens"] > 32 else 1e-3}


def _dense64(sd, K, alpha):
    """The layer's whole matrix, Base + alpha * Ortho, in FP64."""
    q = sd["base_weight"]
    N = q.shape[0]
    nib = torch.stack((q & 0xF, q >> 4), dim=-1).reshape(N, K).to(torch.int16)
    w = ((nib ^ 8) - 8).to(torch.float64)
    s = sd["base_scales"].to(torch.float64).reshape(N, -1)
    w = (w.view(N, s.shape[1], -1) * s.unsqueeze(-1)).view(N, K)
    if alpha > 0:
        rp = sd["ortho_row_ptr"].long()
        rows = torch.repeat_interleave(torch.arange(N, device=q.device), rp[1:] - rp[:-1])
        w.index_put_((rows, sd["ortho_col_indices"].long()), alpha * sd["ortho_values"].to(torch.float64),
                     accumulate=True)
    return w


def exact(case, seed):
    """The outputs of ``run`` in FP64 from plain torch (None for bytes,
    indices and copied values, and for the sieve, whose outputs are selected
    by comparison with a rounded score)."""
    kind = case["kind"]
    if kind == "sieve":
        return None
    inp = _inputs(case, seed)
    K, N = case["K"], case["N"]
    x = inp["x"].to(torch.float64)
    if kind == "load":
        w = inp["w_base"].to(torch.float64)
        G = case["group"] or K
        s = (w.view(N, K // G, G).abs().amax(2) / 7.0).clamp(min=1e-6)
        return {"q": None, "scales": s if case["group"] else s.reshape(N), "row_ptr": None, "col": None, "vals": None,
                "y": None}
    outs = []
    for sd in inp["layers"]:
        y = x @ _dense64(sd, K, case["alpha"]).t()
        if case.get("bias"):
            y = y + inp["bias"].to(torch.float64)
        outs.append(y)
    return outs[0] if kind == "linear" else outs
