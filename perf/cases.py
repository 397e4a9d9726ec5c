"""Performance cases: the decode work a user of this package has it do.

Every case is one call of a public entry point (``decodebench_amd.ops``) or,
for ``layer``, of the decode layer built from them, on inputs that are drawn
from the seed alone.  Kinds:

* ``f1``    RMSNorm -> projection         (``ops.f1_rmsnorm_gemv``)
* ``gemv``  plain projection              (``ops.gemv``)
* ``f2``    gate/up projections + SwiGLU  (``ops.f2_gateup_swiglu``)
* ``f2n``   RMSNorm -> gate/up + SwiGLU   (``ops.f2_rmsnorm_gateup_swiglu``)
* ``f4``    split-KV GQA decode attention (``ops.f4_flashdecode``)
* ``layer`` the decode layer: f1 (QKV), f4, O projection, f2n, down projection

``dtype`` is the weights' type: ``f16``, or ``fp8`` for OCP e4m3 with one fp32
scale per output row.  Activations, KV cache and outputs are fp16.

Ranges: 1 to 64 batch rows, activation widths of 1024 to 8192 (to 14336 for
the plain projection) in steps of 16, 512 to 16384 output rows of any count,
KV lengths of 64 to 32768 with 1, 2, 4 or 8 query heads per KV head.
"""

import math

import torch

from decodebench_amd import ops
from decodebench_amd.demos.llama_decode import layer_fused
from decodebench_amd.quant import quantize_e4m3_rows

D = 128                       # head size
EPS = 1e-6
LAYER = {"d": 4096, "Hq": 32, "Hkv": 8, "F": 14336}
MOST_BYTES = 260_000_000      # of a drawn case, about the largest listed one's
MOST_FLOPS = 16_000_000_000


def _gemv(name, kind, dtype, B, K, N):
    return {"name": name, "kind": kind, "dtype": dtype, "B": B, "K": K, "N": N}


def _f4(name, B, Hq, Hkv, L):
    return {"name": name, "kind": "f4", "B": B, "Hq": Hq, "Hkv": Hkv, "L": L}


def listed():
    return [
        # The smallest call: one token, the square projection of a 2048-wide
        # model; launch and host latency count.
        _gemv("f1_b1_2048", "f1", "f16", 1, 2048, 2048),
        # One token through the QKV projection of a 4096-wide model.
        _gemv("f1_qkv_b1", "f1", "f16", 1, 4096, 6144),
        # One token through the gate/up pair: the largest weights of a layer.
        _gemv("f2_b1", "f2", "f16", 1, 4096, 14336),
        # A serving batch on quantised QKV weights.
        _gemv("f1_qkv_b32_fp8", "f1", "fp8", 32, 4096, 6144),
        # A serving batch through the QKV projection of a 5120-wide model.
        _gemv("f1_b24_k5120", "f1", "f16", 24, 5120, 7168),
        # A small batch on quantised gate/up weights of a 3072-wide model,
        # with an output count that no tile divides.
        _gemv("f2n_b9_k3072_fp8", "f2n", "fp8", 9, 3072, 8201),
        # A large serving batch through the gate/up pair.
        _gemv("f2_b64", "f2", "f16", 64, 4096, 14336),
        # The quantised down projection (long rows) at a small batch.
        _gemv("down_b8_fp8", "gemv", "fp8", 8, 14336, 4096),
        # The down projection of an 11008-wide feed-forward at an odd batch.
        _gemv("down_b41_k11008", "gemv", "f16", 41, 11008, 4096),
        # One user's attention over an ordinary context.
        _f4("f4_b1_l8192", 1, 32, 8, 8192),
        # A serving batch's attention over a context of odd length.
        _f4("f4_b20_l3001", 20, 32, 8, 3001),
        # A whole decode layer for a few users.
        {"name": "layer_b4", "kind": "layer", "dtype": "f16", "B": 4, "L": 2048},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        kind = rng.choice(("f1", "f1", "gemv", "gemv", "f2", "f2n", "f4", "f4", "f4", "layer"))
        dtype = rng.choice(("f16", "fp8"))
        if kind == "layer":
            case = {"kind": kind, "dtype": dtype, "B": _log_int(rng, 1, 8),
                    "L": _log_int(rng, 64, 2048)}
        elif kind == "f4":
            Hkv = rng.choice((2, 4, 8, 8, 16))
            G = rng.choice((1, 2, 4, 4, 8))
            case = {"kind": kind, "B": _log_int(rng, 1, 64), "Hq": Hkv * G, "Hkv": Hkv,
                    "L": _log_int(rng, 64, 32768)}
        else:
            widths = (2048, 3072, 4096, 5120, 8192)
            if kind == "gemv":
                widths += (11008, 14336)
            K = (rng.choice(widths) if rng.random() < 0.6
                 else 16 * _log_int(rng, 64, 896 if kind == "gemv" else 512))
            N = _log_int(rng, 512, 16384)
            if rng.random() < 0.5:
                N = max(512, N // 128 * 128)
            case = {"kind": kind, "dtype": dtype, "B": _log_int(rng, 1, 64), "K": K, "N": N}
        w = work(case)
        # A whole layer's weights alone are more than the bound on bytes.
        if kind == "layer" or (w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS):
            return case


# ------------------------------------------------------------------- inputs
def _randn(gen, *shape, std=1.0, mean=0.0):
    t = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)
    return t.mul_(std).add_(mean).half()


def _weight(gen, N, K, std, dtype):
    """(weights, row scales or None)"""
    W = _randn(gen, N, K, std=std)
    return (W, None) if dtype == "f16" else quantize_e4m3_rows(W)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, B = case["kind"], case["B"]
    if kind == "f4":
        Hq, Hkv, L = case["Hq"], case["Hkv"], case["L"]
        return {"kind": kind, "q": _randn(gen, B, Hq, D), "K": _randn(gen, B, Hkv, L, D),
                "V": _randn(gen, B, Hkv, L, D)}
    if kind == "layer":
        d, Hq, Hkv, F = (LAYER[k] for k in ("d", "Hq", "Hkv", "F"))
        dt = case["dtype"]
        inp = {"x": _randn(gen, B, d), "g1": _randn(gen, d, std=0.1, mean=1.0),
               "g2": _randn(gen, d, std=0.1, mean=1.0),
               "K": _randn(gen, B, Hkv, case["L"], D), "V": _randn(gen, B, Hkv, case["L"], D)}
        for w, s, n, k in (("Wqkv", "s_qkv", (Hq + 2 * Hkv) * D, d), ("Wo", "s_o", d, Hq * D),
                           ("Wg", "s_gate", F, d), ("Wu", "s_up", F, d), ("Wd", "s_down", d, F)):
            inp[w], inp[s] = _weight(gen, n, k, 0.02, dt)
        return {"kind": kind, "inp": inp, "fn": layer_fused(Hq, 1.0 / math.sqrt(D), EPS)}
    K, N, dt = case["K"], case["N"], case["dtype"]
    s = {"kind": kind, "x": _randn(gen, B, K)}
    if kind in ("f1", "f2n"):
        s["g"] = _randn(gen, K, std=0.1, mean=1.0)
    std = 1.0 / math.sqrt(K)
    s["W"], s["s"] = _weight(gen, N, K, std, dt)
    if kind in ("f2", "f2n"):
        s["W2"], s["s2"] = _weight(gen, N, K, std, dt)
    return s


def run(state):
    s, kind = state, state["kind"]
    if kind == "f1":
        return ops.f1_rmsnorm_gemv(s["x"], s["g"], s["W"], EPS, w_scale=s["s"])
    if kind == "gemv":
        return ops.gemv(s["x"], s["W"], w_scale=s["s"])
    if kind == "f2":
        return ops.f2_gateup_swiglu(s["x"], s["W"], s["W2"], s["s"], s["s2"])
    if kind == "f2n":
        return ops.f2_rmsnorm_gateup_swiglu(s["x"], s["g"], s["W"], s["W2"], EPS,
                                            sg=s["s"], su=s["s2"])
    if kind == "f4":
        return ops.f4_flashdecode(s["q"], s["K"], s["V"])
    return s["fn"](s["inp"])


# --------------------------------------------------------------------- work
def work(case):
    """Bytes: weights, scales, cache and activations read once, the output
    written once.  Flops: two per multiply-add of the products."""
    kind, B = case["kind"], case["B"]
    if kind == "f4":
        Hq, Hkv, L = case["Hq"], case["Hkv"], case["L"]
        return {"bytes": 4 * B * Hkv * L * D + 4 * B * Hq * D, "flops": 4 * B * Hq * L * D}
    wb, sb = (2, 0) if case["dtype"] == "f16" else (1, 4)
    if kind == "layer":
        d, Hq, Hkv, F = (LAYER[k] for k in ("d", "Hq", "Hkv", "F"))
        mats = (((Hq + 2 * Hkv) * D, d), (d, Hq * D), (F, d), (F, d), (d, F))
        weights = sum(n * k for n, k in mats)
        nbytes = (weights * wb + sum(n for n, _ in mats) * sb + 4 * B * Hkv * case["L"] * D
                  + 4 * d + 4 * B * d)
        return {"bytes": nbytes, "flops": 2 * B * weights + 4 * B * Hq * case["L"] * D}
    K, N = case["K"], case["N"]
    nw = 2 if kind in ("f2", "f2n") else 1
    gain = 2 * K if kind in ("f1", "f2n") else 0
    return {"bytes": nw * N * (K * wb + sb) + gain + 2 * B * (K + N),
            "flops": 2 * nw * B * N * K}


def tolerance(case):
    """About four times the distance from ``exact`` measured on MI355X, which
    is the fp16 rounding of the outputs and of the intermediates that the
    reference stages round (normalised activations, gate, up and their SiLU,
    attention probabilities); sums are fp32."""
    kind = case["kind"]
    if kind in ("f1", "gemv", "f4"):
        return {"rel": 1.5e-3}
    if kind in ("f2", "f2n"):
        return {"rel": 2.5e-3}
    return {"rel": 4e-3}


# ------------------------------------------------------------ 64-bit results
def _linear64(x, W, s):
    """x . W^T (times the row scales) in 64 bits, in blocks of output rows."""
    y = torch.empty(x.shape[0], W.shape[0], dtype=torch.float64, device=x.device)
    for n in range(0, W.shape[0], 2048):
        y[:, n:n + 2048] = x @ W[n:n + 2048].double().t().contiguous()
    return y if s is None else y * s.double()


def _norm64(x, g):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * g.double()


def _swiglu64(gate, up):
    return gate * torch.sigmoid(gate) * up


def _attention64(q, K, V):
    """q [B,Hq,D], K/V [B,Hkv,L,D], one (batch, KV head) at a time."""
    B, Hq, _ = q.shape
    Hkv = K.shape[1]
    G = Hq // Hkv
    o = torch.empty(B, Hq, D, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(Hkv):
            qh = q[b, h * G:(h + 1) * G].double()
            p = torch.softmax(qh @ K[b, h].double().t().contiguous() / math.sqrt(D), dim=-1)
            o[b, h * G:(h + 1) * G] = p @ V[b, h].double()
    return o


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "f4":
        return _attention64(s["q"], s["K"], s["V"])
    if kind == "layer":
        i, Hq = s["inp"], LAYER["Hq"]
        B = case["B"]
        qkv = _linear64(_norm64(i["x"], i["g1"]), i["Wqkv"], i["s_qkv"])
        attn = _attention64(qkv[:, :Hq * D].reshape(B, Hq, D), i["K"], i["V"])
        h = _norm64(_linear64(attn.reshape(B, Hq * D), i["Wo"], i["s_o"]), i["g2"])
        ff = _swiglu64(_linear64(h, i["Wg"], i["s_gate"]), _linear64(h, i["Wu"], i["s_up"]))
        return _linear64(ff, i["Wd"], i["s_down"])
    x = _norm64(s["x"], s["g"]) if kind in ("f1", "f2n") else s["x"].double()
    y = _linear64(x, s["W"], s["s"])
    return y if kind in ("f1", "gemv") else _swiglu64(y, _linear64(x, s["W2"], s["s2"]))
