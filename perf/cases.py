"""The work a user of this framework has it do, as cases that can be timed and checked.

``listed()`` names the calls: serving the packed weights (decode, batched
decode, speculative or chunked prefill, long prefill), fine-tuning through
frozen quantized weights (forward and backward), calibration (Hessians from
hooked layer inputs) and quantization (one small layer, one decoder block).
``draw()`` gives more calls of the same kinds.  ``prepare()`` makes what the
program holds before the call, ``run()`` is the call, ``exact()`` its answer
in 64 bits from plain torch.

Sizes are those of the 8B- and 13B-shaped decoder layers and the 768-wide
layer that this repository's benchmark and tests use, and sizes drawn around
them.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

MAX_WEIGHTS = 28672 * 4096           # the widest layer served (gate and up fused)
MAX_MACS = 2048 * 28672 * 4096       # the longest prefill
MAX_TRAIN_MACS = 1024 * 4096 * 14336


def linear(name, M, N, K, bits, group, dtype, actorder=False, bias=False):
    return {"name": name, "kind": "linear", "M": M, "N": N, "K": K, "bits": bits, "group": group, "dtype": dtype,
            "actorder": actorder, "bias": bias}


def listed():
    return [
        # one token through an attention output projection: the smallest serving call
        linear("decode_m1_o_proj", 1, 4096, 4096, 4, 128, "fp16"),
        # one token through the projections of a stack of 8B-shaped decoder
        # layers (q/k/v and gate/up fused), replayed as a captured graph
        {"name": "decode_graph_8b", "kind": "decode", "M": 1, "layers": 2, "hidden": 4096, "kv": 1024, "ffn": 14336,
         "bits": 4, "group": 128, "dtype": "bf16"},
        # a decode batch of 16 sequences on 3-bit weights
        linear("decode_m16_w3_up_proj", 16, 14336, 4096, 3, 128, "fp16"),
        # a small odd decode batch on an act-order layer of the 13B shape, with a bias
        linear("decode_m5_actorder_13b", 5, 13824, 5120, 4, 128, "bf16", actorder=True, bias=True),
        # a batch on 8-bit per-channel weights (the 13B shape's 8-bit setting)
        linear("batch_m32_w8_13b", 32, 5120, 5120, 8, -1, "fp16"),
        # 128 rows: a speculative or chunked-prefill batch through down_proj
        linear("batch_m128_down_proj", 128, 4096, 14336, 4, 128, "fp16"),
        # one prompt of 2048 tokens through the fused gate/up projection: the largest serving call
        linear("prefill_2048_gate_up", 2048, 28672, 4096, 4, 128, "bf16"),
        # fine-tuning through frozen weights: forward and the gradient of the input
        {"name": "train_1024_down_proj", "kind": "train", "M": 1024, "N": 4096, "K": 14336, "bits": 4, "group": 128,
         "dtype": "bf16", "actorder": False, "bias": False},
        # calibration: eight sequences of 2048 tokens, one hook call each
        {"name": "hessian_16k_k4096", "kind": "hessian", "K": 4096, "N": 4096, "calls": 8, "seqs": 1, "tokens": 2048,
         "dtype": "fp16"},
        # calibration of the widest layer input: four hook calls of eight sequences
        {"name": "hessian_64k_k14336", "kind": "hessian", "K": 14336, "N": 4096, "calls": 4, "seqs": 8,
         "tokens": 2048, "dtype": "bf16"},
        # a small fp32 layer from its Hessian to packed codes
        {"name": "layer_768_fp32", "kind": "layer", "N": 768, "K": 768, "bits": 4, "group": 128, "dtype": "fp32",
         "actorder": False},
        # one 8B-shaped decoder block: seven layers over four Hessians, act-order
        {"name": "block_8b_actorder", "kind": "block", "hidden": 4096, "kv": 1024, "ffn": 14336, "bits": 4,
         "group": 128, "dtype": "bf16", "actorder": True},
    ]


# ------------------------------------------------------------------ draw --

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_dims(rng, wide):
    """Layer sizes: multiples of 128 as models have them, every fourth odd."""
    K = _log_int(rng, 512, 16384)
    N = _log_int(rng, 512, wide)
    if rng.random() < 0.75:
        K, N = max(128, K // 128 * 128), max(128, N // 128 * 128)
    return N, K


def _shrink(value, cost, most, least=1):
    return value if cost <= most else max(least, int(value * most / cost))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["decode", "train", "hessian", "hessian", "layer", "block"])
    bits = rng.choice([2, 3, 4, 4, 4, 8])
    group = rng.choice([64, 128, 128, 128, -1])
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "linear":
        N, K = _draw_dims(rng, 32768)
        N = _shrink(N, N * K, MAX_WEIGHTS)
        M = 1 if rng.random() < 0.2 else _log_int(rng, 2, 4096)
        M = _shrink(M, M * N * K, MAX_MACS)
        case = linear("", M, N, K, bits, group, dtype, actorder=rng.random() < 0.3, bias=rng.random() < 0.3)
        del case["name"]
        return case
    if kind == "decode":
        hidden = rng.choice([2048, 3072, 3584, 4096])
        return {"kind": "decode", "M": rng.choice([1, 1, 2, 4, 7, 16]), "layers": rng.choice([1, 2]),
                "hidden": hidden, "kv": hidden // rng.choice([1, 4, 8]), "ffn": 256 * rng.randint(hidden // 100, 56),
                "bits": rng.choice([3, 4, 4]), "group": 128, "dtype": dtype}
    if kind == "train":
        N, K = _draw_dims(rng, 14336)
        M = _log_int(rng, 64, 4096)
        M = _shrink(M, M * N * K, MAX_TRAIN_MACS)
        return {"kind": "train", "M": M, "N": N, "K": K, "bits": bits, "group": group, "dtype": dtype,
                "actorder": rng.random() < 0.3, "bias": rng.random() < 0.3}
    if kind == "hessian":
        K = _log_int(rng, 512, 14336)
        if rng.random() < 0.75:
            K = K // 64 * 64
        calls, seqs = rng.randint(1, 8), rng.choice([1, 1, 4, 8])
        return {"kind": "hessian", "K": K, "N": 256, "calls": calls, "seqs": seqs,
                "tokens": _log_int(rng, 64, 65536 // (calls * seqs)), "dtype": rng.choice(["fp16", "bf16", "bf16"])}
    if kind == "layer":
        N, K = _draw_dims(rng, 8192)
        return {"kind": "layer", "N": N, "K": min(K, 5120), "bits": bits, "group": group,
                "dtype": rng.choice(["fp16", "bf16", "fp32"]), "actorder": rng.random() < 0.5}
    hidden = 128 * rng.randint(6, 32)
    return {"kind": "block", "hidden": hidden, "kv": hidden // rng.choice([1, 2]), "ffn": 128 * rng.randint(12, 96),
            "bits": rng.choice([3, 4, 8]), "group": rng.choice([64, 128]), "dtype": dtype,
            "actorder": rng.random() < 0.5}


# ---------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _activations(g, shape, dtype):
    """Normalised activations with a few large channels, as layer inputs have them."""
    x = torch.randn(*shape, generator=g, device=DEV)
    K = shape[-1]
    gain = torch.ones(K, device=DEV)
    gain[torch.randperm(K, generator=g, device=DEV)[:max(1, K // 256)]] = 8.0
    return (x * gain).to(dtype)


def _quantized(g, N, K, bits, group, actorder):
    """Codes (N, K), fp16 scales and zero points (N, groups) and g_idx of a
    layer of N(0, 0.02^2) weights, rounded to the nearest code per group."""
    gs = group if 0 < group < K else K
    G = -(-K // gs)
    maxq = 2 ** bits - 1
    w = torch.randn(N, K, generator=g, device=DEV) * 0.02
    pad = G * gs - K
    v = torch.nn.functional.pad(w, (0, pad), value=0.0).view(N, G, gs)
    lo, hi = v.amin(-1).clamp(max=0), v.amax(-1).clamp(min=0)
    s = ((hi - lo) / maxq).clamp(min=1e-8).to(torch.float16)
    z = torch.round(-lo / s.float()).clamp(0, maxq).to(torch.float16)
    q = (torch.round(v / s.float()[..., None]) + z.float()[..., None]).clamp(0, maxq)
    q = q.view(N, G * gs)[:, :K].to(torch.uint8)
    gi = (torch.arange(K, device=DEV) // gs).to(torch.int32)
    if actorder:
        perm = torch.randperm(K, generator=g, device=DEV)
        gi_in, q_in = torch.empty_like(gi), torch.empty_like(q)
        gi_in[perm] = gi
        q_in[:, perm] = q
        gi, q = gi_in, q_in
    return q.contiguous(), s, z, gi, gs


def _bias(g, case, N):
    return torch.randn(N, generator=g, device=DEV) * 0.1 if case.get("bias") else None


def _quantized_linear(g, N, K, bits, group, actorder, bias):
    from distributed_gptq_amd.models import QuantizedLinear
    q, s, z, gi, gs = _quantized(g, N, K, bits, group, actorder)
    layer = QuantizedLinear(bits, gs, K, N, bias=bias is not None, packed=True).to(DEV)
    layer.pack_weights(q, s, z, gi)
    if bias is not None:
        layer.bias.data = bias
    return layer


def _exact_weight(g, N, K, bits, group, actorder):
    q, s, z, gi, _ = _quantized(g, N, K, bits, group, actorder)
    W = q.double()
    gi = gi.long()
    W -= z.double()[:, gi]
    W *= s.double()[:, gi]
    return W


def _decode_layers(case):
    """(name, rows split over the fused layers, in_features) of each projection, in order."""
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    for i in range(case["layers"]):
        yield "%d.qkv" % i, [h, kv, kv], h
        yield "%d.o" % i, [h], h
        yield "%d.gate_up" % i, [f, f], h
        yield "%d.down" % i, [h], f


def _block_layers(case):
    """name -> (rows, Hessian) and Hessian -> in_features of a decoder block."""
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return ({"q": (h, "qkv"), "k": (kv, "qkv"), "v": (kv, "qkv"), "o": (h, "o"), "gate": (f, "up"), "up": (f, "up"),
             "down": (h, "down")}, {"qkv": h, "o": h, "up": h, "down": f})


def _hessian(g, K):
    """Sum of x x^T over 2 K tokens of calibration activations (fp32) and the sequence count."""
    n = 2 * K
    X = _activations(g, (n, K), torch.bfloat16).float()
    H = torch.zeros(K, K, device=DEV)
    for part in X.split(8192):
        H += part.t() @ part
    H = torch.tril(H)
    return H + torch.tril(H, -1).t(), 16


# --------------------------------------------------------------- prepare --

def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind in ("linear", "train"):
        M, N, K = case["M"], case["N"], case["K"]
        dt = DTYPES[case["dtype"]]
        st["x"] = _activations(g, (M, K), dt)
        bias = _bias(g, case, N)
        if kind == "train":
            st["grad"] = torch.randn(M, N, generator=g, device=DEV).mul_(1e-2).to(dt)
            st["x"].requires_grad_(True)
        st["layer"] = _quantized_linear(g, N, K, case["bits"], case["group"], case["actorder"], bias)
        # a loaded model has had a call through each layer
        with torch.no_grad():
            st["layer"](st["x"][:1])
    elif kind == "decode":
        from distributed_gptq_amd.models import FusedQuantizedLinear
        dt = DTYPES[case["dtype"]]
        st["steps"] = []
        for _, rows, K in _decode_layers(case):
            x = _activations(g, (case["M"], K), dt)
            parts = [_quantized_linear(g, N, K, case["bits"], case["group"], False, None) for N in rows]
            st["steps"].append((FusedQuantizedLinear(parts) if len(parts) > 1 else parts[0], x))

        def step():
            with torch.no_grad():
                return [layer(x) for layer, x in st["steps"]]

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            st["y"] = step()
    elif kind == "hessian":
        from distributed_gptq_amd import GPTQ
        dt = DTYPES[case["dtype"]]
        st["make"] = lambda: GPTQ(st["layer"], bits=4, group_size=128, device=torch.device(DEV, 0))
        st["layer"] = nn.Linear(case["K"], case["N"], bias=False, device=DEV, dtype=dt)
        st["xs"] = [_activations(g, (case["seqs"], case["tokens"], case["K"]), dt) for _ in range(case["calls"])]
    elif kind == "layer":
        from distributed_gptq_amd import GPTQ
        N, K = case["N"], case["K"]
        H, ns = _hessian(g, K)
        st["w"] = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(DTYPES[case["dtype"]])
        layer = nn.Linear(K, N, bias=False, device=DEV, dtype=st["w"].dtype)
        st["gptq"] = GPTQ(layer, bits=case["bits"], group_size=case["group"], actorder=case["actorder"],
                          device=torch.device(DEV, 0))
        st["gptq"].H, st["gptq"].nsamples = H, ns
    else:
        layers, hs = _block_layers(case)
        st["hessians"] = {k: _hessian(g, K) for k, K in hs.items()}
        st["weights"] = {n: (torch.randn(N, hs[k], generator=g, device=DEV) * 0.02).to(DTYPES[case["dtype"]])
                         for n, (N, k) in layers.items()}
        st["hkeys"] = {n: k for n, (_, k) in layers.items()}
    return st


# ------------------------------------------------------------------- run --

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        with torch.no_grad():
            return st["layer"](st["x"])
    if kind == "train":
        y = st["layer"](st["x"])
        wrt = [st["x"]] + ([st["layer"].bias] if case["bias"] else [])
        return [y, *torch.autograd.grad(y, wrt, st["grad"])]
    if kind == "decode":
        st["graph"].replay()
        return st["y"]
    if kind == "hessian":
        q = st["make"]()
        for x in st["xs"]:
            q.add_batch(x)
        return q.H
    if kind == "layer":
        q = st["gptq"]
        q.layer.weight.data = st["w"]
        info = q.fasterquant()
        packed = q.pack_native()
        return {"qweight": packed["qweight"], "codes": q.qcodes, "scale": q.scale, "zero": q.zero,
                "weight": q.layer.weight.data, "factor": q.H_inv, "g_idx": q.g_idx, "error": info["total_error"]}
    from distributed_gptq_amd import pipeline
    res = pipeline.quantize_layers(st["weights"], st["hkeys"], st["hessians"], bits=case["bits"],
                                   group_size=case["group"], actorder=case["actorder"])
    return {n: {"codes": r.codes, "qweight": r.qweight, "scale": r.scale, "zero": r.zero, "g_idx": r.g_idx,
                "weight": r.dequant, "loss": r.losses_sum} for n, r in res.items()}


# ---------------------------------------------------- work and tolerance --

def _size(dtype):
    return 4 if dtype == "fp32" else 2


def _layer_bytes(N, K, bits, group):
    gs = group if 0 < group < K else K
    return N * math.ceil(K * bits / 8) + 4 * N * math.ceil(K / gs)


def _gptq_work(K, rows, case):
    """One Hessian's factorisation (Cholesky and triangular inverse) and the
    sweeps of its layers' ``rows`` (each error times the factor's later columns)."""
    out = rows * K * (_size(case["dtype"]) * 2 + 1) + _layer_bytes(rows, K, case["bits"], case["group"])
    return 4 * K * K + out, 2 * K ** 3 / 3 + rows * K * K


def work(case):
    kind = case["kind"]
    if kind in ("linear", "train"):
        M, N, K = case["M"], case["N"], case["K"]
        b = _layer_bytes(N, K, case["bits"], case["group"]) + 2 * M * (N + K) + (4 * N if case["bias"] else 0) + \
            (4 * K if case["actorder"] else 0)
        if kind == "train":
            return {"bytes": b + 2 * M * (N + K), "flops": 4 * M * N * K}
        return {"bytes": b, "flops": 2 * M * N * K}
    if kind == "decode":
        M = case["M"]
        dims = [(sum(rows), K) for _, rows, K in _decode_layers(case)]
        return {"bytes": sum(_layer_bytes(N, K, case["bits"], case["group"]) + 2 * M * (N + K) for N, K in dims),
                "flops": sum(2 * M * N * K for N, K in dims)}
    if kind == "hessian":
        n, K = case["calls"] * case["seqs"] * case["tokens"], case["K"]
        return {"bytes": 2 * n * K + 4 * K * K, "flops": n * K * (K + 1)}
    if kind == "layer":
        b, f = _gptq_work(case["K"], case["N"], case)
        return {"bytes": b + 4 * case["K"] ** 2, "flops": f}
    layers, hs = _block_layers(case)
    each = [_gptq_work(K, sum(N for N, k in layers.values() if k == key), case) for key, K in hs.items()]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "decode", "train"):
        # one rounding of the weight and one of the result to the activations'
        # type; measured against 64 bits: rel 2.9e-4 and max 1.2e-3 in fp16,
        # 2.4e-3 and 1.2e-2 in bf16
        return {"rel": 1.2e-3, "max": 8e-3} if case["dtype"] == "fp16" else {"rel": 1e-2, "max": 6e-2}
    if kind == "hessian":
        # fp32 sums of exact 16-bit products; measured against 64 bits: rel
        # 3e-7 to 7e-7, max 1.5e-5
        return {"rel": 2e-6, "max": 6e-5}
    # Codes are decisions: a weight near the middle between two codes goes the
    # other way in another order of summation, and its row's later columns go
    # with it.  With the Hessian summed in another order none of the 768-wide
    # layer's codes differ and 4 to 13 % of the 8B-shaped block's do, so for
    # wide layers this bound in effect asks for the same sums.
    return {"rel": 0.02, "max": 0.99, "differ": 0.01}


# ----------------------------------------------------------------- exact --

def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("linear", "train"):
        M, N, K = case["M"], case["N"], case["K"]
        dt = DTYPES[case["dtype"]]
        x = _activations(g, (M, K), dt).double()
        bias = _bias(g, case, N)
        gy = torch.randn(M, N, generator=g, device=DEV).mul_(1e-2).to(dt).double() if kind == "train" else None
        W = _exact_weight(g, N, K, case["bits"], case["group"], case["actorder"])
        y = x @ W.t()
        if bias is not None:
            y += bias.double()
        if kind == "linear":
            return y
        return [y, gy @ W] + ([gy.sum(0)] if bias is not None else [])
    if kind == "decode":
        out = []
        for _, rows, K in _decode_layers(case):
            x = _activations(g, (case["M"], K), DTYPES[case["dtype"]]).double()
            ys = tuple(x @ _exact_weight(g, N, K, case["bits"], case["group"], False).t() for N in rows)
            out.append(ys if len(rows) > 1 else ys[0])
        return out
    if kind == "hessian":
        K = case["K"]
        H = torch.zeros(K, K, dtype=torch.float64, device=DEV)
        for _ in range(case["calls"]):
            x = _activations(g, (case["seqs"], case["tokens"], K), DTYPES[case["dtype"]]).reshape(-1, K)
            for part in x.split(8192):
                part = part.double()
                H += part.t().contiguous() @ part
        return H
    if kind == "layer":
        # The upper factor of the damped inverse.  The codes, and what follows
        # from them, have no 64-bit value to be near: a weight halfway between
        # two codes goes either way, and its row's later columns go with it.
        H, ns = _hessian(g, case["K"])
        scl = 2.0 / ns
        if case["actorder"]:
            d = torch.diagonal(H) * scl
            perm = torch.argsort(torch.where(d == 0, torch.ones_like(d), d), descending=True, stable=True)
            H = H[perm][:, perm]
        Hd = H.double().cpu() * scl
        i = torch.arange(case["K"])
        d = Hd[i, i]
        Hd[i, i] = torch.where(d == 0, torch.ones_like(d), d)
        Hd[i, i] += 0.01 * Hd[i, i].mean()
        L = torch.linalg.cholesky(Hd.flip(0, 1))
        U = torch.linalg.solve_triangular(L, torch.eye(case["K"], dtype=torch.float64), upper=False).flip(0, 1)
        return {"qweight": None, "codes": None, "scale": None, "zero": None, "weight": None, "factor": U, "g_idx": None,
                "error": None}
    return None
