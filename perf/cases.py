"""The calls whose speed matters to a program that uses this library: one per
kind of work it does, through the entry points of ``pyc_amd`` and
``pyc_amd.engine``, and generators for more sizes of the same kinds.

A case is a dict of plain values with an "op":

* ``gemm``      half-precision GEMM with the bias + ReLU epilogue, both layouts
                of the right operand (a stored weight [N,K], or the [K,N] of
                the IR's MATMUL);
* ``engine``    fp32 X @ W + bias -> ReLU through pyc_compile_model /
                pyc_run_model on device tensors;
* ``attention`` fused attention forward, causal or not, head dim 64 or 128;
* ``conv``      NHWC convolution with bias + ReLU;
* ``w8``        one decode layer with fp8 weights;
* ``chain``     the decode MLP chain with fp8 weights in one launch;
* ``layernorm``, ``gelu``.

``prepare`` makes what such a program holds before the call, ``run`` is one
call, ``exact`` the same result in float64 by plain torch.
"""
import math

import torch

import pyc_amd
from pyc_amd import abi, engine

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # A large square product with a stored [N,K] weight: the library's
        # benchmark GEMM.
        {"name": "gemm_8192", "op": "gemm", "dtype": "bf16", "layout": "nt", "M": 8192, "N": 8192, "K": 8192,
         "bias": False, "relu": False},
        # Prompt processing through the MLP's up projection (4096 -> 11008, the
        # decode chain's layer) with a [K,N] weight: any number of tokens.
        {"name": "gemm_prefill", "op": "gemm", "dtype": "bf16", "layout": "nn", "M": 1999, "N": 11008, "K": 4096,
         "bias": True, "relu": True},
        # The smallest product of the reference's own benchmark driver:
        # latency of one launch.
        {"name": "gemm_512", "op": "gemm", "dtype": "bf16", "layout": "nn", "M": 512, "N": 512, "K": 512,
         "bias": False, "relu": False},
        # One fused fp32 layer through the run path, compiled once.
        {"name": "engine_f32", "op": "engine", "M": 1024, "N": 1024, "K": 1024},
        # Training-shaped or long-prompt causal attention.
        {"name": "attn_causal", "op": "attention", "dtype": "bf16", "B": 8, "H": 32, "S": 2048, "D": 128,
         "causal": True},
        # Encoder attention of a small batch: few heads, ragged
        # length, no mask, head dim 64.
        {"name": "attn_encoder", "op": "attention", "dtype": "bf16", "B": 2, "H": 16, "S": 1000, "D": 64,
         "causal": False},
        # The stride-1 3x3 body of a ResNet-style stage.
        {"name": "conv_body", "op": "conv", "dtype": "bf16", "N": 32, "H": 56, "W": 56, "C": 256, "K": 256,
         "R": 3, "stride": 1},
        # The stride-2 3x3 between two stages: a smaller batch, few pixels,
        # many channels.
        {"name": "conv_down", "op": "conv", "dtype": "bf16", "N": 16, "H": 28, "W": 28, "C": 512, "K": 512,
         "R": 3, "stride": 2},
        # One fp8 layer for one token of one sequence.
        {"name": "w8_token", "op": "w8", "M": 1, "N": 4096, "K": 11008, "relu": False},
        # Batched decode through eight MLP layers.
        {"name": "w8_chain", "op": "chain", "M": 32, "D": 4096, "F": 11008, "L": 8},
        # Normalisation of a long prompt's hidden states.
        {"name": "layernorm", "op": "layernorm", "dtype": "bf16", "rows": 16384, "D": 4096, "affine": True},
        # The activation of a ragged prompt's MLP.
        {"name": "gelu", "op": "gelu", "dtype": "bf16", "n": 1999 * 11008},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to(v, step):
    return max(step, (v + step // 2) // step * step)


def _ragged(rng, lo, hi, steps):
    """A size over the logarithm of lo..hi, a multiple of one of `steps`."""
    return _to(_log(rng, lo, hi), rng.choice(steps))


def _half(rng):
    return rng.choice(["bf16", "bf16", "bf16", "f16"])


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "engine", "attention", "attention", "conv", "conv", "w8", "chain",
                     "layernorm", "gelu"])
    if op == "gemm":
        # token counts are any number; widths are mostly whole multiples of
        # 64, sometimes of 8 and now and then odd
        return {"op": op, "dtype": _half(rng), "layout": rng.choice(["nt", "nn"]), "M": _log(rng, 16, 4096),
                "N": _ragged(rng, 64, 11008, [256, 64, 64, 8, 1]), "K": _ragged(rng, 64, 8192, [256, 64, 64, 8, 1]),
                "bias": rng.random() < 0.5, "relu": rng.random() < 0.5}
    if op == "engine":
        return {"op": op, "M": _ragged(rng, 64, 3000, [64, 1]), "N": _ragged(rng, 64, 3000, [64, 64, 4, 1]),
                "K": _ragged(rng, 64, 3000, [64, 64, 4, 1])}
    if op == "attention":
        s = _log(rng, 64, 4096)
        heads = min(256, max(1, (1 << 27) // (s * s)))
        return {"op": op, "dtype": _half(rng), "B": rng.randint(1, max(1, heads // 32)),
                "H": rng.choice([8, 12, 16, 32]), "S": s, "D": rng.choice([64, 128]), "causal": rng.random() < 0.6}
    if op == "conv":
        hw = rng.choice([7, 14, 28, 56, rng.randint(7, 60)])
        most = {7: 2048, 14: 1024, 28: 512}.get(hw, 256)
        r = rng.choice([1, 3, 3])
        return {"op": op, "dtype": _half(rng), "N": rng.randint(1, 32), "H": hw, "W": hw,
                "C": _ragged(rng, 16, most, [64, 64, 32, 8]), "K": _ragged(rng, 16, most, [64, 64, 32, 8]),
                "R": r, "stride": rng.choice([1, 1, 2])}
    if op == "w8":
        return {"op": op, "M": rng.choice([1, 1, 2, 4, rng.randint(1, 32), 32]),
                "N": _ragged(rng, 1024, 14336, [64, 64, 8]), "K": _ragged(rng, 1024, 14336, [128, 128, 16]),
                "relu": rng.random() < 0.5}
    if op == "chain":
        return {"op": op, "M": rng.randint(1, 32), "D": _ragged(rng, 1024, 4096, [128, 256]),
                "F": _ragged(rng, 2048, 11008, [128, 256]), "L": rng.randint(1, 8)}
    if op == "layernorm":
        d = _ragged(rng, 256, 8192, [256, 64, 8, 1])
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]),
                "rows": _log(rng, 1, min(16384, (1 << 26) // d)), "D": d, "affine": rng.random() < 0.8}
    return {"op": "gelu", "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "n": _log(rng, 4096, 1 << 25)}


# ---------------------------------------------------------------- inputs


def _gen(seed, k):
    return torch.Generator(device="cuda").manual_seed(1000 * seed + k)


def _randn(shape, seed, k):
    return torch.randn(shape, generator=_gen(seed, k), device="cuda")


def _unif(shape, seed, k):
    return torch.rand(shape, generator=_gen(seed, k), device="cuda")


def _fp8_layer(N, K, seed, k):
    """Weights ~ Normal(0, 2/K), quantised per output channel: e4m3 bytes [N,K]
    and fp32 scales [N]."""
    w = _randn((N, K), seed, k) * math.sqrt(2.0 / K)
    s = (w.abs().amax(1) / 448.0).clamp_min(1e-30)
    return (w / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), s.contiguous()


def _chain_layers(c, seed):
    out = []
    for l in range(c["L"]):
        for j, (n, k) in enumerate([(c["F"], c["D"]), (c["D"], c["F"])]):
            q, s = _fp8_layer(n, k, seed, 10 + 2 * l + j)
            out.append((q, s, j == 0))
    return out


def _inputs(c, seed):
    """The case's input tensors (None for an absent bias)."""
    op = c["op"]
    if op == "gemm":
        t, m, n, k = DT[c["dtype"]], c["M"], c["N"], c["K"]
        a = _randn((m, k), seed, 1).to(t)
        b = (_randn((n, k) if c["layout"] == "nt" else (k, n), seed, 2) / math.sqrt(k)).to(t)
        return a, b, 0.1 * _randn((n,), seed, 3) if c["bias"] else None
    if op == "engine":
        return (_unif((c["M"], c["K"]), seed, 1) * 2 - 1, _unif((c["K"], c["N"]), seed, 2) * 2 - 1,
                _unif((c["N"],), seed, 3) * 2 - 1)
    if op == "attention":
        return tuple(_randn((c["B"], c["H"], c["S"], c["D"]), seed, k).to(DT[c["dtype"]]) for k in (1, 2, 3))
    if op == "conv":
        t, kred = DT[c["dtype"]], c["R"] * c["R"] * c["C"]
        return (_unif((c["N"], c["H"], c["W"], c["C"]), seed, 1).to(t),
                (_randn((c["K"], c["R"], c["R"], c["C"]), seed, 2) * math.sqrt(2.0 / kred)).to(t),
                0.01 * _randn((c["K"],), seed, 3))
    if op == "w8":
        return (_randn((c["M"], c["K"]), seed, 1).to(torch.bfloat16),) + _fp8_layer(c["N"], c["K"], seed, 2)
    if op == "chain":
        return _randn((c["M"], c["D"]), seed, 1).to(torch.bfloat16), _chain_layers(c, seed)
    if op == "layernorm":
        t, d = DT[c["dtype"]], c["D"]
        x = (_randn((c["rows"], d), seed, 1) * 2 + 1).to(t)
        if not c["affine"]:
            return x, None, None
        return x, (1 + 0.2 * _randn((d,), seed, 2)).to(t), (0.2 * _randn((d,), seed, 3)).to(t)
    return (_randn((c["n"],), seed, 1) * 1.5).to(DT[c["dtype"]]),


def _out_hw(c):
    pad = c["R"] // 2
    return (c["H"] + 2 * pad - c["R"]) // c["stride"] + 1


class _Engine:
    """A compiled module and its bound tensors, as a program keeps them."""

    def __init__(self, c, x, w, b):
        m, n, k = c["M"], c["N"], c["K"]
        ops = [engine.op(abi.OP_INPUT, "x", (m, k)), engine.op(abi.OP_INPUT, "w", (k, n)),
               engine.op(abi.OP_INPUT, "bias", (n,)), engine.op(abi.OP_MATMUL, "matmul0", (), (0, 1)),
               engine.op(abi.OP_ADD, "add0", (), (3, 2)), engine.op(abi.OP_RELU, "relu0", (), (4,)),
               engine.op(abi.OP_OUTPUT, "out0", (m, n), (5,))]
        self.model = engine.Model(ops, backend=abi.BACKEND_CUDA)
        if self.model.status != 0:
            raise RuntimeError("pyc_compile_model failed: %d" % self.model.status)
        self.keep = (x, w, b)
        self.y = torch.empty((m, n), dtype=torch.float32, device="cuda")
        self.call = self.model.bind([engine.device_tensor(t, abi.DTYPE_F32) for t in (x, w, b)],
                                    [engine.device_tensor(self.y, abi.DTYPE_F32)])

    def __del__(self):
        self.model.close()


def prepare(case, seed):
    c, x = case, _inputs(case, seed)
    s = {"case": c, "in": x}
    op = c["op"]
    if op == "gemm":
        s["out"] = torch.empty((c["M"], c["N"]), dtype=DT[c["dtype"]], device="cuda")
        s["symbol"] = "hip_gemm_%s_%s" % (c["dtype"], c["layout"])
        s["epi"] = (abi.EPI_BIAS if c["bias"] else 0) | (abi.EPI_RELU if c["relu"] else 0)
    elif op == "engine":
        s["engine"] = _Engine(c, *x)
    elif op == "attention":
        s["out"] = torch.empty_like(x[0])
        s["symbol"] = "hip_attention_" + c["dtype"]
        s["scale"] = 1.0 / math.sqrt(c["D"])
    elif op == "conv":
        p = _out_hw(c)
        s["out"] = torch.empty((c["N"], p, p, c["K"]), dtype=DT[c["dtype"]], device="cuda")
        s["symbol"] = "hip_conv2d_" + c["dtype"]
    elif op == "w8":
        s["out"] = torch.empty((c["M"], c["N"]), dtype=torch.bfloat16, device="cuda")
    elif op == "chain":
        s["out"] = torch.empty((c["M"], c["D"]), dtype=torch.bfloat16, device="cuda")
        pyc_amd.w8a16_chain_reserve(c["M"], x[1])
    else:
        s["out"] = torch.empty_like(x[0])
    return s


def run(state):
    c, x, op = state["case"], state["in"], state["case"]["op"]
    if op == "engine":
        rc, stats = state["engine"].call()
        if rc != 0:
            raise RuntimeError("pyc_run_model failed (%d): %s" % (rc, stats.execution_path.decode()))
        return state["engine"].y
    y = state["out"]
    if op == "gemm":
        pyc_amd.gemm(state["symbol"], x[0], x[1], y, c["M"], c["N"], c["K"], bias=x[2], epilogue=state["epi"])
    elif op == "attention":
        pyc_amd.attention(state["symbol"], x[0], x[1], x[2], y, c["causal"], state["scale"])
    elif op == "conv":
        p, st = c["R"] // 2, c["stride"]
        pyc_amd.conv2d(state["symbol"], x[0], x[1], y, pad=(p, p), stride=(st, st), bias=x[2], relu=True)
    elif op == "w8":
        pyc_amd.w8a16_gemm(x[0], x[1], x[2], y, c["relu"])
    elif op == "chain":
        pyc_amd.w8a16_chain(x[0], x[1], y)
    elif op == "layernorm":
        pyc_amd.layernorm(x[0], y, x[1], x[2])
    else:
        pyc_amd.gelu(x[0], y)
    return y


# ---------------------------------------------------------------- measures


def work(case):
    c, op = case, case["op"]
    if op in ("gemm", "engine"):
        m, n, k = c["M"], c["N"], c["K"]
        e = 4 if op == "engine" else 2
        return {"bytes": e * (m * k + k * n + m * n) + (4 * n if c.get("bias", True) else 0), "flops": 2 * m * n * k}
    if op == "attention":
        s, heads, d = c["S"], c["B"] * c["H"], c["D"]
        pairs = s * (s + 1) // 2 if c["causal"] else s * s
        return {"bytes": 8 * heads * s * d, "flops": 4 * heads * pairs * d}
    if op == "conv":
        p, kred = _out_hw(c), c["R"] * c["R"] * c["C"]
        m = c["N"] * p * p
        # a 1x1 convolution of stride 2 reads a quarter of x
        xs = m * c["C"] if c["R"] == 1 else c["N"] * c["H"] * c["W"] * c["C"]
        return {"bytes": 2 * (xs + c["K"] * kred + m * c["K"]) + 4 * c["K"], "flops": 2 * m * c["K"] * kred}
    if op == "w8":
        m, n, k = c["M"], c["N"], c["K"]
        return {"bytes": n * k + 4 * n + 2 * m * (n + k), "flops": 2 * m * n * k}
    if op == "chain":
        m, d, f, l = c["M"], c["D"], c["F"], c["L"]
        return {"bytes": l * (2 * d * f + 4 * (d + f)) + 4 * m * d, "flops": 4 * l * m * d * f}
    e = DT[c["dtype"]].itemsize
    if op == "layernorm":
        return {"bytes": e * (2 * c["rows"] * c["D"] + (2 * c["D"] if c["affine"] else 0)),
                "flops": 8 * c["rows"] * c["D"]}
    return {"bytes": 2 * e * c["n"], "flops": 20 * c["n"]}


def tolerance(case):
    """About four times the path's distance from `exact`: one rounding of the
    result to its type, and for attention that of the probabilities, for the
    chain that of every layer's activations."""
    op = case["op"]
    if op == "engine":
        return {"rel": 1e-5}
    if op == "chain":
        return {"rel": 2.7e-2}
    if case.get("dtype") == "f32":
        return {"rel": 1e-6}
    if case.get("dtype") == "f16":
        return {"rel": 1.5e-3 if op == "attention" else 1e-3}
    return {"rel": 1e-2 if op == "attention" else 7e-3}


def _attention64(q, k, v, causal):
    B, H, S, D = q.shape
    q, k, v = (t.reshape(B * H, S, D) for t in (q, k, v))
    out = torch.empty((B * H, S, D), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // (S * S))
    mask = torch.ones((S, S), dtype=torch.bool, device=q.device).triu(1) if causal else None
    for h in range(0, B * H, step):
        kt = k[h:h + step].double().transpose(1, 2).contiguous()
        p = torch.bmm(q[h:h + step].double(), kt) / math.sqrt(D)
        if causal:
            p.masked_fill_(mask, -math.inf)
        out[h:h + step] = torch.bmm(torch.softmax(p, -1), v[h:h + step].double())
    return out.reshape(B, H, S, D)


def _conv64(c, x, w, b):
    r, st, p = c["R"], c["stride"], _out_hw(c)
    pad = r // 2
    xp = torch.nn.functional.pad(x.double(), (0, 0, pad, pad, pad, pad))
    y = b.double().expand(c["N"] * p * p, c["K"]).clone()
    for i in range(r):
        for j in range(r):
            tap = xp[:, i:i + st * (p - 1) + 1:st, j:j + st * (p - 1) + 1:st, :].reshape(-1, c["C"])
            y.addmm_(tap, w[:, i, j, :].double().t().contiguous())
    return y.clamp_min_(0).reshape(c["N"], p, p, c["K"])


def _w8_64(x, q, s, relu):
    y = x @ q.view(torch.float8_e4m3fn).double().t().contiguous() * s.double()
    return y.clamp_min(0) if relu else y


def exact(case, seed):
    c, x, op = case, _inputs(case, seed), case["op"]
    if op in ("gemm", "engine"):
        b = x[1].double()
        y = x[0].double() @ (b.t().contiguous() if c.get("layout") == "nt" else b)
        if x[2] is not None:
            y += x[2].double()
        return y.clamp_min_(0) if c.get("relu", True) else y
    if op == "attention":
        return _attention64(*x, c["causal"])
    if op == "conv":
        return _conv64(c, *x)
    if op == "w8":
        return _w8_64(x[0].double(), x[1], x[2], c["relu"])
    if op == "chain":
        h = x[0].double()
        for q, s, relu in x[1]:
            h = _w8_64(h, q, s, relu)
        return h
    v = x[0].double()
    if op == "layernorm":
        d = v - v.mean(-1, keepdim=True)
        y = d / torch.sqrt(d.square().mean(-1, keepdim=True) + 1e-5)
        return y * x[1].double() + x[2].double() if c["affine"] else y
    return 0.5 * v * (1 + torch.erf(v / math.sqrt(2.0)))
