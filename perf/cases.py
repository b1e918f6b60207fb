"""Timed cases of the low-bit path: the calls a program that trains or serves with this package makes.

Nine kinds of call, each through a public entry point of ``lowbit``:

  linear_fwd     HipLowBitBackend.linear without gradients: activation and weight quantized in the call, then the
                 blockwise-scaled product (an evaluation or generation step of a `--fp8 --fp8-backend hip` model)
  linear_train   the same linear forward and its straight-through backward (a training step of one Linear)
  recipe_train   the linear with the quantized dgrad / wgrad recipe (`--lowbit-backward fp8`)
  stored_linear  a product with a weight stored as NF4 (64-weight blocks), MXFP4 or persistent FP8
  stored_train   Linear with a persistent low-bit weight: forward, and the gradients of input, weight and bias
  moe_fwd        local_moe_forward: the routed expert loop of one rank over quantized expert weights
  moe_train      local_moe forward and backward over bf16 expert weights
  refresh        quantize_nf4_persistent / quantize_fp8_persistent of a weight (after each optimizer step)
  comm           comm_quant_dequant of a dispatch payload, to nearest or with seeded stochastic rounding

All tensors are bf16, the dtype of the path.  Every case is made from its seed on the GPU.
"""

from __future__ import annotations

import argparse
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-train_amd"))

BF16 = torch.bfloat16
DEV = "cuda"

# the largest listed case (the 4096-token expert training step) bounds what a drawn case may cost
MAX_FLOPS = 8.7e12
MAX_BYTES = 6.0e9


def listed():
    return [
        # a generation step: 16 sequences through a 4096-wide projection, the default int grid
        dict(name="linear_fwd_16", kind="linear_fwd", M=16, N=4096, K=4096, fmt="int_grid", bias=False),
        # the small benchmark Linear: 512 tokens with outliers, 1024 wide
        dict(name="linear_fwd_512", kind="linear_fwd", M=512, N=1024, K=1024, fmt="e4m3", bias=True),
        # a training step of a small model's Linear whose sizes are no multiples of anything
        dict(name="linear_train_odd", kind="linear_train", M=1003, N=1541, K=1000, fmt="int_grid", bias=True),
        # the DeepSeek-V3 dense MLP up-projection, forward and straight-through backward at 8192 tokens
        dict(name="linear_train_8192", kind="linear_train", M=8192, N=18432, K=7168, fmt="e4m3", bias=False),
        # the quantized backward recipe at an ordinary width and microbatch
        dict(name="recipe_train_2048", kind="recipe_train", M=2048, N=4096, K=4096, fmt="e4m3", bias=True),
        # generation from a stored NF4 weight: 4 sequences
        dict(name="nf4_linear_4", kind="stored_linear", M=4, N=14336, K=4096, fmt="nf4"),
        # prefill from the same stored weight: 4096 tokens
        dict(name="nf4_linear_4096", kind="stored_linear", M=4096, N=14336, K=4096, fmt="nf4"),
        # a training step of a Linear with a persistent FP8 weight
        dict(name="fp8_layer_train_2048", kind="stored_train", M=2048, N=8192, K=2048, fmt="fp8", bias=True),
        # the expert loop while generating: 32 tokens, top 8 of 32 experts
        dict(name="moe_fwd_32", kind="moe_fwd", T=32, H=7168, I=2048, E=32, k=8, fmt="e4m3"),
        # the expert loop's training step at 4096 tokens
        dict(name="moe_train_4096", kind="moe_train", T=4096, H=7168, I=2048, E=32, k=8, fmt="e4m3"),
        # re-quantization of a persistent NF4 weight after an optimizer step, one scale per row
        dict(name="nf4_refresh", kind="refresh", N=14336, K=4096, fmt="nf4"),
        # stochastic comm-quant of a dispatch payload of an odd number of rows
        dict(name="comm_5001", kind="comm", M=5001, K=7168, rounding="stochastic"),
    ]


def _size(rng, lo: int, hi: int, mult: int = 1) -> int:
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(mult, (v + mult // 2) // mult * mult)


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


def _draw(rng):
    kind = rng.choice(("linear_fwd", "linear_fwd", "linear_train", "recipe_train", "stored_linear", "stored_linear",
                       "stored_train", "moe_fwd", "moe_train", "refresh", "comm"))
    if kind in ("linear_fwd", "linear_train", "recipe_train"):
        lo = 1 if kind == "linear_fwd" else 64
        m = rng.choice((1, 64, 128))  # model widths are round; tests and small models use odd ones too
        return dict(kind=kind, M=_size(rng, lo, 8192), N=_size(rng, 256, 18432, m), K=_size(rng, 256, 7168, m),
                    fmt=rng.choice(("int_grid", "e4m3")), bias=rng.random() < 0.5)
    if kind == "stored_linear":
        return dict(kind=kind, M=_size(rng, 1, 8192), N=_size(rng, 256, 18432, rng.choice((1, 64))),
                    K=_size(rng, 256, 8192, 64), fmt=rng.choice(("nf4", "mxfp4", "fp8")))
    if kind == "stored_train":
        return dict(kind=kind, M=_size(rng, 64, 8192), N=_size(rng, 256, 14336, rng.choice((4, 64))),
                    K=_size(rng, 256, 8192, rng.choice((4, 64, 64))), fmt=rng.choice(("nf4", "fp8")),
                    bias=rng.random() < 0.5)
    if kind in ("moe_fwd", "moe_train"):
        k = rng.choice((1, 2, 4, 8))
        return dict(kind=kind, T=_size(rng, 1 if kind == "moe_fwd" else 64, 4096), H=_size(rng, 512, 7168, 128),
                    I=_size(rng, 256, 2048, 128), E=max(k, _size(rng, 4, 32)), k=k,
                    fmt=rng.choice(("int_grid", "e4m3")))
    if kind == "refresh":
        return dict(kind=kind, N=_size(rng, 64, 18432), K=_size(rng, 256, 8192, rng.choice((8, 64))),
                    fmt=rng.choice(("nf4", "fp8")))
    return dict(kind=kind, M=_size(rng, 1, 16384), K=_size(rng, 256, 8192, rng.choice((1, 128))),
                rounding=rng.choice(("nearest", "stochastic")))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _normal(g, shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(BF16)


def _activation(g, rows, cols):
    """N(0,1) with 1% of the entries scaled x50 (the benchmark's outliers)"""
    x = torch.randn(rows, cols, generator=g, device=DEV)
    return torch.where(torch.rand(rows, cols, generator=g, device=DEV) < 0.01, x * 50.0, x).to(BF16)


def _inputs(c, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = c["kind"]
    if kind in ("linear_fwd", "linear_train", "recipe_train", "stored_train", "stored_linear"):
        M, N, K = c["M"], c["N"], c["K"]
        t = dict(x=_activation(g, M, K), w=_normal(g, (N, K), 0.02),
                 b=_normal(g, (N,), 0.1) if c.get("bias") else None)
        if kind != "linear_fwd" and kind != "stored_linear":
            t["dy"] = _normal(g, (M, N), 1e-3)
        return t
    if kind in ("moe_fwd", "moe_train"):
        T, H, I, E, k = c["T"], c["H"], c["I"], c["E"], c["k"]
        # Zipf(1.2) expert popularity, distinct experts per token (Gumbel top-k)
        logp = -1.2 * torch.log(torch.arange(1, E + 1, dtype=torch.float64, device=DEV))
        u = torch.rand(T, E, generator=g, device=DEV, dtype=torch.float64).clamp(1e-12, 1 - 1e-12)
        score, ids = torch.topk(logp - torch.log(-torch.log(u)), k, dim=1)
        t = dict(x=_normal(g, (T, H)), ids=ids, tw=torch.softmax(score, dim=1).to(BF16),
                 gate=_normal(g, (E, I, H), 0.006), up=_normal(g, (E, I, H), 0.006),
                 down=_normal(g, (E, H, I), 0.006))
        if kind == "moe_train":
            t["dy"] = _normal(g, (T, H), 1e-3)
        return t
    if kind == "refresh":
        return dict(w=_normal(g, (c["N"], c["K"]), 0.02))
    return dict(x=_activation(g, c["M"], c["K"]))


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------

def _resolver(**flags):
    from lowbit.precision import add_mixed_precision_args, build_module_precision_resolver, resolve_precision_config

    parser = argparse.ArgumentParser()
    add_mixed_precision_args(parser)
    ns = parser.parse_args([])
    for key, value in flags.items():
        setattr(ns, key, value)
    return build_module_precision_resolver(resolve_precision_config(ns, torch.device("cuda", 0)))


def prepare(case, seed):
    from lowbit import moe
    from lowbit import persistent as P
    from lowbit.backend import HipLowBitBackend
    from lowbit.contracts import LowBitKernelSpec
    from lowbit.layers import Linear

    kind = case["kind"]
    t = _inputs(case, seed)
    s = dict(kind=kind, case=case)
    if kind in ("linear_fwd", "linear_train", "recipe_train"):
        spec = LowBitKernelSpec("linear", case["K"], case["N"], t["b"] is not None, "tile_1x128", "block_128x128",
                                "nearest")
        s["backend"] = HipLowBitBackend(mode="fp8", kernel_spec=spec, code_format=case["fmt"], seed=1,
                                        backward="fp8" if kind == "recipe_train" else "ste")
        if kind != "linear_fwd":
            for name in ("x", "w", "b"):
                if t[name] is not None:
                    t[name].requires_grad_(True)
        s.update(t)
    elif kind == "stored_linear":
        s["x"] = t["x"]
        if case["fmt"] == "nf4":
            s["codes"], s["scales"] = P.quantize_nf4_blocks(t["w"], 64)
        elif case["fmt"] == "mxfp4":
            s["codes"], s["scales"] = P.quantize_mxfp4(t["w"])
        else:
            s["codes"], s["scales"] = P.quantize_fp8_persistent(t["w"], granularity="per_channel")
    elif kind == "stored_train":
        flags = dict(bf16=True, persistent_lowbit_include=["fc"])
        flags["fp4_param" if case["fmt"] == "nf4" else "fp8_param"] = True
        layer = Linear(case["K"], case["N"], t["b"] is not None, param_dtype=BF16,
                       param_device=torch.device("cuda", 0), module_path="decoder.blocks.0.mlp.fc1",
                       precision_resolver=_resolver(**flags))
        with torch.no_grad():
            layer.weight.copy_(t["w"])
            if t["b"] is not None:
                layer.bias.copy_(t["b"])
        layer.refresh_persistent_lowbit_params()
        s.update(layer=layer, x=t["x"].requires_grad_(True), dy=t["dy"])
    elif kind == "moe_fwd":
        fmt = case["fmt"]
        s["gate_up"] = moe.quantize_expert_weights(moe.stack_gate_up(t["gate"], t["up"]), fmt=fmt)
        s["down"] = moe.quantize_expert_weights(t["down"], fmt=fmt)
        s.update(x=t["x"], ids=t["ids"], tw=t["tw"])
    elif kind == "moe_train":
        s.update(x=t["x"].requires_grad_(True), ids=t["ids"], tw=t["tw"].requires_grad_(True),
                 w_gu=moe.stack_gate_up(t["gate"], t["up"]).requires_grad_(True),
                 w_down=t["down"].requires_grad_(True), dy=t["dy"])
    elif kind == "refresh":
        s["w"] = t["w"]
    else:
        s["x"] = t["x"]
    return s


def run(s):
    from lowbit import moe
    from lowbit import persistent as P

    kind, c = s["kind"], s["case"]
    if kind == "linear_fwd":
        with torch.no_grad():
            return s["backend"].linear(s["x"], s["w"], s["b"])
    if kind in ("linear_train", "recipe_train"):
        y = s["backend"].linear(s["x"], s["w"], s["b"])
        leaves = [v for v in (s["x"], s["w"], s["b"]) if v is not None]
        return [y.detach(), *torch.autograd.grad(y, leaves, s["dy"])]
    if kind == "stored_linear":
        if c["fmt"] == "nf4":
            return P.linear_nf4(s["x"], s["codes"], s["scales"], out_features=c["N"], block=64)
        if c["fmt"] == "mxfp4":
            return P.linear_mxfp4(s["x"], s["codes"], s["scales"], out_features=c["N"])
        return P.linear_fp8p(s["x"], s["codes"], s["scales"])
    if kind == "stored_train":
        layer = s["layer"]
        y = layer(s["x"])
        leaves = [v for v in (s["x"], layer.weight, layer.bias) if v is not None]
        return [y.detach(), *torch.autograd.grad(y, leaves, s["dy"])]
    if kind == "moe_fwd":
        return moe.local_moe_forward(s["x"], s["ids"], s["tw"], s["gate_up"], s["down"], n_experts=c["E"],
                                     fmt=c["fmt"])
    if kind == "moe_train":
        y = moe.local_moe(s["x"], s["ids"], s["tw"], s["w_gu"], s["w_down"], fmt=c["fmt"])
        return [y.detach(), *torch.autograd.grad(y, (s["x"], s["tw"], s["w_gu"], s["w_down"]), s["dy"])]
    if kind == "refresh":
        if c["fmt"] == "nf4":
            return list(P.quantize_nf4_persistent(s["w"], granularity="per_channel"))
        codes, scale = P.quantize_fp8_persistent(s["w"], granularity="per_channel")
        return [codes.view(torch.uint8), scale]
    return moe.comm_quant_dequant(s["x"], granularity="tile_1x128", rounding_mode=c["rounding"], seed=11, offset=3)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(c):
    kind = c["kind"]
    if kind in ("linear_fwd", "linear_train", "recipe_train", "stored_train", "stored_linear"):
        M, N, K = c["M"], c["N"], c["K"]
        wbytes = 2 * N * K
        if kind in ("stored_linear", "stored_train"):
            wbytes = {"nf4": N * K // 2, "mxfp4": N * K // 2, "fp8": N * K}[c["fmt"]]
        if kind in ("linear_fwd", "stored_linear"):
            return {"bytes": 2 * M * K + wbytes + 2 * M * N, "flops": 2 * M * N * K}
        # X, W, dY in; Y, dX, dW out
        return {"bytes": 2 * (2 * M * K + 2 * M * N + N * K) + wbytes, "flops": 6 * M * N * K}
    if kind in ("moe_fwd", "moe_train"):
        T, H, I, E, k = c["T"], c["H"], c["I"], c["E"], c["k"]
        live = min(E, T * k)
        if kind == "moe_fwd":
            return {"bytes": 4 * T * H + 3 * live * H * I, "flops": 6 * T * k * H * I}
        return {"bytes": 8 * T * H + 12 * live * H * I, "flops": 18 * T * k * H * I}
    if kind == "refresh":
        n = c["N"] * c["K"]
        return {"bytes": 2 * n + (n // 2 if c["fmt"] == "nf4" else n), "flops": 2 * n}
    return {"bytes": 4 * c["M"] * c["K"], "flops": 4 * c["M"] * c["K"]}


def tolerance(c):
    kind = c["kind"]
    if kind in ("refresh", "comm"):
        return "exact"  # codes, scales and quantized values: no sums whose order is free
    if kind in ("moe_fwd", "moe_train"):
        # a last-bit change of a bf16 gate, up or h value can move an e4m3 code of h
        return {"rel": 1e-2, "max": 0.5}
    # one bf16 rounding of an fp32 sum: another order of the sum moves a value by one bf16 step
    return {"rel": 4e-3, "max": 0.05}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def _safe_scale(amax, qmax):
    s = amax / torch.full_like(amax, qmax)
    return torch.where(torch.isfinite(s) & (s > 0), s, torch.ones_like(s))


def _codes(x, gr, gc, fmt, rand=None, before=False):
    """Code values q (fp32) and scales per element of x [R, K], one scale per (gr x gc) group"""
    R, K = x.shape
    gr, gc = min(gr, R), min(gc, K)
    Rp, Kp = -(-R // gr) * gr, -(-K // gc) * gc
    xp = torch.zeros(Rp, Kp, device=DEV)
    xp[:R, :K] = x.float()
    v = xp.reshape(Rp // gr, gr, Kp // gc, gc)
    amax = v.abs().amax(dim=(1, 3), keepdim=True)
    qmax = 448.0 if fmt == "e4m3" else 127.0
    s = _safe_scale(amax, qmax)
    q = (v / s).reshape(Rp, Kp)[:R, :K]
    s = s.expand(Rp // gr, gr, Kp // gc, gc).reshape(Rp, Kp)[:R, :K]
    if fmt == "e4m3":
        q = q.clamp(-448, 448).to(torch.float8_e4m3fn).float()
    elif rand is not None:
        q = torch.where(q >= 0, torch.floor(q + rand), torch.ceil(q - rand)).clamp(-127, 127)
    else:
        q = torch.round(q).clamp(-127, 127)
    return q, s


def _dq64(x, gr, gc, fmt):
    q, s = _codes(x, gr, gc, fmt)
    return q.double() * s.double()


def _dqbf(x, gr, gc, fmt):
    """bf16(q * s): the operand of the straight-through gradients"""
    q, s = _codes(x, gr, gc, fmt)
    return (q * s).to(BF16).double()


def _philox_words(n, seed, offset):
    """One uint32 word per element: Philox4x32-10, counter (element / 4, offset), key seed, word element % 4"""
    mask = 0xFFFFFFFF
    e = torch.arange((n + 3) // 4, device=DEV, dtype=torch.int64)
    c = [e & mask, e >> 32, torch.full_like(e, offset & mask), torch.full_like(e, offset >> 32)]
    k0, k1 = seed & mask, seed >> 32

    def mul(a, m):
        p = a * m  # modulo 2^64: both halves are exact bits of the product
        return (p >> 32) & mask, p & mask

    for _ in range(10):
        hi0, lo0 = mul(c[0], 0xD2511F53)
        hi1, lo1 = mul(c[2], 0xCD9E8D57)
        c = [hi1 ^ c[1] ^ k0, lo1, hi0 ^ c[3] ^ k1, lo0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return torch.stack(c, dim=1).reshape(-1)[:n]


NF4 = (-1.0, -0.6961928, -0.52507305, -0.3949175, -0.28444138, -0.18477343, -0.09105004, 0.0, 0.0795803, 0.1609302,
       0.2461123, 0.33791524, 0.44070983, 0.562617, 0.72295684, 1.0)


def _stored_bf16(w, fmt, block):
    """The bf16 values a stored weight w [N, K] stands for"""
    N, K = w.shape
    v = w.float().reshape(-1, block)
    amax = v.abs().amax(dim=1, keepdim=True)
    if fmt == "mxfp4":
        grid = torch.tensor((0, 0.5, 1, 1.5, 2, 3, 4, 6), device=DEV)
        e = torch.floor(torch.log2(amax.double())) - 2
        scale = torch.exp2(e.clamp(-127, 127)).float()
        a = (v / scale).abs().clamp(max=6.0)
        # nearest, ties to the even code
        i = torch.bucketize(a, (grid[1:] + grid[:-1]) / 2)
        mid = (grid[1:] + grid[:-1]) / 2
        tie = (i < 7) & (a == mid[i.clamp(max=6)])
        i = torch.where(tie & (i % 2 == 1), i + 1, i)
        return (torch.sign(v) * grid[i] * scale).reshape(N, K).to(BF16)
    scale = torch.where(torch.isfinite(amax) & (amax > 0), amax, torch.ones_like(amax))
    if fmt == "nf4":
        book = torch.tensor(NF4, device=DEV)
        n = v / scale
        q = torch.empty_like(n)
        for r in range(0, n.shape[0], 8192 if block > 64 else 1 << 20):
            part = n[r:r + (8192 if block > 64 else 1 << 20)]
            best, at = torch.full_like(part, math.inf), torch.zeros_like(part)
            for level in book:
                d = (part - level).abs()
                closer = d < best
                best, at = torch.where(closer, d, best), torch.where(closer, level, at)
            q[r:r + part.shape[0]] = at
        return (q * scale).reshape(N, K).to(BF16)
    q = (v / scale).clamp(-448, 448).to(torch.float8_e4m3fn).float()
    return (q * scale).reshape(N, K).to(BF16)


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind in ("linear_fwd", "linear_train", "recipe_train"):
        fmt = case["fmt"]
        x, w, b = t["x"], t["w"], t["b"]
        y = _dq64(x, 1, 128, fmt) @ _dq64(w, 128, 128, fmt).T
        if b is not None:
            y += b.double()
        if kind == "linear_fwd":
            return y
        dy = t["dy"]
        if kind == "linear_train":
            out = [y, dy.double() @ _dqbf(w, 128, 128, fmt), dy.double().T @ _dqbf(x, 1, 128, fmt)]
        else:
            out = [y, _dq64(dy, 1, 128, fmt) @ _dq64(w, 128, 128, fmt),
                   _dq64(dy, 128, 1, fmt).T @ _dq64(x, 128, 1, fmt)]
        return out if b is None else out + [dy.double().sum(0)]
    if kind == "stored_linear":
        block = {"nf4": 64, "mxfp4": 32, "fp8": case["K"]}[case["fmt"]]
        return t["x"].double() @ _stored_bf16(t["w"], case["fmt"], block).double().T
    if kind == "stored_train":
        wq = _stored_bf16(t["w"], case["fmt"], case["K"]).double()
        x, dy = t["x"].double(), t["dy"].double()
        y = x @ wq.T
        if t["b"] is not None:
            y += t["b"].double()
        out = [y, dy @ wq, dy.T @ x]
        return out if t["b"] is None else out + [dy.sum(0)]
    if kind == "refresh":
        amax = t["w"].double().abs().amax(dim=1, keepdim=True)
        return [None, torch.where(amax > 0, amax, torch.ones_like(amax))]
    if kind == "comm":
        x = t["x"]
        rand = None
        if case["rounding"] == "stochastic":
            rand = (_philox_words(x.numel(), 11, 3) >> 8).float().reshape(x.shape) * 2.0 ** -24
        q, s = _codes(x, x.shape[0], 128, "int_grid", rand)
        return q.double() * s.double()
    return _exact_moe(case, t)


def _exact_moe(case, t):
    """The expert loop with its bf16 projections, activations and codes, sums and gradients in 64 bits"""
    fmt, T, H, I, E, k = case["fmt"], case["T"], case["H"], case["I"], case["E"], case["k"]
    train = case["kind"] == "moe_train"
    ids, tw = t["ids"], t["tw"].double()
    xq, xb = _dq64(t["x"], 1, 128, fmt), _dqbf(t["x"], 1, 128, fmt)
    out = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    if train:
        dy = t["dy"].double()
        dx, dtw = torch.zeros_like(out), torch.zeros_like(tw)
        dgu = torch.zeros(E, I // 128, 2, 128, H, device=DEV)
        ddown = torch.zeros(E, H, I, device=DEV)
    for e in range(E):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if not len(tok):
            continue
        x = xq[tok]
        g = (x @ _dq64(t["gate"][e], 128, 128, fmt).T).to(BF16)
        u = (x @ _dq64(t["up"][e], 128, 128, fmt).T).to(BF16)
        sg = (g.double() * torch.sigmoid(g.double())).to(BF16)
        h = (sg.double() * u.double()).to(BF16)
        y = _dq64(h, 1, 128, fmt) @ _dq64(t["down"][e], 128, 128, fmt).T
        w = tw[tok, slot][:, None]
        out.index_add_(0, tok, y * w)
        if not train:
            continue
        d = dy[tok]
        dtw[tok, slot] = (d * y).sum(1)
        dyr = d * w
        dh = dyr @ _dqbf(t["down"][e], 128, 128, fmt)
        ddown[e] = dyr.T @ _dqbf(h, 1, 128, fmt)
        g64, u64 = g.double(), u.double()
        sig = torch.sigmoid(g64)
        du = dh * sg.double()
        dg = dh * u64 * sig * (1 + g64 * (1 - sig))
        dx.index_add_(0, tok, dg @ _dqbf(t["gate"][e], 128, 128, fmt) + du @ _dqbf(t["up"][e], 128, 128, fmt))
        dgu[e, :, 0] = (dg.T @ xb[tok]).reshape(I // 128, 128, H)
        dgu[e, :, 1] = (du.T @ xb[tok]).reshape(I // 128, 128, H)
    if not train:
        return out
    return [out, dx, dtw, dgu.reshape(E, 2 * I, H), ddown]
