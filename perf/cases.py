"""The work that is timed: one LoRA training step, load or call of every public entry point of
r9700training_amd, from a single token to the largest benchmark workload.

    listed()            the cases that stand for the ranges
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call (weights, inputs, workspaces), on the card
    run(state)          one pass through the public entry points
    work(case)          the bytes and operations the pass cannot do without
    tolerance(case)     how far another correct implementation's outputs may lie
    exact(case, seed)   the same outputs in float64 from plain torch

Sizes are those of the benchmark workloads and the tests (one 1024 x 1024 layer of 128 tokens, the
square 4096 layer, the rank-64 attention projections, the published real-model widths 5120 / 6144 /
12288 / 17408, the 24-layer adapter stack, the 248320-row vocabulary head) and the odd token
counts between them.
"""
from __future__ import annotations

import math

import torch

from r9700training_amd.optim import DeviceAdamW, config
from r9700training_amd.qlinear import (QWeight, bwd_workspace, device_desc, fwd_workspace, gemm_nt_q_dx,
                                       gemm_nt_q_fwd, iqr_decode, lora_expand_bwd, lora_shrink_bwd,
                                       lora_shrink_q_bwd, qlinear_lora_bwd, qlinear_lora_fwd)
from r9700training_amd.quant import (fused_had_quant_i8g, fused_had_quant_i8g_bwd, quant_act_i8g,
                                     quant_act_i8g_bwd)
from r9700training_amd.vocab_head import VocabHead

DEV = "cuda"
MAD_A, MAD_B = 0x2F1E3D, 0x9E3779B9  # a codebook hash (any odd A, any B)
SCALE = 2.0                          # alpha / r of every benchmark workload
# the 24-layer stack's projections (N, K) and the vocabulary head's classes, as the benchmark has them
STACK_PROJ = [(8192, 2048), (2048, 4096), (6144, 2048), (2048, 6144)]
VOCAB_CLASSES = [32768, 65536, 98304, 51712]


def listed():
    return [
        # a serving loop's decode call: one token through one layer, bf16 out
        dict(name="token_fwd", kind="linear", op="fwd", T=1, N=4096, K=4096, r=16, bits=5, form="trellis", out="bf16",
             accumulate=False),
        # the smallest training step: a 1024 x 1024 layer, 128 tokens, rank 8
        dict(name="small_step", kind="linear", op="step", T=128, N=1024, K=1024, r=8, bits=5, form="trellis",
             out="f32", accumulate=False),
        # a ragged batch through a layer with odd widths (a short last trellis run) held as int8
        # codes, bf16 activations, dX added into the residual's gradient
        dict(name="ragged_step", kind="linear", op="step", T=777, N=1408, K=2560, r=32, bits=4, form="codes8",
             out="bf16", accumulate=True),
        # the flagship: the square layer's forward and backward
        dict(name="square_step", kind="linear", op="step", T=4096, N=4096, K=4096, r=16, bits=5, form="trellis",
             out="f32", accumulate=False),
        # a long batch through the attention projection at the largest rank
        dict(name="attn_step", kind="linear", op="step", T=16384, N=8192, K=2048, r=64, bits=5, form="trellis",
             out="f32", accumulate=False),
        # a layer of a checkpoint on its way in: the kernels' form prepared, the decoded grids for
        # the coded trunk
        dict(name="weight_load", kind="load", N=12288, K=5120, bits=5, book="mad", form="trellis"),
        # one layer of the coded (int8) trunk: quantise, product, its adjoint, the shrink's adjoint,
        # the quantiser's adjoint
        dict(name="coded_layer", kind="coded", T=2048, N=4096, K=4096, r=16, x="bf16"),
        # the adapter's two adjoints on their own, as a walk over separate rows calls them
        dict(name="adapter_rows", kind="adapter", T=4096, N=12288, K=5120, r=16),
        # the norm before a coded layer for a short batch
        dict(name="norm_quant", kind="quant", part="rmsnorm", rows=64, n=5120, group=128, x="f32", out=False),
        # the gated MLP activation of a full batch at the real model's width
        dict(name="gated_quant", kind="quant", part="silu_mul", rows=4096, n=17408, group=128, x="bf16", out=True),
        # the head's backward at its full size
        dict(name="vocab_head", kind="vocab", rows=4096, n_embd=2048, classes=4, vocab=sum(VOCAB_CLASSES),
             transform=128),
        # the optimiser's step over every factor of the 24-layer stack, clipped
        dict(name="lora_optimizer", kind="adamw", layers=24, r=16, clip=1.0, decay=0.01),
    ]


def _log(rng, lo, hi):
    return lo * math.exp(rng.random() * math.log(hi / lo))


def _int(rng, lo, hi):
    return max(lo, min(hi, round(_log(rng, lo, hi))))


def _dim(rng, lo=512, hi=17408):
    return 128 * max(lo // 128, min(hi // 128, round(_log(rng, lo, hi) / 128)))


def draw(rng):
    kind = rng.choice(["token", "step", "step", "step", "load", "coded", "adapter", "quant", "quant", "vocab", "adamw"])
    if kind in ("token", "step"):
        T = _int(rng, 1, 256) if kind == "token" else _int(rng, 16, 16384)
        N, K = _dim(rng), _dim(rng)
        while T * N * K > 8e11:
            N, K = _dim(rng), _dim(rng)
        return dict(kind="linear", op="fwd" if kind == "token" else "step", T=T, N=N, K=K,
                    r=rng.choice([0, 8, 16, 16, 32, 64]), bits=rng.choice([3, 4, 5, 5, 6]),
                    form=rng.choice(["trellis", "trellis", "codes8"]), out=rng.choice(["f32", "bf16"]),
                    accumulate=rng.random() < 0.3)
    if kind == "load":
        book = rng.choice(["mad", "mad", "lut"])
        return dict(kind="load", N=_dim(rng, 512, 12288), K=_dim(rng, 512, 12288), bits=rng.choice([3, 4, 5, 6]),
                    book=book, form="codes8" if book == "lut" else rng.choice(["trellis", "codes8"]))
    if kind == "coded":
        return dict(kind="coded", T=_int(rng, 1, 4096), N=_dim(rng, 512, 12288), K=_dim(rng, 512, 6144),
                    r=rng.choice([8, 16, 32, 64]), x=rng.choice(["bf16", "f32"]))
    if kind == "adapter":
        return dict(kind="adapter", T=_int(rng, 16, 8192), N=_dim(rng, 512, 17408), K=_dim(rng, 512, 8192),
                    r=rng.choice([8, 16, 32, 64]))
    if kind == "quant":
        part = rng.choice(["rmsnorm", "silu_mul", "sigmoid_mul"])
        return dict(kind="quant", part=part, rows=_int(rng, 1, 4096), n=_dim(rng, 512, 17408),
                    group=rng.choice([32, 64, 128, 128, 128]), x=rng.choice(["bf16", "bf16", "f32"]),
                    out=rng.random() < 0.5)
    if kind == "vocab":
        classes = rng.randint(1, 4)
        return dict(kind="vocab", rows=_int(rng, 1, 4096), n_embd=_dim(rng, 512, 2560), classes=classes,
                    vocab=classes * 256 * _int(rng, 4, 180), transform=rng.choice([0, 128]))
    return dict(kind="adamw", layers=_int(rng, 1, 24), r=rng.choice([8, 16, 32, 64]), clip=rng.choice([0.0, 1.0]),
                decay=rng.choice([0.0, 0.01]))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, shape, dtype=torch.float32, std=1.0):
    return (std * torch.randn(shape, generator=g, device=DEV)).to(dtype)


def _dtype(name):
    return {"f32": torch.float32, "bf16": torch.bfloat16}[name]


def _planes(g, N, K, bits, book="mad", run_rows=256):
    """One stored weight's planes on the card (random packed codes: every bit pattern is a valid
    code; an f32 scale a row and a factor a 128-column block) and its description."""
    nb = K * bits // 8
    p = dict(codes=torch.randint(0, 256, (N, nb), dtype=torch.uint8, device=DEV, generator=g),
             row=0.0002 + 0.0006 * torch.rand(N, device=DEV, generator=g),
             col=0.75 + 0.5 * torch.rand(K // 128, device=DEV, generator=g), bits=bits, run_rows=run_rows, N=N, K=K)
    planes = dict(codes=p["codes"], scale=p["row"].view(torch.uint8))
    if book == "lut":
        p["lut"] = torch.randint(-126, 127, (1 << 16,), dtype=torch.int8, device=DEV, generator=g)
        planes["lut"] = p["lut"]
    p["desc"] = device_desc(planes, N, K, dict(
        bits=bits, state_bits=16, run_rows=run_rows, rb=1, mad=int(book == "mad"), round_mad=1, mad_a=MAD_A,
        mad_b=MAD_B, codes_row_bytes=nb, scale_dtype=0, scale_block_cols=0, scale_row_bytes=4))
    return p


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _gen(seed))


def run(state):
    return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    return _TOL[case["kind"]](case)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, prepare(case, seed)) if f else None


# ------------------------------------------------------------------ the linear + LoRA layer
def _linear_prepare(c, g):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    p = _planes(g, N, K, c["bits"])
    s = dict(kind="linear", c=c, planes=p, w=QWeight(p["desc"], scale_col=p["col"], codes8=c["form"] == "codes8"))
    bf = torch.bfloat16
    s["X"] = _randn(g, (T, K), bf)
    s["A"] = _randn(g, (r, K), bf, 0.01) if r else None
    s["B"] = _randn(g, (N, r), bf, 0.01) if r else None
    s["Y"] = torch.empty((T, N), dtype=_dtype(c["out"]), device=DEV)
    s["t"] = torch.empty((T, r), device=DEV) if r else None
    s["wsf"] = fwd_workspace(T, N, K, r, DEV)
    if c["op"] == "step":
        s["dY"] = _randn(g, (T, N), bf)
        s["dX"] = _randn(g, (T, K), _dtype(c["out"])) if c["accumulate"] else torch.empty(
            (T, K), dtype=_dtype(c["out"]), device=DEV)
        # the factors' gradients add up over the micro-batches of a step
        s["dA"] = torch.zeros((r, K), device=DEV) if r else None
        s["dB"] = torch.zeros((N, r), device=DEV) if r else None
        s["wsb"] = bwd_workspace(T, N, K, r, DEV)
    return s


def _linear_run(s):
    c = s["c"]
    Y, t = qlinear_lora_fwd(s["w"], s["X"], s["A"], s["B"], SCALE, workspace=s["wsf"], out=s["Y"], t_out=s["t"])
    if c["op"] == "fwd":
        return {"Y": Y, "t": t}
    dX, dA, dB = qlinear_lora_bwd(s["w"], s["X"], s["dY"], s["A"], s["B"], t, SCALE, dX=s["dX"],
                                  accumulate=c["accumulate"], dA=s["dA"], dB=s["dB"], workspace=s["wsb"])
    return {"Y": Y, "t": t, "dX": dX, "dA": dA, "dB": dB}


def _linear_work(c):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    o = 4 if c["out"] == "f32" else 2
    w = N * K * (1.0 if c["form"] == "codes8" else c["bits"] / 8) + 2 * N * K / 128
    f = 2 * T * (K + N) * r
    by, fl = w + 2 * T * K + T * N * o + 2 * r * (N + K) + 4 * T * r, 2 * T * N * K + f
    if c["op"] == "step":
        by += w + 2 * T * (N + K) + T * K * o * (2 if c["accumulate"] else 1) + (2 + 8) * r * (N + K) + 4 * T * r
        fl += 2 * T * N * K + 2 * f
    return {"bytes": by, "flops": fl}


def _linear_tol(c):
    # one bf16 rounding of each weight (1.65e-3 against float64, so 2.3e-3 between two roundings);
    # a bf16 output adds its own
    return {"rel": 5e-3, "max": 0.05} if c["out"] == "f32" else {"rel": 8e-3, "max": 0.08}


def _linear_exact(c, s):
    W = _weight(s["planes"])
    X, r = s["X"].double(), c["r"]
    Y, t = X @ W.T, None
    if r:
        A, B = s["A"].double(), s["B"].double()
        t = X @ A.T
        Y = Y + SCALE * (t @ B.T)
    if c["op"] == "fwd":
        return {"Y": Y, "t": t}
    dY = s["dY"].double()
    dX, dA, dB = dY @ W, None, None
    if r:
        dt = SCALE * (dY @ B)
        dX = dX + dt @ A
        dA, dB = dt.T @ X, SCALE * (dY.T @ t)
    if c["accumulate"]:
        dX = dX + s["dX"].double()
    return {"Y": Y, "t": t, "dX": dX, "dA": dA, "dB": dB}


def _codes(p, r0=0, r1=None):
    """The stored codes of rows r0..r1 (whole trellis runs) decoded in plain torch: a column's 16-bit
    state is its last codes down the rows, wrapping within the run; the value is the byte sum of
    the masked hash of the state, less 126."""
    r1 = p["N"] if r1 is None else r1
    bits, K = p["bits"], p["K"]
    packed = p["codes"][r0:r1].to(torch.int32)
    packed = torch.cat([packed, torch.zeros_like(packed[:, :1])], 1)
    o = torch.arange(K, device=DEV) * bits
    raw = ((packed[:, o >> 3] | (packed[:, (o >> 3) + 1] << 8)) >> (o & 7).to(torch.int32)) & ((1 << bits) - 1)
    out = torch.empty((r1 - r0, K), dtype=torch.float64, device=DEV)
    for a in range(0, r1 - r0, p["run_rows"]):
        run_ = raw[a:a + p["run_rows"]]
        st = torch.zeros_like(run_)
        for j in range((16 + bits - 1) // bits):
            st |= torch.roll(run_, j, 0) << (j * bits)
        st = (st & 0xFFFF).to(torch.int64)
        h = (st * (MAD_A & 0xFFFFFF) + MAD_B) & 0x3F3F3F3F
        out[a:a + p["run_rows"]] = ((h & 0xFF) + ((h >> 8) & 0xFF) + ((h >> 16) & 0xFF) + (h >> 24) - 126).double()
    return out


def _weight(p):
    scale = (p["row"][:, None] * p["col"][None, :]).to(torch.bfloat16).double()
    return _codes(p) * scale.repeat_interleave(128, 1)


# ------------------------------------------------------------------ a stored weight on its way in
def _load_prepare(c, g):
    p = _planes(g, c["N"], c["K"], c["bits"], c["book"])
    return dict(kind="load", c=c, planes=p,
                codes=torch.empty((c["N"], c["K"]), dtype=torch.int8, device=DEV),
                scale=torch.empty((c["N"], c["K"] // 128), dtype=torch.int16, device=DEV))


def _load_run(s):
    p = s["planes"]
    w = QWeight(p["desc"], scale_col=p["col"], codes8=s["c"]["form"] == "codes8")
    iqr_decode(p["desc"], s["codes"], s["scale"])
    return {"stream": w.stream_plane, "scale_t": w.scale_t, "codes": s["codes"], "scale": s["scale"]}


def _load_work(c):
    n = c["N"] * c["K"]
    packed = n * c["bits"] / 8
    return {"bytes": 2 * packed + n + (packed if c["form"] == "trellis" else n) + 4 * n / 128, "flops": 0}


# ------------------------------------------------------------------ a layer of the coded trunk
def _coded_prepare(c, g):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    codes = torch.randint(-126, 127, (N, K), dtype=torch.int8, device=DEV, generator=g)
    scale = (0.0002 + 0.0004 * torch.rand((N, K // 128), device=DEV, generator=g)).to(torch.bfloat16)
    return dict(kind="coded", c=c, codes=codes, scale=scale,
                w=QWeight.from_decoded(codes, scale.view(torch.int16)),
                x=_randn(g, (T, K), _dtype(c["x"])), dY=_randn(g, (T, N), torch.bfloat16),
                A=_randn(g, (r, K), torch.bfloat16, 0.01), t_cot=_randn(g, (T, r)),
                Y=torch.empty((T, N), device=DEV), da=torch.empty((T, K), device=DEV))


def _coded_run(s):
    a, a_scale = quant_act_i8g(s["x"], 128, rotated=True)
    Y = gemm_nt_q_fwd(s["codes"], s["scale"], a, a_scale, Y=s["Y"])
    da = gemm_nt_q_dx(s["w"], s["dY"], a_scale, dA=s["da"])
    da, ds, dA = lora_shrink_q_bwd(a, a_scale, s["A"], s["t_cot"], da=da)
    dx = quant_act_i8g_bwd(s["x"], a_scale, da, 128, rotated=True)
    return {"a": a, "a_scale": a_scale, "Y": Y, "da": da, "ds": ds, "dA": dA, "dx": dx}


def _coded_work(c):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    x = 2 if c["x"] == "bf16" else 4
    # quantise; the product; its adjoint; the shrink's adjoint (da read and written, a, t_cot); the
    # quantiser's adjoint
    by = T * K * (x + 1) + (T * K + N * K + 4 * T * N) + (N * K + 2 * T * N + 4 * T * K) + (8 * T * K + T * K) + \
        T * K * (x + 4 + 4) + 5 * 4 * T * K / 128 + 4 * N * K / 128 + 6 * r * K + 4 * T * r
    return {"bytes": by, "flops": 4 * T * N * K + 4 * T * r * K}


def _hadamard(n):
    H = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while H.shape[0] < n:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    return H


def _rotate(v, group):
    return (v.reshape(-1, group) @ _hadamard(group)).reshape(v.shape)


def _quantise(v, group):
    """Codes and scales (f32, as the codes' readers take them) of rotated values, in float64."""
    q = v.reshape(v.shape[0], -1, group)
    s = q.abs().amax(2) * (1.0 / 127.0)
    s = torch.where(s > 0, s, torch.ones_like(s))
    codes = torch.clamp(torch.round(q * (1.0 / s)[..., None]), -127, 127).reshape(v.shape)
    return codes, s


def _straight_through(v, s32, gc, group):
    """The rotated quantiser's adjoint of the codes' cotangent gc at the written scales."""
    s = s32.double().repeat_interleave(group, 1)
    return _rotate(torch.where((v * (1.0 / s)).abs() > 127.0, torch.zeros_like(gc), gc / s), group)


def _coded_exact(c, s):
    K = c["K"]
    v = _rotate(s["x"].double(), 128)
    a, sc = _quantise(v, 128)
    s32 = sc.float()
    wide = s32.double().repeat_interleave(128, 1)
    W = s["codes"].double() * s["scale"].double().repeat_interleave(128, 1)
    A, t_cot = s["A"].double(), s["t_cot"].double()
    gx = t_cot @ A
    da = wide * (s["dY"].double() @ W) + gx * wide
    return {"a": None, "a_scale": sc, "Y": (a * wide) @ W.T, "da": da,
            "ds": (gx * a).reshape(c["T"], K // 128, 128).sum(2), "dA": t_cot.T @ (a * wide),
            "dx": _straight_through(v, s32, da, 128)}


# ------------------------------------------------------------------ the adapter's adjoints
def _adapter_prepare(c, g):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    bf = torch.bfloat16
    return dict(kind="adapter", c=c, X=_randn(g, (T, K), bf), dY=_randn(g, (T, N), bf), A=_randn(g, (r, K), bf, 0.01),
                B=_randn(g, (N, r), bf, 0.01), t=_randn(g, (T, r)), dX=torch.empty((T, K), device=DEV),
                dA=torch.zeros((r, K), device=DEV), dB=torch.zeros((N, r), device=DEV))


def _adapter_run(s):
    t_cot, dB = lora_expand_bwd(s["dY"], s["B"], SCALE, t=s["t"], dB=s["dB"])
    dX, dA = lora_shrink_bwd(s["X"], s["A"], t_cot, dX=s["dX"], dA=s["dA"])
    return {"t_cot": t_cot, "dX": dX, "dA": dA, "dB": dB}


def _adapter_work(c):
    T, N, K, r = c["T"], c["N"], c["K"], c["r"]
    return {"bytes": 2 * T * (N + K) + 4 * T * K + (2 + 8) * r * (N + K) + 12 * T * r, "flops": 4 * T * r * (N + K)}


def _adapter_exact(c, s):
    X, dY, A, B, t = (s[k].double() for k in ("X", "dY", "A", "B", "t"))
    t_cot = SCALE * (dY @ B)
    return {"t_cot": t_cot, "dX": t_cot @ A, "dA": t_cot.T @ X, "dB": SCALE * (dY.T @ t)}


# ------------------------------------------------------------------ the fused quantiser producers
def _quant_prepare(c, g):
    rows, n, dt = c["rows"], c["n"], _dtype(c["x"])
    part = c["part"]
    s = dict(kind="quant", c=c, x0=_randn(g, (rows, 2 * n if part == "silu_mul" else n), dt), x1=None,
             gc=_randn(g, (rows, n)), gout=_randn(g, (rows, n)) if c["out"] else None)
    if part == "rmsnorm":
        s["x1"] = (1.0 + _randn(g, (n,), std=0.1)).to(dt)
    elif part == "sigmoid_mul":
        s["x1"] = _randn(g, (rows, n), dt)
    # the gradients of the producer's inputs add up over their readers
    s["dx0"] = _randn(g, tuple(s["x0"].shape))
    s["dx1"] = _randn(g, (rows, n)) if part == "sigmoid_mul" else None
    return s


def _quant_run(s):
    c = s["c"]
    codes, scale, y = fused_had_quant_i8g(c["part"], s["x0"], s["x1"], c["group"], want_y=c["out"])
    dx0, dx1 = fused_had_quant_i8g_bwd(c["part"], s["x0"], s["x1"], c["group"], scale, s["gc"], g_out=s["gout"],
                                       dx0=s["dx0"], dx1=s["dx1"])
    return {"codes": codes, "scale": scale, "y": y, "dx0": dx0, "dx1": dx1}


def _quant_work(c):
    rows, n = c["rows"], c["n"]
    x = 2 if c["x"] == "bf16" else 4
    ins = 1 if c["part"] == "rmsnorm" else 2  # values an output is made of
    by = 2 * ins * x + 1 + 4 + 8 * ins + (2 + 4 if c["out"] else 0) + 8.0 / c["group"]
    return {"bytes": rows * n * by, "flops": 0}


def _quant_exact(c, s):
    n, group, part = c["n"], c["group"], c["part"]
    x0 = s["x0"].double()
    x1 = s["x1"].double() if s["x1"] is not None else None
    if part == "rmsnorm":
        rs = 1.0 / torch.sqrt((x0 * x0).sum(1, keepdim=True) / n + 1e-6)
        y = x0 * rs * x1
    elif part == "silu_mul":
        gate, up = x0[:, :n], x0[:, n:]
        sg = 1.0 / (1.0 + torch.exp(-gate))
        y = gate * sg * up
    else:
        sg = 1.0 / (1.0 + torch.exp(-x0))
        y = sg * x1
    v = _rotate(y, group)
    _, sc = _quantise(v, group)
    d = _straight_through(v, sc.float(), s["gc"].double(), group)
    if s["gout"] is not None:
        d = d + s["gout"].double()
    dx1 = None
    if part == "rmsnorm":
        t = (d * x0 * x1).sum(1, keepdim=True)
        dx0 = s["dx0"].double() + rs * x1 * d - rs ** 3 * x0 * t / n
    elif part == "silu_mul":
        dx0 = s["dx0"].double() + torch.cat([d * up * (sg * (1.0 + gate * (1.0 - sg))), d * gate * sg], 1)
    else:
        dx0 = s["dx0"].double() + d * sg * (1.0 - sg) * x1
        dx1 = s["dx1"].double() + d * sg
    return {"codes": None, "scale": sc, "y": y if c["out"] else None, "dx0": dx0, "dx1": dx1}


# ------------------------------------------------------------------ the vocabulary head's backward
def _vocab_rows(c):
    """Rows of each class: whole 256-row runs in the benchmark head's proportions."""
    n, vocab = c["classes"], c["vocab"]
    if n == 4 and vocab == sum(VOCAB_CLASSES):
        return list(VOCAB_CLASSES)
    runs, part = vocab // 256, [1, 2, 3, 2][:n]
    rows = [max(1, runs * k // sum(part)) for k in part]
    rows[-1] += runs - sum(rows)
    return [256 * k for k in rows]


def _vocab_prepare(c, g):
    K, vocab = c["n_embd"], c["vocab"]
    perm = torch.randperm(vocab, device=DEV, generator=g).to(torch.int32)
    classes, planes, at = [], [], 0
    for n in _vocab_rows(c):
        p = _planes(g, n, K, 5)
        p["ids"] = perm[at:at + n].sort().values.contiguous()
        at += n
        planes.append(p)
        classes.append((p["desc"], p["ids"], p["col"]))
    head = VocabHead(K, vocab, classes, transform=c["transform"])
    return dict(kind="vocab", c=c, planes=planes, head=head,
                dy=torch.randn((c["rows"], vocab), dtype=torch.bfloat16, device=DEV, generator=g),
                d_x=torch.zeros((c["rows"], K), device=DEV),
                ws=torch.empty(head.workspace_bytes(c["rows"]), dtype=torch.uint8, device=DEV))


def _vocab_run(s):
    # the head's input gradient starts from zero each step
    return s["head"].transpose(s["dy"], s["d_x"].zero_(), s["ws"])


def _vocab_work(c):
    rows, K, vocab = c["rows"], c["n_embd"], c["vocab"]
    return {"bytes": 2 * rows * vocab + vocab * K * 5 / 8 + 8 * vocab + 4 * rows * K, "flops": 2 * rows * vocab * K}


def _vocab_exact(c, s):
    out = torch.zeros((c["rows"], c["n_embd"]), dtype=torch.float64, device=DEV)
    for p in s["planes"]:
        for a in range(0, p["N"], 8192):
            b = min(a + 8192, p["N"])
            W = _codes(p, a, b) * p["row"][a:b, None].to(torch.bfloat16).double()
            out += s["dy"][:, p["ids"][a:b].long()].double() @ (W * p["col"].double().repeat_interleave(128)[None, :])
    return _rotate(out, 128) if c["transform"] else out


# ------------------------------------------------------------------ the adapters' optimiser
def _adamw_prepare(c, g):
    r = c["r"]
    shapes = [s for _ in range(c["layers"]) for N, K in STACK_PROJ for s in ((r, K), (N, r))]
    sizes = [a * b for a, b in shapes]

    def split(flat):
        return [x.view(s) for x, s in zip(flat.split(sizes), shapes)]

    w = _randn(g, (sum(sizes),), std=0.01)
    wb = torch.empty(sum(sizes), dtype=torch.bfloat16, device=DEV)
    grads = _randn(g, (sum(sizes),), std=0.001)
    opt = DeviceAdamW(split(w), config(lr=2e-4, clip_norm=c["clip"], weight_decay=c["decay"], warmup_steps=10,
                                       total_steps=1000), bf16_out=split(wb))
    return dict(kind="adamw", c=c, w=w, wb=wb, flat_grads=grads, grads=split(grads), opt=opt)


def _adamw_run(s):
    # the moments show in the weights of the passes after the first
    s["opt"].step(s["grads"])
    return {"w": s["w"], "w_bf16": s["wb"]}


def _adamw_work(c):
    n = c["layers"] * sum(c["r"] * (N + K) for N, K in STACK_PROJ)
    # the gradients (also for the norm), weights and both moments in; weights, moments, copies out
    return {"bytes": n * (4 + 12 + 12 + 2), "flops": 0}


def _adamw_exact(c, s):
    w, g = s["w"].double(), s["flat_grads"].double()
    if c["clip"] > 0:
        g = g * min(1.0, c["clip"] / float(g.norm()))
    b1, b2 = (float(torch.tensor(x, dtype=torch.float32)) for x in (0.9, 0.999))
    lr, eps, wd = (float(torch.tensor(x, dtype=torch.float32)) for x in (2e-4 / 10, 1e-8, c["decay"]))
    m, v = (1 - b1) * g, (1 - b2) * g * g
    w = w - lr * (m / (1 - b1) / (torch.sqrt(v / (1 - b2)) + eps) + wd * w)
    return {"w": w, "w_bf16": w}


_PREPARE = dict(linear=_linear_prepare, load=_load_prepare, coded=_coded_prepare, adapter=_adapter_prepare,
                quant=_quant_prepare, vocab=_vocab_prepare, adamw=_adamw_prepare)
_RUN = dict(linear=_linear_run, load=_load_run, coded=_coded_run, adapter=_adapter_run, quant=_quant_run,
            vocab=_vocab_run, adamw=_adamw_run)
_WORK = dict(linear=_linear_work, load=_load_work, coded=_coded_work, adapter=_adapter_work, quant=_quant_work,
             vocab=_vocab_work, adamw=_adamw_work)
_EXACT = dict(linear=_linear_exact, coded=_coded_exact, adapter=_adapter_exact, quant=_quant_exact,
              vocab=_vocab_exact, adamw=_adamw_exact)
_TOL = dict(
    linear=_linear_tol,
    load=lambda c: "exact",  # codes and scales are bytes
    coded=lambda c: {"rel": 5e-3, "max": 0.05},  # its adjoint's product rounds the weight once to bf16
    # the f32 adapter activations enter the products as two bf16 halves (16 significant bits)
    adapter=lambda c: {"rel": 2e-5, "max": 2e-4},
    # float64 arithmetic written as f32 (y as bf16); a tie's code may fall either way
    quant=lambda c: {"rel": 1e-6 if not c["out"] else 8e-3, "max": 0.02 if c["out"] else 1e-5, "differ": 1e-5},
    vocab=lambda c: {"rel": 2e-5, "max": 2e-4},  # 32-bit sums over the whole vocabulary
    adamw=lambda c: {"rel": 8e-3, "max": 0.02},  # the bf16 copies; the f32 weights are the reference's bits
)
