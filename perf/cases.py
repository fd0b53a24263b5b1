"""The work that programs have this framework do, as cases that can be timed and checked.

A case is one call of a public entry point at the sizes of the repository's own configurations
(`workloads.CONFIGS`: tiny, Wan-1.3B, Wan2.2-5B, FLUX-style, e4m3 base), its tests, or of a
piece of them: the DiT block linears q / k / v / o (hidden -> hidden), ffn.0 (hidden -> ffn)
and ffn.2 (ffn -> hidden), with rows of several roles or samples routed to their adapters, and
the modulated LayerNorm in front of them. A training pass returns the output and every
gradient.

Paths (`case["path"]`):
  linear   multi_lora_linear; dtype bf16 (bf16 activations and base) or f32 (all float32),
           masters: float32 adapters over the bf16 base
  gated    multi_lora_linear_gated, the float32 residual stream
  stacked  shared_input_multi_lora, q / k / v on one input
  fp8      multi_lora_linear_fp8, the frozen base in e4m3
  norm     modulated_layer_norm
Segments are `lengths` rows each, segment s with adapter `adapters[s]` (-1: base only).
"""
import math

import torch

from __graft_entry__ import load_package

mlora = load_package()
DEV = "cuda"


def _ints(text):
    return [int(v) for v in str(text).split(",")]


def _text(values):
    return ",".join(str(v) for v in values)


def _linear(name, path, K, N, ranks, lengths, adapters, **more):
    case = dict(name=name, path=path, K=K, N=N, ranks=_text(ranks), lengths=_text(lengths),
                adapters=_text(adapters), scale=1.0, dtype="bf16", masters=False, backward=True)
    case.update(more)
    return case


def listed():
    return [
        # the reference's CPU-runnable demo network: its smallest call, forward and backward in float32
        _linear("tiny_f32", "linear", 256, 256, (8, 8), (256, 256), (0, 1), dtype="f32"),
        # precision='fp32' training of one Wan-1.3B linear on a short clip (6 latent frames of 30 x 52
        # patches), generator and critic
        _linear("clip_q_f32", "linear", 1536, 1536, (64, 64), (4680, 4680), (0, 1), dtype="f32"),
        # cross-attention k / v on the 512 text tokens during sampling: no gradient, latency counts
        _linear("text_kv", "linear", 1536, 1536, (64,), (512,), (0,), backward=False),
        # one chunk of 3 latent frames (1560 tokens each): 2 frames of the generator, 1 of the critic
        _linear("chunk_q", "linear", 1536, 1536, (64, 64), (3120, 1560), (0, 1)),
        # native models: float32 adapter masters of rank 128 over the bf16 base, one role's full clip
        _linear("masters_q", "linear", 1536, 1536, (128,), (32760,), (0,), masters=True),
        # the Wan-1.3B block at both roles' full clips: q / k / v in one call
        _linear("wan_qkv", "stacked", 1536, 1536, (64, 64), (32760, 32760), (0, 1)),
        # ... the o projection that closes the attention branch into the float32 residual stream
        _linear("wan_o_gated", "gated", 1536, 1536, (64, 64), (32760, 32760), (0, 1)),
        # ... and ffn.2, the longest contraction
        _linear("wan_ffn2", "linear", 8960, 1536, (64, 64), (32760, 32760), (0, 1)),
        # ffn.0 over the e4m3 base with four adapters on uneven segments
        _linear("wan_ffn0_fp8", "fp8", 1536, 8960, (64, 64, 64, 64), (10471, 27603, 8013, 19433), (0, 1, 2, 3)),
        # Wan2.2-5B: three adapters of rank 128 on uneven segments
        _linear("wan22_ffn0", "linear", 3072, 14336, (128, 128, 128), (6511, 15360, 5409), (0, 1, 2), scale=2.0),
        # FLUX-style sampling: 16 samples with an adapter each, of ranks 16 to 128, forward only
        _linear("flux_ffn0_fwd", "linear", 3072, 12288, (16, 128, 64, 32, 64, 16, 128, 128, 32, 64, 16, 64, 128, 32, 16, 64),
                (4608,) * 16, range(16), backward=False),
        # the modulated LayerNorm that opens a sublayer, on the float32 stream of both roles, training
        dict(name="wan_norm", path="norm", batch=2, tokens=32760, W=1536, hidden="f32"),
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, v // multiple * multiple)


def draw(rng):
    path = rng.choice(("linear", "linear", "linear", "linear", "gated", "stacked", "fp8", "norm"))
    if path == "norm":
        W = rng.choice((_log_int(rng, 256, 5120, 8), 1536, 3072, 5120))
        batch = rng.randint(1, 4)
        hidden = rng.choice(("f32", "bf16"))
        return dict(path=path, batch=batch, tokens=_log_int(rng, 64, min(32760, 2 * 32760 * 1536 // (batch * W))),
                    W=W, hidden=hidden)
    dtype = rng.choice(("bf16", "bf16", "f32")) if path == "linear" else "bf16"
    wide = rng.random() < 0.5
    K = rng.choice((_log_int(rng, 256, 3072, 16), 1536, 3072))
    N = rng.choice((_log_int(rng, 256, 3072, 16), 1536, 3072))
    if wide and dtype == "bf16" and path != "stacked":
        ffn = rng.choice((8960, 12288, 14336))
        K, N = (ffn, N) if rng.random() < 0.5 else (K, ffn)
    # no more products than a quarter of the largest listed case; float32 runs on a slower unit
    most = 27280 * 3072 * 14336 / 4 / (16 if dtype == "f32" else 3 if path == "stacked" else 1)
    tokens = _log_int(rng, 200, int(max(400, min(65520, most / (K * N)))))
    n = rng.choice((1, 2, 2, 3, 4, 8))
    if path == "gated":
        tokens = max(1, tokens // n) * n  # one gate row per sample
        lengths = [tokens // n] * n
    else:
        cuts = sorted(rng.randint(0, tokens) for _ in range(n - 1))
        lengths = [b - a for a, b in zip([0, *cuts], [*cuts, tokens])]
    rank = rng.choice((16, 32, 64, 64, 128, 128, 256))
    ranks = [rank if path == "stacked" else rng.choice((rank, rank, max(8, rank // 2))) for _ in range(n)]
    adapters = list(range(n))
    if n > 1 and rng.random() < 0.3:
        adapters[rng.randrange(n)] = -1  # the teacher's rows: base only
    masters = dtype == "bf16" and path in ("linear", "stacked") and rng.random() < 0.3
    case = _linear("", path, K, N, ranks, lengths, adapters, scale=rng.choice((1.0, 2.0)), dtype=dtype,
                   masters=masters, backward=rng.random() < 0.7)
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs

def _inputs(case, seed):
    """Everything the call reads, on the GPU: activations and gradients N(0, 1), base N(0, 1/in),
    lora_a U(±1/sqrt(in)) (its Kaiming initialisation), lora_b N(0, 0.02) (a trained adapter)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def randn(*shape, std=1.0, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device=DEV).mul_(std).to(dtype)

    if case["path"] == "norm":
        B, T, W = case["batch"], case["tokens"], case["W"]
        hdt = torch.float32 if case["hidden"] == "f32" else torch.bfloat16
        return dict(x=randn(B, T, W, dtype=hdt), table=randn(1, 6, W, std=W ** -0.5, dtype=torch.float32),
                    component=randn(B, 6, W, std=0.2, dtype=torch.float32), dy=randn(B, T, W))
    K, N = case["K"], case["N"]
    ranks, lengths = _ints(case["ranks"]), _ints(case["lengths"])
    M = sum(lengths)
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    adt = torch.float32 if case["masters"] else dt
    G = 3 if case["path"] == "stacked" else 1
    d = dict(x=randn(M, K, dtype=dt),
             w=[randn(N, K, std=K ** -0.5, dtype=dt) for _ in range(G)],
             b=[randn(N, std=K ** -0.5, dtype=dt) for _ in range(G)],
             As=[[(torch.rand(r, K, generator=g, device=DEV) * 2 - 1).mul_(K ** -0.5).to(adt) for r in ranks]
                 for _ in range(G)],
             Bs=[[randn(N, r, std=0.02, dtype=adt) for r in ranks] for _ in range(G)])
    if case["path"] == "gated":
        d["residual"] = randn(M, N, dtype=torch.float32)
        d["gate"] = randn(len(lengths), N, std=0.5, dtype=torch.float32)
    if case["backward"]:
        d["dy"] = [randn(M, N, dtype=torch.float32 if case["path"] == "gated" else dt) for _ in range(G)]
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    state = dict(case=case, d=d)
    if case["path"] == "norm":
        for k in ("x", "table", "component"):
            d[k].requires_grad_(True)
        return state
    state["routing"] = mlora.SegmentRouting.from_lengths(_ints(case["lengths"]), _ints(case["adapters"]))
    state["scales"] = [case["scale"]] * len(_ints(case["ranks"]))
    leaves = [d["x"], *(a for As in d["As"] for a in As), *(b for Bs in d["Bs"] for b in Bs)]
    if case["path"] == "gated":
        leaves.append(d["residual"])
    if case["backward"]:
        for t in leaves:
            t.requires_grad_(True)
    state["leaves"] = leaves
    # what a model keeps beside its frozen base: the transposed copy that dX reads, or the e4m3 base
    if case["path"] == "fp8":
        state["wq"], state["ws"] = mlora.kernels.quantize_rows_fp8(d["w"][0])
        state["wq_t"] = state["wq"].t().contiguous()
    elif case["path"] != "stacked" and case["dtype"] == "bf16" and case["backward"]:
        state["w_t"] = d["w"][0].t().contiguous()
    return state


def run(state):
    case, d = state["case"], state["d"]
    if case["path"] == "norm":
        y = mlora.modulated_layer_norm(d["x"], d["table"], d["component"], 1, 0)
        return [y.detach(), *torch.autograd.grad(y, [d["x"], d["table"], d["component"]], d["dy"])]
    with torch.set_grad_enabled(case["backward"]):
        routing, scales = state["routing"], state["scales"]
        w, b, As, Bs = d["w"][0], d["b"][0], d["As"][0], d["Bs"][0]
        if case["path"] == "linear":
            ys = [mlora.multi_lora_linear(d["x"], w, b, As, Bs, scales, routing, weight_t=state.get("w_t"))]
        elif case["path"] == "gated":
            ys = [mlora.multi_lora_linear_gated(d["x"], w, b, As, Bs, scales, routing, d["residual"], d["gate"],
                                                weight_t=state.get("w_t"))]
        elif case["path"] == "fp8":
            ys = [mlora.multi_lora_linear_fp8(d["x"], state["wq"], state["ws"], b, As, Bs, scales, routing,
                                              wq_t=state["wq_t"])]
        else:
            ys = list(mlora.shared_input_multi_lora(d["x"], d["w"], d["b"], d["As"], d["Bs"], scales, routing))
    if not case["backward"]:
        return ys
    return [*(y.detach() for y in ys), *torch.autograd.grad(ys, state["leaves"], d["dy"])]


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    if case["path"] == "norm":
        n, W = case["batch"] * case["tokens"], case["W"]
        ex = 4 if case["hidden"] == "f32" else 2
        # the hidden state in, the output out; then the hidden state and dY in, dX out
        return {"bytes": n * W * (ex + 2 + ex + 2 + ex), "flops": 30 * n * W}
    K, N = case["K"], case["N"]
    ranks, lengths, adapters = _ints(case["ranks"]), _ints(case["lengths"]), _ints(case["adapters"])
    M, G = sum(lengths), 3 if case["path"] == "stacked" else 1
    e = 4 if case["dtype"] == "f32" else 2
    ea = 4 if case["masters"] or case["dtype"] == "f32" else 2
    ew = 1 if case["path"] == "fp8" else e
    eo = 4 if case["path"] == "gated" else e
    used = sorted({a for a, m in zip(adapters, lengths) if a >= 0 and m > 0})
    adapter_bytes = G * ea * sum(ranks[a] * (K + N) for a in used)
    lora = G * sum(2 * m * ranks[a] * (K + N) for a, m in zip(adapters, lengths) if a >= 0)
    nbytes = M * K * e + G * (K * N * ew + M * N * eo) + adapter_bytes
    if case["path"] == "gated":
        nbytes += M * N * 4
    flops = 2 * M * K * N * G + lora
    if case["backward"]:
        # dY, the input and the base again, dX and the adapter gradients
        nbytes += M * K * e * 2 + G * (K * N * ew + M * N * eo) + 2 * adapter_bytes
        flops += 2 * M * K * N * G + 2 * lora
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["path"] != "norm" and case["dtype"] == "f32":
        # float32 sums of thousands of products: 3e-7 to 1.4e-6 from the exact result
        return {"rel": 6e-6, "max": 1e-3}
    if case["path"] == "fp8":
        # the e4m3 operands are the same; one bf16 rounding of the results, and a value that falls on
        # the other side of an e4m3 tie now and then
        return {"rel": 7e-3, "max": 0.1}
    # one rounding of each result to bf16: 1.7e-3 from the exact result
    return {"rel": 7e-3, "max": 0.1}


# ------------------------------------------------------------------ 64 bits

def _e4m3_rows(t):
    """Per-row absmax e4m3 quantisation: (values, scale) in 64 bits."""
    amax = t.abs().amax(dim=1, keepdim=True)
    amax = torch.where(amax > 0, amax, torch.full_like(amax, 448.0))
    most = torch.full_like(amax, 448.0)  # tensor / tensor: a true quotient (scalar / tensor multiplies by a reciprocal)
    return (t * (most / amax)).to(torch.float8_e4m3fn).double(), (amax / most).double()


def exact(case, seed):
    d = _inputs(case, seed)
    if case["path"] == "norm":
        x, g = d["x"].double(), d["dy"].double()
        table, comp = d["table"].double()[0], d["component"].double()
        W = case["W"]
        n = x - x.mean(dim=2, keepdim=True)
        rstd = (n.square().mean(dim=2, keepdim=True) + 1e-6).rsqrt()
        n *= rstd
        s = 1 + (table[1] + comp[:, 1]).unsqueeze(1)
        y = n * s + (table[0] + comp[:, 0]).unsqueeze(1)
        dcomp = torch.zeros_like(comp)
        dcomp[:, 1], dcomp[:, 0] = (g * n).sum(dim=1), g.sum(dim=1)
        gn = g * s
        dx = (gn - gn.mean(dim=2, keepdim=True) - n * (gn * n).sum(dim=2, keepdim=True) / W) * rstd
        return [y, dx, dcomp.sum(dim=0, keepdim=True), dcomp]
    lengths, adapters = _ints(case["lengths"]), _ints(case["adapters"])
    scale, G, x = case["scale"], len(d["w"]), d["x"].double()
    ys, dx, dres = [], None, None
    dAs = [[torch.zeros_like(a, dtype=torch.float64) for a in As] for As in d["As"]]
    dBs = [[torch.zeros_like(b, dtype=torch.float64) for b in Bs] for Bs in d["Bs"]]
    off = [0]
    for m in lengths:
        off.append(off[-1] + m)
    if case["path"] == "gated":
        gate = d["gate"].double().repeat_interleave(torch.tensor(lengths, device=DEV), dim=0)
    for g in range(G):
        As, Bs = [[t.double() for t in ts] for ts in (d["As"][g], d["Bs"][g])]
        if case["path"] == "fp8":
            wq, ws = _e4m3_rows(d["w"][g].float())
            xq, xs = _e4m3_rows(d["x"].float())
            y = (xq @ wq.t()) * xs * ws.t() + d["b"][g].double()
        else:
            w = d["w"][g].double()
            y = x @ w.t() + d["b"][g].double()
        for s, a in enumerate(adapters):
            if a >= 0 and lengths[s]:
                rows = slice(off[s], off[s + 1])
                y[rows] += scale * ((x[rows] @ As[a].t()) @ Bs[a].t())
        ys.append(d["residual"].double() + y * gate if case["path"] == "gated" else y)
        if not case["backward"]:
            continue
        dy = d["dy"][g].double()
        if case["path"] == "gated":
            dres, dy = dy, dy * gate
        if case["path"] == "fp8":
            dyq, dys = _e4m3_rows(d["dy"][g].float() * ws.float().t())
            part = (dyq @ wq) * dys
        else:
            part = dy @ w
        for s, a in enumerate(adapters):
            if a >= 0 and lengths[s]:
                rows = slice(off[s], off[s + 1])
                gr = scale * (dy[rows] @ Bs[a])
                part[rows] += gr @ As[a]
                dAs[g][a] += gr.t() @ x[rows]
                dBs[g][a] += scale * (dy[rows].t() @ (x[rows] @ As[a].t()))
        dx = part if dx is None else dx + part
    if not case["backward"]:
        return ys
    out = [*ys, dx, *(t for ts in dAs for t in ts), *(t for ts in dBs for t in ts)]
    return out + ([dres] if dres is not None else [])
