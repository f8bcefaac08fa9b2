"""Cases that stand for the work users give this framework, for timing and for comparing builds.

A case is one MoE layer's grouped GEMM work on one GPU: `groups` experts, `rows` routed tokens in
all, weights of `n` x `k` per expert. Its other fields:

  op      "fwd", "dgrad", "wgrad", "bwd" (dgrad and wgrad of one layer) or "step" (all three)
  dtype   "bf16", "fp16", "e4m3" or "e5m2"; an fp8 gradient of "dgrad", "wgrad", "bwd" and "step"
          is e5m2 (the hybrid training recipe), the other operand `dtype`
  sizes   "host": row counts known to the host; "device": an int64 tensor that a router wrote
  spread  "even" (equal groups) or "skewed" (ragged, some may be empty)
  via     "plan": the plan objects a program keeps for its layer's buffers; "call": the functions
          that take and return torch tensors

A case's row counts are the same for every seed but for their order over the groups, so `work` is
exact. Activations are N(0, 1), weights N(0, 1 / k) and gradients N(0, 1) / 64, as they are at the
layers of a normalised network; fp8 tensors are quantised with tensor-wise scales (amax to the
format's largest value), one scale per expert for weights.
"""
import importlib
import math
import random

import torch

gg = importlib.import_module("groupgemm-cktile-optimized_amd")

DEV = "cuda"
TORCH_TYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
GG_TYPE = {"bf16": gg.DType.BF16, "fp16": gg.DType.FP16, "e4m3": gg.DType.FP8_E4M3, "e5m2": gg.DType.FP8_E5M2}
FP8 = ("e4m3", "e5m2")


def _case(name, op, dtype, sizes, spread, via, groups, rows, n, k):
    return {"name": name, "op": op, "dtype": dtype, "sizes": sizes, "spread": spread, "via": via, "groups": groups,
            "rows": rows, "n": n, "k": k}


def listed():
    return [
        # The smallest layer of the benchmark's configurations: launches and latency.
        _case("plumbing", "fwd", "bf16", "host", "even", "plan", 4, 1024, 512, 1024),
        # Serving, decode: a few tokens per expert, the weights of many experts read once. Sizes
        # come from the router and stay on the GPU.
        _case("decode_gate_up", "fwd", "bf16", "device", "skewed", "plan", 32, 512, 4096, 7168),
        # The same in fp8, the other projection, fewer local experts and a larger batch.
        _case("decode_down_fp8", "fwd", "e4m3", "device", "skewed", "plan", 8, 256, 7168, 2048),
        # Serving, a short prompt: enough tokens per expert to fill half a tile.
        _case("short_prompt", "fwd", "bf16", "host", "even", "plan", 8, 1024, 4096, 7168),
        # One dense expert whose tiles barely fill the GPU once.
        _case("low_occupancy", "fwd", "bf16", "host", "even", "plan", 1, 2048, 7168, 2048),
        # Many experts with row and column counts that no tile divides.
        _case("tails", "fwd", "bf16", "host", "even", "plan", 32, 16640, 2880, 2880),
        # The headline benchmark: prefill or training forward of a gate + up projection.
        _case("gate_up", "fwd", "bf16", "host", "even", "plan", 8, 32768, 4096, 7168),
        # The largest: dense experts in fp16.
        _case("dense_fp16", "fwd", "fp16", "host", "even", "plan", 8, 32768, 14336, 4096),
        # Training, gradient of the activations of a down projection.
        _case("down_dgrad", "dgrad", "bf16", "host", "even", "plan", 8, 32768, 7168, 2048),
        # Training, gradient of the weights with the router's ragged sizes.
        _case("ragged_wgrad", "wgrad", "bf16", "device", "skewed", "plan", 32, 16640, 2880, 2880),
        # Training in fp8: both gradients of a layer.
        _case("fp8_backward", "bwd", "e4m3", "host", "skewed", "plan", 8, 32768, 4096, 7168),
        # A layer's training step from a torch program: forward and both gradients, router's sizes.
        _case("layer_step", "step", "bf16", "device", "skewed", "call", 16, 8192, 2816, 2048),
    ]


def draw(rng):
    def log_uniform(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        op = rng.choice(["fwd"] * 6 + ["dgrad", "dgrad", "wgrad", "wgrad", "bwd", "step"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "e4m3", "e4m3"] + (["e5m2"] if op == "fwd" else []))
        via = rng.choice(["plan", "plan", "plan", "call"])
        sizes = rng.choice(["host", "device"])
        if via == "call" and dtype in FP8 and op in ("fwd", "step"):
            sizes = "host"  # the fp8 forward function takes host sizes
        groups = log_uniform(1, 64)
        rows = groups * log_uniform(1, 8192)
        if groups > 1:
            rows += rng.randrange(groups)
        # layer widths: whole tiles, a multiple of 64, or the finest a row of 16-byte pieces allows
        # (fp8: of 16)
        fine = 16 if dtype in FP8 else 8
        n, k = (max(s, log_uniform(512, 14336) // s * s) for s in (rng.choice([256, 64, fine]), rng.choice([256, 64, fine])))
        case = {"op": op, "dtype": dtype, "sizes": sizes, "spread": rng.choice(["even", "skewed"]), "via": via,
                "groups": groups, "rows": rows, "n": n, "k": k}
        w = work(case)
        # below the largest listed case in time, and (device-size weight gradients) inside the
        # entry points' 2 GiB per operand
        slow = w["flops"] / (2.4e15 if dtype in FP8 else 1.2e15) + w["bytes"] / 4e12
        if slow < 2.2e-3 and (rows + 1024) * max(n, k) * 2 < 2**31:
            return case


def _counts(case):
    """Rows of each group, the same for every seed."""
    g, rows = case["groups"], case["rows"]
    if case["spread"] == "even":
        return [rows // g + (i < rows % g) for i in range(g)]
    rng = random.Random("%d/%d/%d/%d" % (g, rows, case["n"], case["k"]))
    share = [rng.gammavariate(3.0, 1.0) for _ in range(g)]  # a router's load: spread of 0.6 of the mean
    cut, at = [0], 0.0
    for s in share[:-1]:
        at += s
        cut.append(int(rows * at / sum(share)))
    cut.append(rows)
    return [b - a for a, b in zip(cut, cut[1:])]


def _randn(shape, scale, dtype, gen, per_group=False):
    """(tensor, fp32 scales or None): N(0, scale^2) values in a 16-bit type, or quantised to fp8 with
    one scale, or one for each leading index."""
    if dtype not in FP8:
        return torch.randn(shape, dtype=TORCH_TYPE[dtype], device=DEV, generator=gen).mul_(scale), None
    top = torch.finfo(TORCH_TYPE[dtype]).max
    out = torch.empty(shape, dtype=TORCH_TYPE[dtype], device=DEV)
    if per_group:
        scales = torch.empty(shape[0], dtype=torch.float32, device=DEV)
        for i in range(shape[0]):
            v = torch.randn(shape[1:], device=DEV, generator=gen).mul_(scale)
            scales[i] = v.abs().amax() / top
            out[i] = (v / scales[i]).to(TORCH_TYPE[dtype])
        return out, scales
    v = torch.randn(shape, device=DEV, generator=gen).mul_(scale)
    scales = (v.abs().amax() / top).reshape(1)
    out.copy_((v / scales).to(TORCH_TYPE[dtype]))
    return out, scales


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    counts = _counts(case)
    random.Random(seed).shuffle(counts)
    g, rows, n, k, op, dtype = (case[f] for f in ("groups", "rows", "n", "k", "op", "dtype"))
    s = {"case": case, "counts": counts}
    s["lens"] = torch.tensor(counts, dtype=torch.int64, device=DEV) if case["sizes"] == "device" else None
    if op != "dgrad":
        s["x"], s["x_scale"] = _randn((rows, k), 1.0, dtype, gen)
    if op != "wgrad":
        s["w"], s["w_scale"] = _randn((g, n, k), k**-0.5, dtype, gen, per_group=True)
    if op != "fwd":
        s["dy"], s["dy_scale"] = _randn((rows, n), 1.0 / 64, "e5m2" if dtype in FP8 else dtype, gen)
    if op not in ("fwd", "dgrad") and dtype in FP8:
        s["x_scales"] = s["x_scale"].expand(g).contiguous()  # weight gradients take x's scale per expert
    return s


def _plan(op, s):
    """(plan, its output buffer) for one pass over the state's buffers."""
    case = s["case"]
    g, rows, n, k, dtype = (case[f] for f in ("groups", "rows", "n", "k", "dtype"))
    f8 = dtype in FP8
    a, a_scale = (s["x"], s["x_scale"]) if op == "fwd" else (s["dy"], s["dy_scale"])
    b, b_scale = (s["x"], s.get("x_scales")) if op == "wgrad" else (s["w"], s["w_scale"])
    a_type = GG_TYPE["e5m2" if f8 and op != "fwd" else dtype]
    shape = {"fwd": (rows, n), "dgrad": (rows, k), "wgrad": (g, n, k)}[op]
    out = torch.empty(shape, dtype=torch.bfloat16 if f8 else TORCH_TYPE[dtype], device=DEV)
    p = [t.data_ptr() for t in (a, b, out)]
    sp = [t.data_ptr() for t in (a_scale, b_scale)] if f8 else [0, 0]
    stream = torch.cuda.current_stream().cuda_stream
    if s["lens"] is not None:
        code = {"fwd": gg.OP_FORWARD, "dgrad": gg.OP_DGRAD, "wgrad": gg.OP_WGRAD}[op]
        return gg.DeviceLensPlan(code, a_type, GG_TYPE[dtype], g, rows, n, k, s["lens"].data_ptr(), 0, *p, stream, *sp), out
    if op != "fwd":
        return gg.BackwardPlan(op, a_type, n, k, s["counts"], *p, stream, other_dtype=GG_TYPE[dtype], grad_scale=sp[0],
                               other_scale=sp[1]), out
    if f8:
        return gg.Fp8Plan(a_type, n, k, s["counts"], p[0], p[1], sp[0], sp[1], p[2], stream), out
    be = gg.make_mi355x_backend()
    why = be.prepare(gg.GroupedGemmProblem(a_type, g, n, k, s["counts"], *p), stream)
    if why:
        raise RuntimeError(why)
    return be, out


PASSES = {"fwd": ("fwd",), "dgrad": ("dgrad",), "wgrad": ("wgrad",), "bwd": ("dgrad", "wgrad"),
          "step": ("fwd", "dgrad", "wgrad")}


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["via"] == "plan":
        s["plans"] = [_plan(op, s) for op in PASSES[case["op"]]]
    return s


def _call(op, s):
    sizes = s["counts"] if s["lens"] is None else s["lens"]
    if s["case"]["dtype"] in FP8:
        if op == "fwd":
            return gg.grouped_gemm_fp8(s["x"], s["w"], sizes, s["x_scale"], s["w_scale"])
        if op == "dgrad":
            return gg.grouped_gemm_dgrad_fp8(s["dy"], s["w"], sizes, s["dy_scale"], s["w_scale"])
        return gg.grouped_gemm_wgrad_fp8(s["dy"], s["x"], sizes, s["dy_scale"], s["x_scales"])
    if op == "fwd":
        return gg.grouped_gemm(s["x"], s["w"], sizes)
    if op == "dgrad":
        return gg.grouped_gemm_dgrad(s["dy"], s["w"], sizes)
    return gg.grouped_gemm_wgrad(s["dy"], s["x"], sizes)


def run(state):
    case = state["case"]
    if case["via"] == "call":
        return {op: _call(op, state) for op in PASSES[case["op"]]}
    stream = torch.cuda.current_stream().cuda_stream
    for plan, _ in state["plans"]:
        plan.run(stream)
    return {op: out for op, (_, out) in zip(PASSES[case["op"]], state["plans"])}


def work(case):
    rows, n, k, dtype = (case[f] for f in ("rows", "n", "k", "dtype"))
    es = 1 if dtype in FP8 else 2
    used = sum(c > 0 for c in _counts(case))  # weights of groups without rows are not read
    x, y, w = rows * k, rows * n, n * k
    moved = {"fwd": es * (x + used * w) + 2 * y, "dgrad": es * (y + used * w) + 2 * x,
             "wgrad": es * (x + y) + 2 * case["groups"] * w}
    passes = PASSES[case["op"]]
    return {"bytes": sum(moved[p] for p in passes), "flops": 2.0 * rows * n * k * len(passes)}


def tolerance(case):
    # The outputs' own rounding: against float64 the relative error is 1.7e-3 in bf16 and 2.1e-4 in
    # fp16, and sums in another order move an output by at most one unit in the last place (1 / 128
    # and 1 / 1024 of it).
    if case["dtype"] == "fp16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 6e-3, "max": 3e-2}


def exact(case, seed):
    s = _inputs(case, seed)
    rows, n, k, g = (case[f] for f in ("rows", "n", "k", "groups"))
    shape = {"fwd": (rows, n), "dgrad": (rows, k), "wgrad": (g, n, k)}
    out = {op: torch.zeros(shape[op], dtype=torch.float64, device=DEV) for op in PASSES[case["op"]]}

    def wide(name, pick, scale):
        v = s[name][pick].to(torch.float64)
        return v if scale is None else v * scale.to(torch.float64)

    at = 0
    for i, m in enumerate(s["counts"]):
        r, at = slice(at, at + m), at + m
        if m == 0:
            continue
        x = wide("x", r, s["x_scale"]) if "x" in s else None
        w = wide("w", i, None if s["w_scale"] is None else s["w_scale"][i]) if "w" in s else None
        dy = wide("dy", r, s["dy_scale"]) if "dy" in s else None
        if "fwd" in out:
            out["fwd"][r] = x @ w.T
        if "dgrad" in out:
            out["dgrad"][r] = dy @ w
        if "wgrad" in out:
            out["wgrad"][i] = dy.T.contiguous() @ x
    return out
