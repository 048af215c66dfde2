"""The workloads this library is timed on: the calls a program makes through
libnova_hip's C ABI (descriptors in hand, as a lowered module or the bench
holds them) and whole programs through libnova_run, over the range of sizes
those calls see.  Each case makes its inputs on the GPU from a seed and
returns every output of the call.

Kinds (a case's "kind"):
  matmul       nova.matmul in f32, the exact kernels (bit-identical to the
               CPU pipeline) or, with "mfma", the f32 matrix cores
  bmm          linalg.batch_matmul on 16-bit operands with f32 output
  linear       nova.linear (+ nova.gelu) on 16-bit operands, weight given as
               the transposed view of an [N, K] tensor, 16-bit output
  linear_bwd   nova.linear_backward on 16-bit operands, f32 gradients
  layer_norm   nova.layer_norm and nova.layer_norm_backward
  sce          nova.sce with nova.sce_backward (the fused entry point)
  gpt_step     a whole GPT training step in f32 through libnova_run, device
               resident, with exact or matrix-core f32 GEMMs
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "nova-compiler_amd"))
import nova_hip as nh  # noqa: E402
import nova_run  # noqa: E402
from gpt_program import gpt_step  # noqa: E402

F64 = torch.float64


def listed():
    return [
        # The smallest call: one f32 matmul of a program's small layers,
        # bound by its launch and one short chain per output.
        {"name": "matmul_f32_256", "kind": "matmul", "M": 256, "N": 256, "K": 256, "mfma": False},
        # The headline batch GEMM, and the largest contraction.
        {"name": "bmm_bf16_8x4096", "kind": "bmm", "dtype": "bf16", "batch": 8, "M": 4096,
         "N": 4096, "K": 4096},
        # The two products of an attention over 197 tokens (196 patches and
        # a class token), 8 images x 12 heads of 64: Q.K^T, then P.V.
        {"name": "bmm_f16_96x197x197x64", "kind": "bmm", "dtype": "f16", "batch": 96, "M": 197,
         "N": 197, "K": 64},
        {"name": "bmm_f16_96x197x64x197", "kind": "bmm", "dtype": "f16", "batch": 96, "M": 197,
         "N": 64, "K": 197},
        # An MLP up-projection over a full batch of 4096 tokens ...
        {"name": "linear_gelu_bf16_4096tok", "kind": "linear", "dtype": "bf16", "tokens": 4096,
         "K": 4096, "N": 11008, "gelu": True},
        # ... over one prompt, whose length is no multiple of anything ...
        {"name": "linear_gelu_bf16_1000tok", "kind": "linear", "dtype": "bf16", "tokens": 1000,
         "K": 4096, "N": 11008, "gelu": True},
        # ... and over one decoding step of 16 sequences.
        {"name": "linear_gelu_bf16_16tok", "kind": "linear", "dtype": "bf16", "tokens": 16,
         "K": 4096, "N": 11008, "gelu": True},
        # The backward of an MLP layer at the GPT step's widths over a
        # ragged micro-batch.
        {"name": "linear_bwd_bf16_6000x384x1536", "kind": "linear_bwd", "dtype": "bf16",
         "tokens": 6000, "K": 384, "N": 1536},
        # LayerNorm of a training step, forward and backward.
        {"name": "layer_norm_16384x4096", "kind": "layer_norm", "rows": 16384, "D": 4096},
        # The loss of a training step over a 32000-word vocabulary.
        {"name": "sce_4096x32000", "kind": "sce", "rows": 4096, "C": 32000},
        # A whole training step at the reference program's sizes, on the
        # matrix cores ...
        {"name": "gpt_step_mfma_8x1024", "kind": "gpt_step", "mfma": True, "B": 8, "T": 1024,
         "V": 50304, "D": 384, "H": 1536},
        # ... and a small step in the default mode, bit-exact f32 GEMMs.
        {"name": "gpt_step_exact_2x256", "kind": "gpt_step", "mfma": False, "B": 2, "T": 256,
         "V": 50304, "D": 384, "H": 1536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64, sometimes any number."""
    w = _log(rng, lo, hi)
    return max(lo, w // 64 * 64) if rng.random() < 0.75 else w


def draw(rng):
    kind = rng.choice(["matmul", "bmm", "bmm", "linear", "linear", "linear_bwd", "layer_norm", "sce",
                       "gpt_step"])
    if kind == "matmul":
        return {"kind": kind, "M": _log(rng, 16, 1024), "N": _log(rng, 16, 1024),
                "K": _log(rng, 16, 1024), "mfma": rng.random() < 0.5}
    if kind == "bmm":
        dtype = rng.choice(["bf16", "f16"])
        if rng.random() < 0.5:  # attention products over T tokens, heads of d
            T, d = _log(rng, 49, 1024), rng.choice([32, 64, 80, 128])
            batch = max(1, min(_log(rng, 12, 384), (1 << 26) // (T * T)))
            n, k = (T, d) if rng.random() < 0.5 else (d, T)
            return {"kind": kind, "dtype": dtype, "batch": batch, "M": T, "N": n, "K": k}
        m, n, k = (_width(rng, 128, 4096) for _ in range(3))
        return {"kind": kind, "dtype": dtype, "batch": rng.randint(1, 8), "M": m, "N": n, "K": k}
    if kind in ("linear", "linear_bwd"):
        c = {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16"]),
             "tokens": _log(rng, 1 if kind == "linear" else 128, 4096), "K": _width(rng, 128, 8192),
             "N": _width(rng, 128, 8192)}
        if kind == "linear":
            c["gelu"] = rng.random() < 0.5
        return c
    if kind == "layer_norm":
        d = _width(rng, 64, 8192)
        return {"kind": kind, "rows": _log(rng, 16, max(32, min(16384, (1 << 26) // d))), "D": d}
    if kind == "sce":
        c = _log(rng, 100, 60000)
        return {"kind": kind, "rows": _log(rng, 16, max(32, min(8192, (1 << 27) // c))), "C": c}
    mfma = rng.random() < 0.5
    d = rng.choice([64, 128, 192, 256, 384])
    b, t = rng.randint(1, 8), _log(rng, 32, 1024)
    v = _log(rng, 512, 50304)
    if not mfma:  # the exact GEMMs are slower: at most 2048 tokens
        b = max(1, min(b, 2048 // t))
    return {"kind": kind, "mfma": mfma, "B": b, "T": t, "V": v, "D": d, "H": 4 * d}


# ---------------------------------------------------------------------------

_DT = {"bf16": torch.bfloat16, "f16": torch.float16}
_CODE = {"bf16": nh.DT_BF16, "f16": nh.DT_F16}


def _inputs(case, seed):
    """The call's inputs, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))

    def normal(*s, std=1.0, mean=0.0):
        return torch.empty(s, device="cuda").normal_(mean, std, generator=g)

    def uniform(*s):
        return torch.empty(s, device="cuda").uniform_(-1.0, 1.0, generator=g)

    def ints(hi, *s):
        return torch.randint(0, hi, s, device="cuda", generator=g)

    c, kind = case, case["kind"]
    if kind == "matmul":
        return {"A": uniform(c["M"], c["K"]), "B": uniform(c["K"], c["N"])}
    if kind == "bmm":
        dt = _DT[c["dtype"]]
        return {"A": uniform(c["batch"], c["M"], c["K"]).to(dt),
                "B": uniform(c["batch"], c["K"], c["N"]).to(dt)}
    if kind == "linear":
        dt = _DT[c["dtype"]]
        return {"x": normal(c["tokens"], c["K"]).to(dt), "W": normal(c["N"], c["K"], std=0.02).to(dt),
                "b": normal(c["N"], std=0.02).to(dt)}
    if kind == "linear_bwd":
        dt = _DT[c["dtype"]]
        return {"go": normal(c["tokens"], c["N"]).to(dt), "x": normal(c["tokens"], c["K"]).to(dt),
                "W": normal(c["N"], c["K"], std=0.02).to(dt)}
    if kind == "layer_norm":
        return {"x": normal(c["rows"], c["D"]), "gamma": normal(c["D"], std=0.1, mean=1.0),
                "beta": normal(c["D"], std=0.1), "gy": normal(c["rows"], c["D"])}
    if kind == "sce":
        return {"logits": normal(c["rows"], c["C"], std=2.0),
                "labels": ints(c["C"], c["rows"]).to(torch.int32)}
    B, T, V, D, H = (c[k] for k in "BTVDH")
    return {"tok": ints(V, B, T).to(torch.int16), "tgt": ints(V, B, T).to(torch.int16),
            "pos": torch.arange(T, device="cuda").reshape(1, T),
            "wte": normal(V, D, std=0.02), "wpe": normal(T, D, std=0.02),
            "g1": normal(D, std=0.02, mean=1.0), "be1": normal(D, std=0.02),
            "w1": normal(D, H, std=0.02), "c1": normal(H, std=0.02), "w2": normal(H, D, std=0.02),
            "c2": normal(D, std=0.02), "g2": normal(D, std=0.02, mean=1.0),
            "be2": normal(D, std=0.02), "wlm": normal(D, V, std=0.02)}


def _call(name, *args):
    """A C-ABI entry point and its arguments, ready to be called."""
    d = [nh.memref_of(a) if isinstance(a, torch.Tensor) else a for a in args]
    refs = [nh.ref(a) if isinstance(a, ctypes.Structure) else a for a in d]
    return getattr(nh.lib(), "_mlir_ciface_nova_hip_" + name), refs, d


def prepare(case, seed):
    c, kind = case, case["kind"]
    t = _inputs(case, seed)
    out, calls = {}, []

    def empty(*s, dtype=torch.float32):
        return torch.empty(s, device="cuda", dtype=dtype)

    nh._bind_stream()
    if kind == "matmul":
        out["C"] = empty(c["M"], c["N"])
        if c["mfma"]:
            flags = nh.gemm_flags(nh.DT_F32, nh.DT_F32) | nh.GEMM_F32_MFMA
            calls = [_call("gemm", t["A"][None], t["B"][None], out["C"][None], None, flags)]
        else:
            calls = [_call("matmul_f32", t["A"], t["B"], out["C"])]
    elif kind == "bmm":
        out["C"] = empty(c["batch"], c["M"], c["N"])
        calls = [_call("batch_matmul_%s_f32" % c["dtype"], t["A"], t["B"], out["C"])]
    elif kind == "linear":
        code = _CODE[c["dtype"]]
        out["y"] = empty(c["tokens"], c["N"], dtype=_DT[c["dtype"]])
        epi = nh.EPI_BIAS_GELU if c["gelu"] else nh.EPI_BIAS
        calls = [_call("linear", t["x"], t["W"].t(), t["b"], out["y"],
                       nh.gemm_flags(code, code, epi, code))]
    elif kind == "linear_bwd":
        out["gx"] = empty(c["tokens"], c["K"])
        out["gw"] = empty(c["N"], c["K"])  # in the weight's own layout
        out["gb"] = empty(c["N"])
        calls = [_call("linear_backward", t["go"], t["x"], t["W"].t(), out["gx"], out["gw"].t(),
                       out["gb"], nh.gemm_flags(_CODE[c["dtype"]], nh.DT_F32))]
    elif kind == "layer_norm":
        R, D = c["rows"], c["D"]
        for k, s in (("y", (R, D)), ("sum", (R,)), ("rstd", (R,)), ("dx", (R, D)), ("dgamma", (D,)),
                     ("dbeta", (D,))):
            out[k] = empty(*s)
        calls = [_call("layer_norm_f32", t["x"], t["gamma"], t["beta"], out["y"], out["sum"],
                       out["rstd"], ctypes.c_float(1e-5)),
                 _call("layer_norm_backward_f32", t["gy"], t["x"], t["gamma"], out["sum"],
                       out["rstd"], out["dx"], out["dgamma"], out["dbeta"])]
    elif kind == "sce":
        out["loss"], out["grad"] = empty(1), empty(c["rows"], c["C"])
        calls = [_call("sce_fwd_bwd_f32", t["logits"], t["labels"], out["loss"], out["grad"])]
    else:
        prog = nova_run.Program(gpt_step(*(c[k] for k in "BTVDH")))
        prog.set_f32_gemm(nova_run.F32_GEMM_MFMA if c["mfma"] else nova_run.F32_GEMM_EXACT)
        res = [empty(*shape) for _, shape in prog.results("gpt_step")]
        return {"prog": prog, "args": list(t.values()), "out": res}
    return {"calls": calls, "out": out, "in": t}


def run(state):
    if "prog" in state:
        return state["prog"].run_device("gpt_step", *state["args"], results=state["out"])
    for fn, refs, _ in state["calls"]:
        rc = fn(*refs)
        if rc:
            nh.check(rc)
    return state["out"]


def work(case):
    c, kind = case, case["kind"]
    if kind == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if kind == "bmm":
        b, M, N, K = c["batch"], c["M"], c["N"], c["K"]
        return {"bytes": b * (2 * (M * K + K * N) + 4 * M * N), "flops": 2 * b * M * N * K}
    if kind == "linear":
        M, N, K = c["tokens"], c["N"], c["K"]
        return {"bytes": 2 * (M * K + K * N + N + M * N), "flops": 2 * M * N * K}
    if kind == "linear_bwd":
        M, N, K = c["tokens"], c["N"], c["K"]
        return {"bytes": 2 * (M * N + M * K + K * N) + 4 * (M * K + K * N + N),
                "flops": 4 * M * N * K + M * N}
    if kind == "layer_norm":
        R, D = c["rows"], c["D"]
        return {"bytes": 4 * (5 * R * D + 4 * R + 5 * D), "flops": 25 * R * D}
    if kind == "sce":
        R, C = c["rows"], c["C"]
        return {"bytes": 8 * R * C + 4 * R + 4, "flops": 8 * R * C}
    B, T, V, D, H = (c[k] for k in "BTVDH")
    N, weights = B * T, V * D + T * D + 2 * D * H + H + 5 * D + D * V
    return {"bytes": 8 * weights + 4 * N + 8 * T, "flops": 6 * N * D * V + 12 * N * D * H}


def tolerance(case):
    """About four times the error of these paths against exact()."""
    kind = case["kind"]
    if kind == "matmul" and not case["mfma"]:
        return "exact"  # the op's contract: one rounding order
    if kind == "linear":  # one rounding to the output type: 1.7e-3, 2.1e-4
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 1e-3, "max": 0.05}
    if kind == "gpt_step":  # 0.6e-6 to 4.7e-6
        return {"rel": 2e-5, "max": 2e-3}
    if kind in ("layer_norm", "sce"):  # up to 1.7e-7
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 4e-6, "max": 4e-4}  # 32-bit sums of up to 8192 terms: up to 0.6e-6


def exact(case, seed):
    kind = case["kind"]
    t = {k: v.to(F64) if v.is_floating_point() else v for k, v in _inputs(case, seed).items()}
    if kind in ("matmul", "bmm"):
        return {"C": torch.matmul(t["A"], t["B"])}
    if kind == "linear":
        y = t["x"] @ t["W"].t().contiguous() + t["b"]
        return {"y": torch.nn.functional.gelu(y, approximate="tanh") if case["gelu"] else y}
    if kind == "linear_bwd":
        return {"gx": t["go"] @ t["W"], "gw": t["go"].t().contiguous() @ t["x"],
                "gb": t["go"].sum(0)}
    if kind == "layer_norm":
        x, D = t["x"], case["D"]
        mean = x.mean(1, keepdim=True)
        rstd = 1.0 / torch.sqrt((x - mean).square().mean(1, keepdim=True) + 1e-5)
        xh = (x - mean) * rstd
        g = t["gy"] * t["gamma"]
        dx = (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True)) * rstd
        return {"y": xh * t["gamma"] + t["beta"], "sum": x.sum(1), "rstd": rstd[:, 0], "dx": dx,
                "dgamma": (t["gy"] * xh).sum(0), "dbeta": t["gy"].sum(0)}
    if kind == "sce":
        R = case["rows"]
        lab = t["labels"].long()
        lp = torch.log_softmax(t["logits"], 1)
        rows = torch.arange(R, device="cuda")
        loss = -lp[rows, lab].mean().reshape(1)
        grad = lp.exp_()
        grad[rows, lab] -= 1.0
        return {"loss": loss, "grad": grad / R}
    return _gpt_exact(case, t)


def _gpt_exact(case, t):
    """The training step in 64 bits, by autograd, in the program's result order."""
    B, T, V, D, H = (case[k] for k in "BTVDH")
    tok, tgt = ((t[k].long() & 0xffff).reshape(-1) for k in ("tok", "tgt"))
    names = ("wte", "wpe", "g1", "be1", "w1", "c1", "w2", "c2", "g2", "be2")
    p = {k: t[k].requires_grad_(True) for k in names}
    F = torch.nn.functional
    h = p["wte"][tok] + p["wpe"].repeat(B, 1)
    u = F.layer_norm(h, (D,), p["g1"], p["be1"]) @ p["w1"] + p["c1"]
    r = h + F.gelu(u, approximate="tanh") @ p["w2"] + p["c2"]
    flat = F.layer_norm(r, (D,), p["g2"], p["be2"])
    # The head by hand: its logits are most of the memory.
    f = flat.detach()
    logits = f @ t["wlm"]
    rows = torch.arange(B * T, device="cuda")
    lse = torch.logsumexp(logits, 1)
    loss = (lse - logits[rows, tgt]).mean().reshape(1)
    d = logits.sub_(lse[:, None]).exp_()
    d[rows, tgt] -= 1.0
    d /= B * T
    dwlm = f.t().contiguous() @ d
    flat.backward(d @ t["wlm"].t().contiguous())
    return [loss] + [p[k].grad for k in names] + [dwlm]
