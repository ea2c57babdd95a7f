"""Performance cases of the mHC layer on one GPU: what a program that uses this package has it do.

Five kinds of call, each through the module or function that a program calls:

  infer     MHCLayer.forward under torch.no_grad (decoding, serving)
  train     MHCLayer.forward and the gradients of x and of every parameter
  dynamic   MHCLayer.forward_dynamic (per-token mappings) and its gradients
  rewire    MHCRewire around a square Linear and its gradients, the Linear's weight among them
  residual  residual_add_agg

The ranges (``draw``): stream counts from 2 to 64, channels from 32 to 8192 with ragged ones among them, 1 to 32768
tokens (128 and up in training), fp32, bf16 and fp16 activations, the output in fp32 (the default) or in the activations' dtype.
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mhc-mlx_amd"))

from mhc_mlx_amd import MHCLayer, MHCRewire, residual_add_agg  # noqa: E402

ITERS, EPS = 20, 1e-6
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
PARAMS = ("H_pre_raw", "H_post_raw", "H_res_raw", "rms_weight")


def _case(kind, tokens, n, C, dtype, out=None):
    return {"kind": kind, "tokens": tokens, "n": n, "C": C, "dtype": dtype, "out": out or dtype}


def listed():
    return [
        # a decoding step of a small batch: one launch, latency-bound
        dict(_case("infer", 32, 4, 2048, "bf16"), name="infer_32x4x2048_bf16"),
        # one token through the stream count that MHCRewire defaults to, with the default fp32 output
        dict(_case("infer", 1, 32, 1024, "bf16", "fp32"), name="infer_1x32x1024_bf16_fp32"),
        # a small fp32 training step with a ragged token count and a width that is no power of two
        dict(_case("train", 257, 8, 1000, "fp32"), name="train_257x8x1000_fp32"),
        # the headline training step: 8 sequences of 4096 tokens
        dict(_case("train", 32768, 4, 4096, "bf16"), name="train_32768x4x4096_bf16"),
        # training with 32 streams in bf16, and the same in fp32 (the parameters' and the default output's dtype)
        dict(_case("train", 8192, 32, 512, "bf16"), name="train_8192x32x512_bf16"),
        dict(_case("train", 4096, 32, 512, "fp32"), name="train_4096x32x512_fp32"),
        # 16 streams in fp16, ragged: an odd token count, a width that is no multiple of 128
        dict(_case("train", 3001, 16, 1100, "fp16"), name="train_3001x16x1100_fp16"),
        # the largest stream count that the kernels take
        dict(_case("train", 2048, 64, 512, "bf16"), name="train_2048x64x512_bf16"),
        # per-token mappings: many small projections beside the activations
        dict(_case("dynamic", 16384, 16, 1024, "bf16"), name="dynamic_16384x16x1024_bf16"),
        dict(_case("dynamic", 8192, 4, 4096, "bf16"), name="dynamic_8192x4x4096_bf16"),
        # MHCRewire with its default 32 streams around a Linear(1024, 1024): 32 channels a stream, fp32 output
        dict(_case("rewire", 8192, 32, 32, "bf16", "fp32"), name="rewire_8192x32x32_bf16_fp32"),
        # the block helper between two layers: bf16 activations, fp32 results
        dict(_case("residual", 8192, 4, 4096, "bf16", "fp32"), name="residual_8192x4x4096_bf16"),
    ]


def draw(rng):
    kind = rng.choice(("infer", "train", "train", "dynamic", "rewire", "residual"))
    n = rng.choice((2, 4, 4, 4, 8, 8, 16, 16, 32, 32, 64, rng.randint(3, 15), rng.randint(17, 63)))
    dtype = rng.choice(("bf16", "bf16", "fp32", "fp16"))
    out = dtype if rng.random() < 0.6 else "fp32"
    if kind == "residual":
        out = "fp32"  # its results are fp32
    step = rng.choice((128, 128, 8, 1))
    most_c = 8192 if kind != "rewire" else max(32, 4096 // n)  # a Linear of at most 4096 x 4096
    C = max(step, int(math.exp(rng.uniform(math.log(32), math.log(most_c)))) // step * step)
    least_t = 1 if kind in ("infer", "residual") else 128  # a training step has a batch, a decoding step may be one token
    most_t = max(least_t, min(32768.0, 1.2e8 / (n * C)))
    if kind == "dynamic":
        most_t = max(least_t, min(most_t, 3.3e7 / (n * n)))
    if kind == "rewire":
        most_t = max(least_t, min(most_t, 3.4e10 / (n * C) ** 2))  # the Linear's share is a library product
    tokens = int(math.exp(rng.uniform(math.log(least_t), math.log(most_t))))
    return _case(kind, tokens, n, C, dtype, out)


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Every tensor of a case, from the seed alone: N(0, 1) activations, cotangents and logits, norm weights near 1."""
    T, n, C = case["tokens"], case["n"], case["C"]
    dt, out = DTYPES[case["dtype"]], DTYPES[case["out"]]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)

    d = {}
    if case["kind"] == "rewire":
        d["x"] = normal(T, n * C, dtype=dt)
        d["weight"] = (normal(n * C, n * C) / math.sqrt(n * C)).to(dt)
        d["dout"] = normal(T, n * C, dtype=out)
    else:
        d["x"] = normal(T, n, C, dtype=dt)
        if case["kind"] == "residual":
            d["res"] = normal(T, n, C, dtype=dt)
        elif case["kind"] != "infer":
            d["dout"] = normal(T, n, C, dtype=out)
    per = (T,) if case["kind"] == "dynamic" else ()
    d["H_pre_raw"] = normal(*per, n)
    d["H_post_raw"] = normal(*per, n)
    d["H_res_raw"] = normal(*per, n, n)
    d["rms_weight"] = 1.0 + 0.02 * normal(C)
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    n, C, kind = case["n"], case["C"], case["kind"]
    s = {"case": dict(case), "return_dtype": DTYPES[case["out"]]}
    if kind == "residual":
        s.update(x=d["x"], res=d["res"], H_pre=torch.sigmoid(d["H_pre_raw"]))
        return s
    kw = dict(sinkhorn_iters=ITERS, eps=EPS, device="cuda")
    if kind == "rewire":
        inner = torch.nn.Linear(n * C, n * C, bias=False, device="cuda", dtype=DTYPES[case["dtype"]])
        module = MHCRewire(inner, n * C, n=n, return_dtype=s["return_dtype"], **kw)
        layer = module.mhc
        with torch.no_grad():
            inner.weight.copy_(d["weight"])
    else:
        module = layer = MHCLayer(n, C, **kw)
    with torch.no_grad():
        for name in PARAMS if kind != "dynamic" else PARAMS[3:]:
            getattr(layer, name).copy_(d[name])
    s["module"] = module
    s["x"] = d["x"]
    if kind == "infer":
        return s
    s["x"].requires_grad_(True)
    s["dout"] = d["dout"]
    if kind == "dynamic":
        s["H"] = [d[name].requires_grad_(True) for name in PARAMS[:3]]
        s["wrt"] = [s["x"], *s["H"], layer.rms_weight]
    elif kind == "rewire":
        s["wrt"] = [s["x"], *(getattr(layer, name) for name in PARAMS[:3]), module.inner.weight]
    else:
        s["wrt"] = [s["x"], *(getattr(layer, name) for name in PARAMS)]
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "residual":
        with torch.no_grad():
            return residual_add_agg(s["x"], s["res"], s["H_pre"])
    if kind == "infer":
        with torch.no_grad():
            return s["module"](s["x"], return_dtype=s["return_dtype"])
    if kind == "dynamic":
        out = s["module"].forward_dynamic(s["x"], *s["H"], return_dtype=s["return_dtype"])
    elif kind == "rewire":
        out = s["module"](s["x"])
    else:
        out = s["module"](s["x"], return_dtype=s["return_dtype"])
    return (out.detach(), *torch.autograd.grad(out, s["wrt"], s["dout"]))


def work(case):
    T, n, C = case["tokens"], case["n"], case["C"]
    sx, so = DTYPES[case["dtype"]].itemsize, DTYPES[case["out"]].itemsize
    tile = T * n * C
    params = 4 * ((T if case["kind"] == "dynamic" else 1) * (n * n + 2 * n) + C)
    if case["kind"] == "residual":
        return {"bytes": tile * (2 * sx + so) + 4 * T * C + 4 * n, "flops": 3 * tile}
    mix = 2 * n * tile  # M X; the backward has M^T dout and dout X^T
    if case["kind"] == "infer":
        return {"bytes": tile * (sx + so) + params, "flops": mix + 6 * tile}
    if case["kind"] == "rewire":
        return {"bytes": tile * (2 * sx + 2 * so) + 2 * sx * (n * C) ** 2 + 2 * params,
                "flops": 3 * mix + 8 * tile + 6 * tile * n * C}
    return {"bytes": tile * (2 * sx + 2 * so) + 2 * params, "flops": 3 * mix + 20 * tile}


def tolerance(case):
    if case["kind"] == "rewire" and case["dtype"] != "fp32":  # the Linear's 16-bit input, output and gradients
        return {"rel": 1.2e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.6e-3, "max": 1.4e-2}
    if "bf16" in (case["dtype"], case["out"]):
        return {"rel": 8e-3, "max": 4e-2}  # one rounding of an output: 2^-9 of it
    if "fp16" in (case["dtype"], case["out"]):
        return {"rel": 1e-3, "max": 6e-3}
    return {"rel": 1e-5, "max": 2e-4}


# ---------------------------------------------------------------- the same in 64 bits
def _sinkhorn64(H):
    P = torch.exp(H - H.amax(-1, keepdim=True))
    for _ in range(ITERS):
        r = P.sum(-1, keepdim=True)
        P = P * torch.where(r > EPS, 1.0 / r, torch.ones_like(r))
        c = P.sum(-2, keepdim=True)
        P = P * torch.where(c > EPS, 1.0 / c, torch.zeros_like(c))
    return P


def _layer64(x, a, p, M, w):
    y = (a.unsqueeze(-1) * x).sum(-2)
    yn = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * w
    return torch.matmul(M, x) + p.unsqueeze(-1) * yn.unsqueeze(-2)


def _rewire64(x, a, p, M, weight):
    T, n, C = x.shape
    inner = torch.matmul((a.unsqueeze(-1) * x).reshape(T, n * C), weight.t()).reshape(T, n, C)
    return p.unsqueeze(-1) * (inner + torch.matmul(M * a, x))


def exact(case, seed):
    d = {k: v.double() if k not in ("x", "dout", "res") else v for k, v in _inputs(case, seed).items()}
    kind, T, n, C = case["kind"], case["tokens"], case["n"], case["C"]
    if kind == "residual":
        out = d["x"].double() + d["res"].double()
        return out, (torch.sigmoid(d["H_pre_raw"]).unsqueeze(-1) * out).sum(-2)
    x = d["x"].reshape(T, n, C)
    out = torch.empty(T, n, C, dtype=torch.float64, device="cuda")
    grad = kind != "infer"
    dx = torch.empty_like(out) if grad else None
    per = kind == "dynamic"
    H = [d[k].requires_grad_(grad) for k in PARAMS[:3]]
    last = (d["weight"] if kind == "rewire" else d["rms_weight"]).requires_grad_(grad)
    chunk = max(1, (1 << 25) // (n * C))
    with torch.set_grad_enabled(grad):
        full = [torch.sigmoid(H[0]), 2.0 * torch.sigmoid(H[1]), _sinkhorn64(H[2])]
        leaves = [t.detach().requires_grad_(grad) for t in full]
        sums = [torch.zeros_like(t) for t in (*leaves, last)] if grad else None
        for at in range(0, T, chunk):
            part = slice(at, min(T, at + chunk))
            xc = x[part].double().requires_grad_(grad)
            hc = [t[part] if per else t for t in leaves]
            o = (_rewire64 if kind == "rewire" else _layer64)(xc, *hc, last)
            out[part] = o.detach()
            if grad:
                got = torch.autograd.grad(o, [xc, *leaves, last], d["dout"].reshape(T, n, C)[part].double())
                dx[part] = got[0]
                for s, v in zip(sums, got[1:]):
                    s += v
        if not grad:
            return out
        dH = torch.autograd.grad(full, H, sums[:3])
    if kind == "rewire":
        out, dx = out.reshape(T, n * C), dx.reshape(T, n * C)
    return (out, dx, *dH, sums[3])
