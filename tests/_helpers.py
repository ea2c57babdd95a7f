"""Shared test helpers: seeded inputs, dtype rounding, error metrics."""

import numpy as np
import torch

from oracle import mhc_oracle as O

from mhc_mlx_amd.reference import mixing_matrix_from_logits

TORCH_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def rng(seed: int) -> np.random.Generator:
    return np.random.default_rng(seed)


def to_dtype_np(a: np.ndarray, dt: str) -> np.ndarray:
    """Round float data to dt's grid (returned as float32 values)."""
    a = np.asarray(a, dtype=np.float32)
    if dt == "bf16":
        return O.bf16_round(a)
    if dt == "f16":
        return O.f16_round(a)
    return a


def dev_tensor(a: np.ndarray, dt: str = "f32", device: str = "cuda") -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(device).to(TORCH_DT[dt])


def np_of(t: torch.Tensor) -> np.ndarray:
    return t.detach().float().cpu().numpy().astype(np.float64)


def rel_err(got, ref, floor: float = 1e-30) -> float:
    """max |got - ref| / max(max |ref|, floor)  (the reference tests' relative metric).

    ``floor`` turns the metric into an absolute one for references whose
    largest element is below it (a gradient that is zero or nearly so).
    """
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    den = max(float(np.abs(ref).max()) if ref.size else 0.0, floor)
    return float(np.abs(got - ref).max()) / den if ref.size else 0.0


def max_abs(got, ref) -> float:
    return float(np.abs(np.asarray(got, np.float64) - np.asarray(ref, np.float64)).max())


# tolerance per output dtype (reference tests: fp32 1e-5, fp16 5e-3, bf16 2e-2)
TOL = {"f32": 1e-5, "f16": 5e-3, "bf16": 2e-2}

# Parameter gradients (dH_pre, dH_post, dH_res, d_rms_weight, dM) for every input dtype: the oracle
# sees the inputs already rounded to their I/O dtype, so the two sides differ only by fp32 rounding
# in the products and in fixed-order partial sums.  For zero-mean products summed as partial sums of
# depth d the expected relative error is about 2^-24 sqrt(d); the deepest sums tested (config 2: 64
# tokens x 8 channels per thread before a fixed tree) give ~1.3e-6 by that estimate and measure
# 9.5e-7, so the fp32 bar of the reference tests, 1e-5, holds with margin at every size.
GRAD_TOL = 1e-5


def params(g: np.random.Generator, n: int, C: int, per_token_B: int | None = None):
    """Seeded raw parameters: N(0,1) logits, rms weight 1 + 0.02 N(0,1)."""
    shp = (n,) if per_token_B is None else (per_token_B, n)
    hpre = g.standard_normal(shp).astype(np.float32)
    hpost = g.standard_normal(shp).astype(np.float32)
    hres = g.standard_normal(shp + (n,)).astype(np.float32)
    w = (1.0 + 0.02 * g.standard_normal(C)).astype(np.float32)
    return hpre, hpost, hres, w


def layer64(x, H, w, eps=1e-5, iters=20):
    """mhc_forward_reference (reference.py:164-184) in torch float64 on x's device, for calls too large for numpy."""
    a, p = torch.sigmoid(H[0].double()), 2 * torch.sigmoid(H[1].double())
    M = mixing_matrix_from_logits(H[2].double(), iters=iters, eps=eps)
    y = (a.unsqueeze(-1) * x.double()).sum(-2)
    yn = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + eps) * w.double()
    return torch.matmul(M, x.double()) + p.unsqueeze(-1) * yn.unsqueeze(-2)


def tokens_dot(a, b):
    """sum over tokens and channels of a[t, i, c] b[t, j, c], as one matrix product.  (torch's sum over many blocks in
    float64 has given a wrong value on the GPU now and then, so references form their long sums this way.)"""
    def rows(t):
        return t.transpose(0, 1).reshape(t.shape[1], -1)

    return torch.matmul(rows(a), rows(b).t().contiguous())


def layer_grads64(x, H, w, dout, eps=1e-5, iters=20):
    """(dx, dH_pre, dH_post, dH_res, d_w) of layer64 for the cotangent dout, in torch float64 on x's device."""
    per_token, C = H[0].dim() == 2, x.shape[2]
    H = [h.detach().double().requires_grad_(True) for h in H]
    act = torch.sigmoid(H[0]), 2 * torch.sigmoid(H[1]), mixing_matrix_from_logits(H[2], iters=iters, eps=eps)
    a, p, M = (t.detach() for t in act)
    x, g, w = x.detach().double(), dout.double(), w.detach().double()
    y, d = (a.unsqueeze(-1) * x).sum(-2), (p.unsqueeze(-1) * g).sum(-2)
    inv = torch.rsqrt(y.square().mean(-1, keepdim=True) + eps)
    dy = d * inv * w - inv ** 3 / C * (d * y * w).sum(-1, keepdim=True) * y
    yn = y * inv * w
    dx = torch.matmul(M.transpose(-1, -2).contiguous(), g) + a.unsqueeze(-1) * dy.unsqueeze(-2)
    dw = torch.matmul(torch.ones(1, x.shape[0], dtype=x.dtype, device=x.device), d * y * inv)[0]
    if per_token:
        sums = ((dy.unsqueeze(-2) * x).sum(-1), (g * yn.unsqueeze(-2)).sum(-1), torch.matmul(g, x.transpose(-1, -2).contiguous()))
    else:
        sums = tokens_dot(x, dy.unsqueeze(1))[:, 0], tokens_dot(g, yn.unsqueeze(1))[:, 0], tokens_dot(g, x)
    return (dx, *torch.autograd.grad(act, H, sums), dw)


def kernels_missing(fn, *names: str) -> list[str]:
    """Those of `names` that are no part of the name of any kernel that fn() launches."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    ran = [e.key for e in prof.key_averages()]
    return [n for n in names if not any(n in k for k in ran)]
