"""GPU parity of the narrow-token layer kernels (csrc/lv.hpp, n <= 8) against the float64 oracle.

They take tokens that are no whole workgroup of whole aligned chunks.  The sizes sit at the edges of their splits: 16, 32
and 64 lanes per token, one wave and several, one to four chunks per wave, the two-pass form, rows taken one, four and
eight elements at a time, n below its 2, 4 or 8 slots, and a last workgroup that is not full.
"""

import numpy as np
import pytest
import torch

from oracle import mhc_oracle as O
from tests._helpers import (GRAD_TOL, TOL, TORCH_DT, dev_tensor, kernels_missing, layer64, layer_grads64,
                            np_of, params, rel_err, rng, to_dtype_np)

from mhc_mlx_amd import ops

pytestmark = pytest.mark.gpu

EPS = 1e-5
SHAPES = [(37, 2, 1), (19, 3, 16), (70, 4, 64), (33, 4, 65), (18, 8, 100), (9, 5, 128), (21, 1, 132), (5, 2, 300),
          (7, 4, 777), (3, 6, 1000), (6, 4, 1040), (4, 8, 1030), (3, 2, 2056), (2, 3, 4100), (2, 8, 2500), (3, 4, 8008),
          (2, 4, 9001), (2, 7, 4200), (3, 7, 2501)]


@pytest.mark.parametrize("T,n,C", SHAPES)
@pytest.mark.parametrize("xdt,odt", [("f32", "f32"), ("bf16", "f32"), ("f16", "f16"), ("bf16", "bf16")])
@pytest.mark.parametrize("per_token", [False, True])
@pytest.mark.parametrize("grid", [None, 1])
def test_lv_forward_and_backward(T, n, C, xdt, odt, per_token, grid, knobs):
    """Output and every gradient, the backward on the whole chip and on one workgroup that walks every token; reruns are
    bitwise equal."""
    if grid is not None:
        knobs("MHC_FWD_GRID", grid)
        knobs("MHC_BWD_GRID", grid)
    g = rng(9700 + T + n + C)
    x, dout = to_dtype_np(g.standard_normal((T, n, C)), xdt), to_dtype_np(g.standard_normal((T, n, C)), odt)
    ps = params(g, n, C, per_token_B=T if per_token else None)
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward

    def run():
        xt = dev_tensor(x, xdt).requires_grad_(True)
        pt = [dev_tensor(v).requires_grad_(True) for v in ps]
        out = fn(xt, *pt, sinkhorn_iters=20, eps=EPS, output_dtype=None if odt == "f32" else xt.dtype)
        return [out.detach(), *torch.autograd.grad(out, [xt, *pt], dev_tensor(dout, odt))]

    got, again = run(), run()
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    refs = [O.mhc_forward_reference(x, *ps, sinkhorn_iters=20, eps=EPS),
            *O.mhc_backward_reference(x, *ps, dout, sinkhorn_iters=20, eps=EPS)]
    for name, a, r in zip(("out", "dx", "dH_pre", "dH_post", "dH_res", "d_w"), got, refs):
        tol = TOL[odt] if name == "out" else (TOL[xdt] if name == "dx" else GRAD_TOL)
        # dH_pre: at n = 1, and with one channel, the output does not depend on H_pre (the RMS norm undoes its scale) and
        # dH_pre is a difference of terms of the size of the sums behind it, about sqrt(T n C)
        floor = np.sqrt(T * n * C) if name == "dH_pre" and (n == 1 or C == 1) else 1e-3
        assert rel_err(np_of(a), r, floor=floor) < tol, (name, rel_err(np_of(a), r, floor=floor))


@pytest.mark.parametrize("T,n,C", [(18, 8, 100), (9, 5, 128), (5, 8, 252), (4, 8, 1028), (3, 7, 1030), (2, 8, 2500)])
@pytest.mark.parametrize("per_token", [False, True])
def test_lv_f16_with_f32_output(T, n, C, per_token, knobs):
    """fp16 streams with fp32 outputs at 4 < n <= 8, where the backward reads its rows a second time."""
    test_lv_forward_and_backward(T, n, C, "f16", "f32", per_token, None, knobs)


@pytest.mark.parametrize("n,C", [(4, 100), (8, 516), (3, 2000)])
def test_lv_matches_the_tile_kernel(n, C, knobs):
    """The same gradients as the tile kernel (MHC_BWD_LEGACY=1) to fp32 summation order, from operands whose addresses are
    no multiple of four elements too."""
    T = 50
    g = rng(9800 + n)
    x, dout = (dev_tensor(g.standard_normal((T, n, C))) for _ in range(2))
    ps = [dev_tensor(v) for v in params(g, n, C)]
    res = []
    for legacy, shift in ((0, 0), (0, 1), (1, 0)):
        knobs("MHC_BWD_LEGACY", legacy)
        buf = torch.empty(x.numel() + 1, device="cuda")
        xs = buf[shift:shift + x.numel()].view(T, n, C).copy_(x).detach().requires_grad_(True)
        pt = [p.clone().requires_grad_(True) for p in ps]
        out = ops.mhc_layer_forward(xs, *pt, eps=EPS)
        res.append([out.detach(), *torch.autograd.grad(out, [xs, *pt], dout)])
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert rel_err(np_of(a), np_of(b)) < 1e-5


@pytest.mark.parametrize("T,n,C", [(37, 4, 64), (1, 2, 33), (18, 8, 100), (5, 3, 128), (37, 4, 200), (3, 4, 777)])
@pytest.mark.parametrize("xdt,odt", [("f32", "f32"), ("bf16", "bf16"), ("f16", "f32")])
@pytest.mark.parametrize("eps", [0.0, 1e-30])
def test_lv_without_eps(T, n, C, xdt, odt, eps, knobs):
    """eps = 0, and an eps whose inv^3 overflows: a wave's token places past the last token have no RMS norm, and nothing
    of them may reach the parameter gradients (16, 32 and 64 lanes per token; counts that leave places empty)."""
    g = rng(9900 + T + C)
    x, dout = to_dtype_np(g.standard_normal((T, n, C)), xdt), to_dtype_np(g.standard_normal((T, n, C)), odt)
    ps = params(g, n, C)
    xt = dev_tensor(x, xdt).requires_grad_(True)
    pt = [dev_tensor(v).requires_grad_(True) for v in ps]
    out = ops.mhc_layer_forward(xt, *pt, sinkhorn_iters=20, eps=eps, output_dtype=None if odt == "f32" else xt.dtype)
    got = [out.detach(), *torch.autograd.grad(out, [xt, *pt], dev_tensor(dout, odt))]
    refs = [O.mhc_forward_reference(x, *ps, sinkhorn_iters=20, eps=eps),
            *O.mhc_backward_reference(x, *ps, dout, sinkhorn_iters=20, eps=eps)]
    for name, a, r in zip(("out", "dx", "dH_pre", "dH_post", "dH_res", "d_w"), got, refs):
        tol = TOL[odt] if name == "out" else (TOL[xdt] if name == "dx" else GRAD_TOL)
        assert rel_err(np_of(a), r, floor=1e-3) < tol, (name, rel_err(np_of(a), r, floor=1e-3))


@pytest.mark.parametrize("n,C", [(4, 64), (3, 33), (8, 100), (4, 300), (6, 777)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_lv_non_finite_stays_in_its_token(n, C, bad):
    """Several tokens share a wave: an infinity or a NaN of one reaches that token's rows and no other's."""
    T, t = 11, 5
    g = rng(9950 + C)
    x = dev_tensor(g.standard_normal((T, n, C)))
    x[t, n - 1, C // 2] = bad
    xt = x.requires_grad_(True)
    out = ops.mhc_layer_forward(xt, *(dev_tensor(v) for v in params(g, n, C)), eps=EPS)
    dx, = torch.autograd.grad(out, xt, dev_tensor(g.standard_normal((T, n, C))))
    others = [k for k in range(T) if k != t]
    assert torch.isfinite(out[others]).all() and torch.isfinite(dx[others]).all()
    assert not torch.isfinite(out[t, :, C // 2]).any() and torch.isnan(dx[t]).any()


def _fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(np.float32)


@pytest.mark.parametrize("T,n,C", [(400, 8, 100), (130, 7, 1001), (130, 8, 2001), (300, 8, 252)])
def test_lv_rounds_no_more_than_its_sums_need(T, n, C):
    """fp32 out and dx are no further from float64 than the same sums in numpy's fp32 with the mix first and the
    (larger) RMS term added last; the RMS term first rounds every product against it, 1.3 times the error.  The bound's 15%
    covers the order of the RMS sums, whose error a token's channels share."""
    g = rng(9990 + n)
    x, dout = (g.standard_normal((T, n, C)).astype(np.float32) for _ in range(2))
    M = O.mixing_matrix_from_logits(g.standard_normal((n, n)), 20, EPS).astype(np.float32)
    a, p = g.uniform(size=n).astype(np.float32), (2 * g.uniform(size=n)).astype(np.float32)
    w = (1 + 0.02 * g.standard_normal(C)).astype(np.float32)
    ts = [dev_tensor(v).requires_grad_(True) for v in (x, M, a, p, w)]
    out = ops.mhc_forward_fused_hip_autograd(*ts, eps=EPS)
    dx, = torch.autograd.grad(out, ts[0], dev_tensor(dout))

    y, d = np.zeros((T, C), np.float32), np.zeros((T, C), np.float32)
    for i in range(n):
        y, d = _fma(a[i], x[:, i], y), _fma(p[i], dout[:, i], d)
    ss = (y.astype(np.float64) ** 2).sum(-1, keepdims=True).astype(np.float32)
    inv = np.float32(1) / np.sqrt(ss / np.float32(C) + np.float32(EPS))
    kf = (inv * inv * inv / np.float32(C)) * (d.astype(np.float64) * y * w).sum(-1, keepdims=True).astype(np.float32)
    yn, dy = y * inv * w, d * inv * w - kf * y
    exact = (O.mhc_forward_fused_reference(x, M, a, p, w, eps=EPS), O.mhc_fused_backward(x, M, a, p, w, dout, eps=EPS)[0])
    for got, ref, mat, rows, last, scale in ((np_of(out), exact[0], M, x, yn, p), (np_of(dx), exact[1], M.T, dout, dy, a)):
        own = np.empty_like(x)
        for i in range(n):
            s = np.zeros((T, C), np.float32)
            for k in range(n):
                s = _fma(mat[i, k], rows[:, k], s)
            own[:, i] = _fma(scale[i], last, s)
        assert np.linalg.norm(got - ref) < 1.15 * np.linalg.norm(own - ref), np.linalg.norm(got - ref) / np.linalg.norm(own - ref)


# both sides of the lines at which the forward's dispatch changes kernels: tokens per CU, rows that share 128-byte lines,
# channels, calls beyond the caches
DISPATCH_FWD = [(200, 5, 512, "f32", "f32", True), (129, 6, 512, "bf16", "f32", True), (512, 8, 1000, "bf16", "f32", True),
                (513, 8, 1000, "bf16", "f32", True), (300, 7, 3000, "f32", "f32", True), (300, 7, 3072, "f32", "f32", True),
                (1100, 8, 64, "f16", "f32", True), (2100, 6, 1536, "bf16", "f32", True), (1300, 6, 136, "f32", "f32", True),
                (2100, 3, 6144, "bf16", "bf16", True), (9200, 4, 4096, "bf16", "bf16", True),
                (4100, 5, 1536, "bf16", "bf16", False), (4100, 5, 1536, "f16", "f32", False), (4000, 5, 1536, "bf16", "bf16", False),
                (5000, 6, 1536, "bf16", "f32", False), (2100, 6, 3072, "bf16", "bf16", False), (4000, 3, 3072, "bf16", "bf16", False),
                (8100, 3, 3000, "f32", "f32", False)]


@pytest.mark.parametrize("T,n,C,xdt,odt,per_token", DISPATCH_FWD)
def test_lv_forward_dispatch(T, n, C, xdt, odt, per_token):
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n + C)
    x = torch.randn(T, n, C, generator=g, device="cuda").to(TORCH_DT[xdt])
    per = (T,) if per_token else ()
    H = [torch.randn(*per, *s, generator=g, device="cuda") for s in ((n,), (n,), (n, n))]
    w = 1 + 0.02 * torch.randn(C, generator=g, device="cuda")
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward
    with torch.no_grad():
        out = fn(x, *H, w, sinkhorn_iters=20, eps=EPS, output_dtype=None if odt == "f32" else x.dtype)
    assert out.dtype == TORCH_DT[odt]
    for t in range(0, T, 1000):  # (in pieces: the reference is four times as wide)
        part = slice(t, min(T, t + 1000))
        ref = layer64(x[part], [h[part] for h in H] if per_token else H, w)
        assert float((out[part] - ref).abs().max() / ref.abs().max()) < TOL[odt]


DISPATCH_BWD = [(256, 4, 512, "bf16", "bf16", True), (257, 4, 512, "bf16", "bf16", True), (513, 4, 1024, "bf16", "bf16", True),
                (300, 4, 6144, "bf16", "bf16", True), (345, 4, 6144, "f16", "f16", True), (200, 3, 1024, "bf16", "bf16", True),
                (512, 3, 768, "bf16", "f32", True), (513, 3, 768, "f32", "f32", True), (400, 4, 2048, "f16", "f32", True),
                (250, 4, 512, "f32", "f32", True), (6200, 8, 512, "bf16", "bf16", True),
                (1100, 4, 1536, "bf16", "bf16", False), (1000, 4, 1536, "bf16", "bf16", False), (8200, 8, 512, "f16", "f16", False),
                (12300, 4, 512, "f32", "f32", False), (12300, 2, 1100, "f32", "f32", False), (12300, 3, 520, "bf16", "f32", False)]


@pytest.mark.parametrize("T,n,C,xdt,odt,per_token", DISPATCH_BWD)
def test_lv_backward_dispatch(T, n, C, xdt, odt, per_token):
    """Both sides of the lines at which the backward's dispatch changes kernels, every gradient against float64."""
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n + C)
    x = torch.randn(T, n, C, generator=g, device="cuda").to(TORCH_DT[xdt])
    dout = torch.randn(T, n, C, generator=g, device="cuda").to(TORCH_DT[odt])
    per = (T,) if per_token else ()
    leaves = [x, *(torch.randn(*per, *s, generator=g, device="cuda") for s in ((n,), (n,), (n, n))),
              1 + 0.02 * torch.randn(C, generator=g, device="cuda")]
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward
    ins = [t.clone().requires_grad_(True) for t in leaves]
    out = fn(*ins, sinkhorn_iters=20, eps=EPS, output_dtype=None if odt == "f32" else x.dtype)
    got = torch.autograd.grad(out, ins, dout)
    want = layer_grads64(leaves[0], leaves[1:4], leaves[4], dout, EPS)
    for name, a, r in zip(("dx", "dH_pre", "dH_post", "dH_res", "d_w"), got, want):
        assert float((a - r).abs().max() / r.abs().max()) < (TOL[xdt] if name == "dx" else GRAD_TOL), name


@pytest.mark.parametrize("T,n,C,xdt", [(9000, 3, 33, "f32"), (9000, 4, 64, "bf16"), (4500, 4, 100, "f32"), (2300, 4, 260, "bf16"),
                                       (2300, 8, 200, "f32"), (700, 2, 777, "f16"), (700, 4, 1040, "f32"), (560, 7, 1030, "f32"),
                                       (530, 3, 4100, "bf16"), (530, 8, 2501, "f32")])
@pytest.mark.parametrize("per_token", [False, True])
def test_lv_forward_walks_its_tokens(T, n, C, xdt, per_token, knobs):
    """One workgroup per CU: every wave (16, 32 or 64 lanes per token) or workgroup (two and more waves per token) takes
    two tokens at least, so the reduction buffers alternate and per-token parameters are loaded again."""
    knobs("MHC_FWD_GRID", 1)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    vec = 8 if xdt != "f32" and C % 8 == 0 else 4
    lanes = 64 if per_token or C > 32 * vec else (32 if C > 16 * vec else 16)
    assert T > 2 * cus * (4 * (64 // lanes) if C <= 64 * vec else 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n + C)
    x = torch.randn(T, n, C, generator=g, device="cuda").to(TORCH_DT[xdt])
    per = (T,) if per_token else ()
    H = [torch.randn(*per, *s, generator=g, device="cuda") for s in ((n,), (n,), (n, n))]
    w = 1 + 0.02 * torch.randn(C, generator=g, device="cuda")
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward
    with torch.no_grad():
        out = fn(x, *H, w, sinkhorn_iters=20, eps=EPS)
    ref = layer64(x, H, w, EPS)
    assert float((out - ref).abs().max() / ref.abs().max()) < 1e-5


@pytest.mark.parametrize("T,n,C,xdt,per_token,fwd,bwd", [
    (37, 4, 64, "f32", False, "lv_fwd_kernel", "lv_bwd_kernel"),
    (9, 4, 1001, "bf16", True, "lv_fwd_kernel", "lv_bwd_kernel"),
    (9, 8, 2501, "f32", False, "lv_fwd_kernel", "lv_bwd_kernel"),
    (9, 7, 2501, "bf16", False, "lv_fwd_kernel", "bwd_tile_kernel"),  # two 16-bit operands element by element, n > 4, C > 2048
    (9, 5, 1000, "f32", True, "fused_fwd_kernel", "lv_bwd_kernel"),
    (9, 4, 1024, "bf16", True, "lv_fwd_kernel", "fused_bwd_lw_kernel"),
    (9, 4, 4096, "bf16", False, "fused_fwd_full_kernel", "fused_bwd_lw_kernel")])
def test_lv_kernels_run(T, n, C, xdt, per_token, fwd, bwd):
    """Which kernels take a call, in each direction (outputs of x's dtype)."""
    per = (T,) if per_token else ()
    x = torch.randn(T, n, C, device="cuda").to(TORCH_DT[xdt]).requires_grad_(True)
    H = [torch.randn(*per, *s, device="cuda").requires_grad_(True) for s in ((n,), (n,), (n, n))]
    w = torch.ones(C, device="cuda").requires_grad_(True)
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward

    def step():
        out = fn(x, *H, w, eps=EPS, output_dtype=x.dtype)
        torch.autograd.grad(out, [x, *H, w], torch.ones_like(out))

    assert not kernels_missing(step, fwd, bwd)
