"""GPU parity of the fp32-MFMA layer kernels (csrc/lf32_fwd.hip, csrc/lf32_bwd.hip) against the float64 oracle.

They serve 8 < n <= 64 where the 16-bit MFMA kernels do not: fp32 or mixed dtypes, any C and row alignment.  The
sizes sit at the edges of their splits: the 16-row blocks of streams (n = 9, 16, 17, 32, 33, 48, 49, 64), the
64-channel slabs (C below, at and past a multiple), the element-wise rows (C not a multiple of 4), one slab per wave,
two and four, and the two-pass form for longer tokens.
"""

import numpy as np
import pytest
import torch

from oracle import mhc_oracle as O
from tests._helpers import (GRAD_TOL, TOL, TORCH_DT, dev_tensor, kernels_missing, layer64, np_of, params,
                            rel_err, rng, to_dtype_np, tokens_dot)

from mhc_mlx_amd import ops

pytestmark = pytest.mark.gpu

EPS = 1e-5
SHAPES = [(3, 9, 4), (4, 12, 1999), (3, 16, 2000), (70, 16, 64), (5, 16, 68), (300, 12, 100), (7, 16, 516), (4, 13, 1100), (3, 16, 2304),
          (40, 17, 65), (9, 32, 512), (6, 32, 516), (3, 24, 1030), (5, 32, 1096), (2, 20, 2500),
          (4, 33, 61), (6, 48, 512), (3, 49, 130), (5, 64, 192), (2, 64, 1000), (2, 40, 516)]


def _inputs(T, n, C, xdt, gdt, per_token):
    g = rng(9100 + T + n + C)
    x = to_dtype_np(g.standard_normal((T, n, C)), xdt)
    dout = to_dtype_np(g.standard_normal((T, n, C)), gdt)
    return x, dout, params(g, n, C, per_token_B=T if per_token else None)


@pytest.mark.parametrize("T,n,C", SHAPES)
@pytest.mark.parametrize("xdt,odt", [("f32", "f32"), ("bf16", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("per_token", [False, True])
def test_lf32_forward(T, n, C, xdt, odt, per_token, knobs):
    """Every split, one token per workgroup; the VALU kernels (MHC_FWD_MFMA=0) give the same to fp32 summation order."""
    x, _, ps = _inputs(T, n, C, xdt, xdt, per_token)
    xt, pt = dev_tensor(x, xdt), [dev_tensor(v) for v in ps]
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward

    def run():
        with torch.no_grad():
            return fn(xt, *pt, sinkhorn_iters=20, eps=EPS, output_dtype=None if odt == "f32" else xt.dtype)

    out, again = run(), run()
    assert torch.equal(out, again)
    ref = O.mhc_forward_reference(x, *ps, sinkhorn_iters=20, eps=EPS)
    # fp32: 64 products of rounded fp32 factors, summed in fp32; 16-bit: one rounding of that
    tol = 1e-5 if odt == "f32" else TOL[odt]
    assert rel_err(np_of(out), ref) < tol, rel_err(np_of(out), ref)
    knobs("MHC_FWD_MFMA", 0)
    assert rel_err(np_of(run()), np_of(out)) < tol


def test_lf32_forward_unaligned_and_non_finite():
    """x and out at addresses that are no multiple of a row's four elements take the element-wise rows, with the same
    values; an infinity and a NaN stay in the tokens and channels that they belong to."""
    T, n, C = 6, 20, 256
    x, _, ps = _inputs(T, n, C, "f32", "f32", False)
    pt = [dev_tensor(v) for v in ps]
    x[1, 3, 70] = np.inf
    x[4, 19, 255] = np.nan
    buf = torch.empty(T * n * C + 1, device="cuda")
    off = buf[1:].view(T, n, C)
    off.copy_(dev_tensor(x))
    with torch.no_grad():
        a = ops.mhc_layer_forward(dev_tensor(x), *pt, eps=EPS)
        b = ops.mhc_layer_forward(off, *pt, eps=EPS)
    assert torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0))
    bad = ~torch.isfinite(a)
    assert not bad[[0, 2, 3, 5]].any()
    assert bad[1, :, 70].all() and bad[4].all()  # a NaN reaches its token's RMS factor
    assert torch.isfinite(a[1][:, [0, 69, 71, 255]]).all()


@pytest.mark.parametrize("T,n,C", SHAPES)
@pytest.mark.parametrize("xdt,gdt", [("f32", "f32"), ("bf16", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("per_token", [False, True])
@pytest.mark.parametrize("grid", [None, 2])
def test_lf32_backward(T, n, C, xdt, gdt, per_token, grid, knobs):
    """Every gradient, with a grid of the whole chip and with two workgroups that walk many tokens each; reruns are
    bitwise equal."""
    if grid is not None:
        knobs("MHC_BWD_GRID", grid)
    x, dout, ps = _inputs(T, n, C, xdt, gdt, per_token)
    fn = ops.mhc_layer_forward_dynamic if per_token else ops.mhc_layer_forward

    def run():
        xt = dev_tensor(x, xdt).requires_grad_(True)
        pt = [dev_tensor(v).requires_grad_(True) for v in ps]
        out = fn(xt, *pt, sinkhorn_iters=20, eps=EPS, output_dtype=None if gdt == "f32" else xt.dtype)
        return torch.autograd.grad(out, [xt, *pt], dev_tensor(dout, gdt))

    got, again = run(), run()
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    refs = O.mhc_backward_reference(x, *ps, dout, sinkhorn_iters=20, eps=EPS)
    names = ("dx", "dH_pre", "dH_post", "dH_res", "d_w")
    for name, a, r in zip(names, got, refs):
        tol = TOL[xdt] if name == "dx" else GRAD_TOL
        assert rel_err(np_of(a), r) < tol, (name, rel_err(np_of(a), r))


@pytest.mark.parametrize("n,C", [(12, 100), (24, 260), (40, 68)])
def test_lf32_backward_activated_h(n, C):
    """The op-level VJP (activated H in and out) takes the same kernels."""
    T = 9
    x, dout, (hpre, hpost, hres, w) = _inputs(T, n, C, "f32", "f32", False)
    M = O.mixing_matrix_from_logits(hres, 20, EPS)
    a, p = 1.0 / (1.0 + np.exp(-hpre)), 2.0 / (1.0 + np.exp(-hpost))
    xt = dev_tensor(x).requires_grad_(True)
    ts = [dev_tensor(v).requires_grad_(True) for v in (a, p)]
    Mt = dev_tensor(M).requires_grad_(True)
    wt = dev_tensor(w).requires_grad_(True)
    out = ops.mhc_forward_fused_hip_autograd(xt, Mt, ts[0], ts[1], wt, eps=EPS)
    got = torch.autograd.grad(out, [xt, Mt, ts[0], ts[1], wt], dev_tensor(dout))
    ref_in = [t.detach().double().requires_grad_(True) for t in (xt, Mt, ts[0], ts[1], wt)]
    xd, Md, ad, pd, wd = ref_in
    y = (ad[None, :, None] * xd).sum(1)
    yn = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * wd
    ref = torch.matmul(Md, xd) + pd[None, :, None] * yn[:, None, :]
    for g, r in zip(got, torch.autograd.grad(ref, ref_in, dev_tensor(dout).double())):
        assert rel_err(np_of(g), r.cpu().numpy()) < GRAD_TOL


@pytest.mark.parametrize("T,n,C", [(130, 24, 100), (130, 32, 512), (600, 17, 512), (130, 48, 130), (130, 64, 512), (600, 40, 65)])
def test_lf32_dM_is_as_exact_as_the_valu_kernels(T, n, C, knobs):
    """dM at fp32 is no further from float64 than the VALU kernel's (MHC_BWD_MFMA=0): a slab's products are not one chain
    of 64, which is 1.3 to 1.7 times as far.  The bound's 25% covers the spread of a norm over n^2 entries and the chains of
    32 at n <= 32."""
    g = rng(9200 + n)
    x, dout = (dev_tensor(g.standard_normal((T, n, C))) for _ in range(2))
    ps = [dev_tensor(v) for v in (g.uniform(size=(n, n)) / n, g.uniform(size=n), 2 * g.uniform(size=n), np.ones(C))]
    ref = tokens_dot(dout.double(), x.double())
    err = []
    for mfma in (1, 0):
        knobs("MHC_BWD_MFMA", mfma)
        M = ps[0].clone().requires_grad_(True)
        out = ops.mhc_forward_fused_hip_autograd(x, M, *ps[1:], eps=EPS)
        err.append(float((torch.autograd.grad(out, M, dout)[0] - ref).norm() / ref.norm()))
    assert err[0] < 1.25 * err[1], err


@pytest.mark.parametrize("T,n,C,xdt", [(600, 9, 36, "f32"), (600, 12, 101, "bf16"), (600, 16, 260, "f32"), (530, 9, 1101, "f16"),
                                       (530, 16, 2304, "f32"), (600, 24, 100, "f32"), (600, 32, 130, "bf16"), (530, 20, 577, "f32"),
                                       (530, 32, 1096, "f32"), (550, 40, 68, "bf16"), (550, 64, 64, "f32"), (530, 49, 516, "f32"),
                                       (530, 33, 600, "f32")])
@pytest.mark.parametrize("per_token", [False, True])
def test_lf32_forward_walks_its_tokens(T, n, C, xdt, per_token, knobs):
    """One workgroup per CU takes two tokens and more: the next token's loads ahead of this one's stores, per-token
    parameters one token ahead or staged again, alternating reduction buffers, y's buffer of the two-pass form."""
    knobs("MHC_FWD_GRID", 1)
    assert T > 2 * torch.cuda.get_device_properties(0).multi_processor_count
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


@pytest.mark.parametrize("n,C", [(9, 36), (16, 200), (24, 101), (40, 64), (64, 130)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_lf32_backward_keeps_non_finite_values_in_their_token(n, C, bad, knobs):
    """Two workgroups walk every token: what one token holds reaches no other's dx."""
    knobs("MHC_BWD_GRID", 2)
    T, t = 9, 4
    g = rng(9300 + n)
    x = dev_tensor(g.standard_normal((T, n, C)))
    x[t, n - 1, C // 2] = bad
    xt = x.requires_grad_(True)
    out = ops.mhc_layer_forward(xt, *(dev_tensor(v) for v in params(g, n, C)), eps=EPS)
    dx, = torch.autograd.grad(out, xt, dev_tensor(g.standard_normal((T, n, C))))
    others = [k for k in range(T) if k != t]
    assert torch.isfinite(out[others]).all() and torch.isfinite(dx[others]).all()
    assert torch.isnan(dx[t]).any()


@pytest.mark.parametrize("T,n,C,xdt,odt", [(5, 9, 100, "f32", "f32"), (5, 16, 1000, "f16", "f16"), (5, 32, 512, "f32", "f32"),
                                           (5, 48, 516, "bf16", "f32"), (5, 64, 130, "f32", "f32")])
def test_lf32_kernels_run(T, n, C, xdt, odt):
    """The shapes above are the fp32-MFMA kernels' in both directions."""
    x, dout, ps = _inputs(T, n, C, xdt, odt, False)
    xt, pt = dev_tensor(x, xdt).requires_grad_(True), [dev_tensor(v).requires_grad_(True) for v in ps]

    def step():
        out = ops.mhc_layer_forward(xt, *pt, eps=EPS, output_dtype=None if odt == "f32" else xt.dtype)
        torch.autograd.grad(out, [xt, *pt], dev_tensor(dout, odt))

    assert not kernels_missing(step, "lf32_fwd_kernel", "lf32_bwd_kernel")
