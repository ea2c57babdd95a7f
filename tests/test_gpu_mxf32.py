"""GPU parity of the fp32-MFMA post-combine (csrc/mxf32.hpp) against the float64 oracle.

It serves MHCRewire's post-combine above n = 8 (and ragged rows above n = 4) where C is no multiple of 64.  The sizes
sit at the edges of its splits: the 16-row blocks of streams, slabs of 64 columns that hold part of a token, one token
or many, a partial last slab, rows taken one element at a time, and waves that walk several slabs.
"""

import numpy as np
import pytest
import torch

from oracle import mhc_oracle as O
from tests._helpers import (GRAD_TOL, TOL, TORCH_DT, dev_tensor, kernels_missing, np_of, params, rel_err, rng,
                            to_dtype_np, tokens_dot)

from mhc_mlx_amd import ops
from mhc_mlx_amd.reference import mixing_matrix_from_logits

pytestmark = pytest.mark.gpu

SHAPES = [(3, 5, 3), (70, 6, 18), (5, 8, 31), (40, 9, 4), (9, 16, 64), (33, 16, 20), (2, 13, 1000), (11, 17, 32),
          (65, 32, 32), (7, 32, 2), (3, 24, 100), (5, 33, 12), (2, 48, 76), (9, 49, 7), (4, 64, 32), (1, 64, 1)]


@pytest.mark.parametrize("T,n,C", SHAPES)
@pytest.mark.parametrize("xdt,odt", [("f32", "f32"), ("bf16", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("grid", [None, 1])
def test_mxf32_post_combine(T, n, C, xdt, odt, grid, knobs):
    """Output and every gradient, reruns bitwise equal; with one workgroup per CU at most."""
    if grid is not None:
        knobs("MHC_MIX_FWD_GRID", grid)
        knobs("MHC_MIX_BWD_GRID", grid)
    g = rng(9300 + T + n + C)
    x, y = (to_dtype_np(g.standard_normal((T, n, C)), xdt) for _ in range(2))
    dout = to_dtype_np(g.standard_normal((T, n, C)), odt)
    hpre, hpost, hres, _ = params(g, n, C)

    def run():
        ts = [dev_tensor(v, xdt).requires_grad_(True) for v in (x, y)]
        ps = [dev_tensor(v).requires_grad_(True) for v in (hpre, hpost, hres)]
        out = ops.post_combine(*ts, *ps, sinkhorn_iters=20, eps=1e-5, output_dtype=None if odt == "f32" else ts[0].dtype)
        return [out.detach(), *torch.autograd.grad(out, [*ts, *ps], dev_tensor(dout, odt))]

    got, again = run(), run()
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    refs = [O.post_combine(x, y, hpre, hpost, hres, 20, 1e-5),
            *O.post_combine_backward(x, y, hpre, hpost, hres, dout, 20, 1e-5)]
    for name, a, r in zip(("out", "dx", "dy", "dH_pre", "dH_post", "dH_res"), got, refs):
        tol = TOL[odt] if name == "out" else (TOL[xdt] if name in ("dx", "dy") else GRAD_TOL)
        assert rel_err(np_of(a), r, floor=1e-3) < tol, (name, rel_err(np_of(a), r))


@pytest.mark.parametrize("T,n,C", [(8000, 12, 20), (21000, 12, 7), (4500, 12, 32), (8000, 24, 20), (4500, 24, 32), (21000, 24, 7),
                                   (8000, 40, 20), (4500, 64, 32)])
def test_mxf32_many_slabs_per_wave(T, n, C, knobs):
    """One workgroup per CU: every wave walks two slabs at least, the next one's loads ahead of this one's rows; against
    float64 and the VALU kernels (MHC_MIX32=0)."""
    assert T * C // 64 > 2 * 4 * torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n)
    x, y, dout = (torch.randn(T, n, C, generator=g, device="cuda") for _ in range(3))
    M = torch.rand(n, n, generator=g, device="cuda")
    res = []
    for on in (1, 0):
        knobs("MHC_MIX32", on)
        knobs("MHC_MIX_FWD_GRID", 1)
        knobs("MHC_MIX_BWD_GRID", 1)
        ts = [t.clone().requires_grad_(True) for t in (x, M, y)]
        out = ops.stream_mix_add_hip_autograd(*ts)
        res.append([out.detach(), *torch.autograd.grad(out, ts, dout)])
    xd, Md, gd = x.double(), M.double(), dout.double()
    res.append([torch.matmul(Md, xd) + y.double(), torch.matmul(Md.t().contiguous(), gd), tokens_dot(gd, xd), gd])
    for a, b, r in zip(*res):
        assert float((a - r).abs().max() / r.abs().max()) < 1e-5
        assert float((a - b).abs().max() / r.abs().max()) < 1e-5


@pytest.mark.parametrize("n,C", [(6, 31), (12, 4), (20, 20), (40, 12), (64, 1)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_mxf32_keeps_non_finite_values_in_their_channel(n, C, bad):
    """A slab holds several tokens: an infinity or a NaN of x reaches its own token and channel of out, one of dout those
    of dx and dy."""
    T, t, c = 33, 16, C // 2
    g = rng(9700 + n)
    x, y, dout = (dev_tensor(g.standard_normal((T, n, C))) for _ in range(3))
    x[t, 1, c] = dout[t, n - 1, c] = bad
    M = dev_tensor(g.uniform(size=(n, n)))
    ts = [v.requires_grad_(True) for v in (x, M, y)]
    out = ops.stream_mix_add_hip_autograd(*ts)
    dx, _, dy = torch.autograd.grad(out, ts, dout)
    for v in (out, dx, dy):
        broken = ~torch.isfinite(v)
        assert broken[t, :, c].any()
        broken[t, :, c] = False
        assert not broken.any()


def test_mxf32_unaligned_rows():
    """Operands at addresses that are no multiple of four elements give the same values."""
    T, n, C = 30, 12, 24
    g = rng(9500)
    vals = [dev_tensor(g.standard_normal((T, n, C))) for _ in range(3)]
    hp, hq, hr, _ = (dev_tensor(v) for v in params(g, n, C))
    res = []
    for shift in (0, 1):
        ts = []
        for v in vals:
            buf = torch.empty(v.numel() + 1, device="cuda")
            t = buf[shift:shift + v.numel()].view(T, n, C)
            ts.append(t.copy_(v))
        xs, ys = (t.detach().requires_grad_(True) for t in ts[:2])
        ps = [p.clone().requires_grad_(True) for p in (hp, hq, hr)]
        out = ops.post_combine(xs, ys, *ps)
        res.append([out.detach(), *torch.autograd.grad(out, [xs, ys, *ps], ts[2])])
    for a, b in zip(*res):
        assert rel_err(np_of(a), np_of(b)) < 1e-6


@pytest.mark.parametrize("T,n,C", [(300, 12, 100), (2000, 16, 20), (500, 24, 40), (900, 32, 32), (130, 6, 333), (100, 40, 100)])
def test_mxf32_rounds_no_more_than_its_sums_need(T, n, C):
    """fp32 out is no further from float64 than the same sum in numpy's fp32 with the (larger) y added last; begun with y,
    every product is rounded against it, three to five times the error.  The bound's 15% covers the order of the mix."""
    g = rng(9600 + n)
    x, y = (g.standard_normal((T, n, C)).astype(np.float32) for _ in range(2))
    M = (g.uniform(size=(n, n)) / n).astype(np.float32)
    out = np_of(ops.stream_mix_add_hip(dev_tensor(x), dev_tensor(M), dev_tensor(y)))
    ref = np.matmul(M.astype(np.float64), x) + y
    own = np.zeros((T, n, C), np.float32)
    for k in range(n):
        own = (M[:, k, None].astype(np.float64) * x[:, None, k] + own).astype(np.float32)
    own = own + y
    assert np.linalg.norm(out - ref) < 1.15 * np.linalg.norm(own - ref), np.linalg.norm(out - ref) / np.linalg.norm(own - ref)


@pytest.mark.parametrize("T,n,C", [(300, 16, 100), (2000, 24, 20), (900, 32, 36), (600, 48, 100), (400, 64, 100)])
def test_mxf32_dM_is_as_exact_as_the_valu_kernels(T, n, C, knobs):
    """dM at fp32 is no further from float64 than the VALU kernel's (MHC_MIX32=0); see the layer's test of the same name."""
    g = rng(9650 + n)
    x, dout, y = (dev_tensor(g.standard_normal((T, n, C))) for _ in range(3))
    ref = tokens_dot(dout.double(), x.double())
    err = []
    for on in (1, 0):
        knobs("MHC_MIX32", on)
        M = dev_tensor(g.uniform(size=(n, n)) / n).requires_grad_(True)
        out = ops.stream_mix_add_hip_autograd(x, M, y)
        err.append(float((torch.autograd.grad(out, M, dout)[0] - ref).norm() / ref.norm()))
    assert err[0] < 1.25 * err[1], err


@pytest.mark.parametrize("T,n,C,xdt,odt", [(4600, 12, 1000, "f32", "f32"), (2150, 16, 1000, "f32", "f32"), (2050, 16, 1000, "f32", "f32"),
                                           (3800, 16, 1000, "f32", "f32"), (3800, 16, 1000, "bf16", "f32"),
                                           (3100, 16, 1032, "bf16", "bf16"), (3800, 16, 1000, "f16", "f16"),
                                           (3100, 16, 1024, "f32", "f32")])
def test_mxf32_dispatch_of_large_calls(T, n, C, xdt, odt):
    """8 < n <= 16 on both sides of the lines at which calls beyond the caches go to the VALU kernels, against float64."""
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n)
    R = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, y, dout = R(T, n, C).to(TORCH_DT[xdt]), R(T, n, C).to(TORCH_DT[xdt]), R(T, n, C).to(TORCH_DT[odt])
    hp, hq, hr = R(n), R(n), R(n, n)
    ins = [t.clone().requires_grad_(True) for t in (x, y, hp, hq, hr)]
    out = ops.post_combine(*ins, sinkhorn_iters=20, eps=1e-5, output_dtype=TORCH_DT[odt])
    got = torch.autograd.grad(out, ins, dout)
    H = [t.double().requires_grad_(True) for t in (hp, hq, hr)]
    act = torch.sigmoid(H[0]), 2 * torch.sigmoid(H[1]), mixing_matrix_from_logits(H[2], iters=20, eps=1e-5)
    a, p, M = (t.detach() for t in act)
    xd, yd, gd = x.double(), y.double(), dout.double()
    Mf = p[:, None] * M * a
    ref = torch.matmul(Mf, xd) + p[:, None] * yd
    S, Y = tokens_dot(gd, xd), tokens_dot(gd, yd).diagonal()  # sums of g_i x_j and of g_i y_i
    sums = torch.matmul((S * M).t().contiguous(), p), torch.matmul(S * M, a) + Y, p[:, None] * S * a
    want = (torch.matmul(Mf.t().contiguous(), gd), p[:, None] * gd, *torch.autograd.grad(act, H, sums))
    assert float((out.detach() - ref).abs().max() / ref.abs().max()) < TOL[odt]
    for name, a, r in zip(("dx", "dy", "dH_pre", "dH_post", "dH_res"), got, want):
        assert float((a - r).abs().max() / r.abs().max()) < (TOL[xdt] if name in ("dx", "dy") else GRAD_TOL), name


@pytest.mark.parametrize("T,n,C", [(3, 5, 3), (9, 16, 64), (11, 17, 32), (2, 48, 76), (3, 64, 20)])
def test_mxf32_kernels_run(T, n, C):
    """The shapes above are the fp32-MFMA kernels' in both directions."""
    ts = [torch.randn(*s, device="cuda").requires_grad_(True) for s in ((T, n, C), (n, n), (T, n, C))]

    def step():
        out = ops.stream_mix_add_hip_autograd(*ts)
        torch.autograd.grad(out, ts, torch.ones_like(out))

    assert not kernels_missing(step, "mxf_fwd_kernel", "mxf_bwd_kernel")
