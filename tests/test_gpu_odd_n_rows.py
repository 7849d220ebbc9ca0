"""The layers and stream operators at n = 3, 5, 6, 7 on each of their row
kernels: register rows (16-byte aligned arrays of a multiple of 4 channels),
channel-loop rows (any alignment and width up to 12288 channels, ragged
hidden sizes) and the generic kernels beyond; against the float64 oracle with
the layer tests' tolerances."""
import pytest
import torch

import mhc_ascend_amd as mhc
from mhc_ascend_amd import native
from oracle import reference as R
from tests.conftest import assert_close, grad_atol
from tests.test_gpu_dynamic import _check_dyn, _oracle_dyn
from tests.test_gpu_static import _check_static, _oracle_static

pytestmark = pytest.mark.gpu


def _place(t, device, shift):
    """t on the device, contiguous, `shift` elements past an aligned address."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=device)
    v = buf[shift:shift + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.is_contiguous() and (v.data_ptr() % 16 == 0) == (shift == 0)
    return v


# widths: edges of the register chunks, a ragged one, one past the register
# rows of n = 5..7 and one past the channel-loop rows
@pytest.mark.parametrize("n", [3, 5, 6, 7])
@pytest.mark.parametrize("B,C,shift", [(1, 4, 0), (9, 1040, 0), (700, 64, 0), (600, 2052, 0), (9, 1040, 1), (4, 1001, 0),
                                       (530, 1001, 1), (3, 4100, 0), (2, 12292, 0)])
@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
def test_static_rows(device, n, B, C, shift, x_dtype):
    d = R.static_layer_inputs(B, n, C, seed=n * 31 + B + C, x_dtype=x_dtype)
    x = _place(d["x"], device, shift).requires_grad_(True)
    ps = [d[k].to(device).requires_grad_(True) for k in ("weight", "H_pre", "H_post", "H_res")]
    out = mhc.mhc_layer_static(x, *ps)
    gx, *gp = torch.autograd.grad(out, [x, *ps], _place(d["grad"], device, shift))
    _check_static(d, (out, gx, gp), _oracle_static(d), x_dtype == torch.bfloat16, f"n={n} B={B} C={C} +{shift}")


@pytest.mark.parametrize("n,B,C,shift", [(3, 9, 128, 0), (3, 9, 128, 1), (3, 5, 160, 0), (3, 520, 1024, 0),
                                         (5, 7, 64, 0), (5, 7, 64, 1), (6, 9, 1040, 0), (6, 70, 80, 0), (7, 3, 4128, 0),
                                         (7, 300, 96, 0)])
@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
def test_dynamic_rows(device, n, B, C, shift, x_dtype):
    d = R.dynamic_layer_inputs(B, n, C, seed=n * 37 + B + C, x_dtype=x_dtype, alpha=0.2, phi_std=0.03, b_std=0.5)
    x = _place(d["x"], device, shift).requires_grad_(True)
    names = ["weight", "phi_pre", "phi_post", "phi_res", "alpha_pre", "alpha_post", "alpha_res", "b_pre", "b_post",
             "b_res"]
    ps = [d[k].to(device).requires_grad_(True) for k in names]
    out = mhc.mhc_layer_fused_dynamic_training(x, *ps)
    gx, *gp = torch.autograd.grad(out, [x, *ps], _place(d["grad"], device, shift))
    _check_dyn((out, gx, gp), _oracle_dyn(d), x_dtype, f"n={n} B={B} C={C} +{shift}")


@pytest.mark.parametrize("n", [3, 5, 6, 7])
@pytest.mark.parametrize("B,C,shift", [(5, 8, 0), (33, 1040, 0), (33, 1040, 1), (4, 1001, 0), (3, 4104, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_operator_rows(device, n, B, C, shift, dtype):
    g = torch.Generator().manual_seed(n + B + C)
    x = torch.randn(B, n, C, generator=g).to(dtype)
    y = torch.randn(B, C, generator=g).to(dtype)
    h1, h2 = torch.randn(B, n, generator=g), torch.randn(B, n, generator=g)
    m = torch.rand(B, n, n, generator=g)
    ca, co = torch.randn(B, C, generator=g).to(dtype), torch.randn(B, n, C, generator=g)
    # one rounding to bf16 of each result, 32-bit sums before it
    rtol, frac = (1e-3, 1e-5) if dtype == torch.float32 else (2.0 ** -8, 1e-3)

    xd = _place(x, device, shift).requires_grad_(True)
    hd = h1.to(device).requires_grad_(True)
    out = mhc.stream_aggregate(xd, hd)
    gx, gh = torch.autograd.grad(out, [xd, hd], _place(ca, device, shift))
    xr, hr = x.double().requires_grad_(True), h1.double().requires_grad_(True)
    ref = R.stream_aggregate(xr, hr)[0]
    rx, rh = torch.autograd.grad(ref, [xr, hr], ca.double())
    for nm, a, e in (("out", out, ref), ("dx", gx, rx), ("dh", gh, rh)):
        assert_close(a, e, rtol if nm != "dh" else 1e-3, grad_atol(e, frac if nm != "dh" else 1e-4), f"aggregate {nm}")

    xd = _place(x, device, shift).requires_grad_(True)
    yd = _place(y, device, shift).requires_grad_(True)
    hd, md = h2.to(device).requires_grad_(True), m.to(device).requires_grad_(True)
    out = mhc.stream_distribute_mix_add(yd, hd, md, xd)
    got = torch.autograd.grad(out, [yd, hd, md, xd], _place(co, device, shift))
    leaves = [t.double().requires_grad_(True) for t in (y, h2, m, x)]
    ref = R.stream_distribute_mix_add(*leaves)[0]
    want = torch.autograd.grad(ref, leaves, co.double())
    assert_close(out, ref, 1e-4, 1e-5, "distribute out")
    for nm, a, e in zip(("dy", "dh", "dM", "dx"), got, want):
        stored = nm in ("dy", "dx")
        assert_close(a, e, rtol if stored else 1e-3, grad_atol(e, frac if stored else 1e-4), f"distribute {nm}")


def _f32(t):
    return t.float().double()


def _mix32(h, y, m, x, last):
    """out_i = h_i y + sum_j m_ij x_j as fp32 fused products (exact in float64,
    rounded to fp32 each), the y term after the others or before them."""
    f = _f32
    n = x.shape[1]
    rows = []
    for i in range(n):
        s = torch.zeros_like(y) if last else f(h[i] * y)
        for j in range(n):
            s = f(s + m[i, j] * x[:, j])
        rows.append(f(s + h[i] * y) if last else s)
    return torch.stack(rows, 1)


@pytest.mark.parametrize("C", [512, 509])
@pytest.mark.parametrize("n", [3, 5, 6, 7])
def test_error_of_the_mix(device, n, C):
    """out of fp32 rows (register and channel-loop rows), from the coefficients that
    the library formed: the rms error against float64 is that of fp32 products with
    the term that is no stream's added after the mix, and not that with it rounded
    along with every product: the line lies between the two, formed on the same data,
    nearer to the second (r_h has its own rounding) (0.93 and 1.1 times 2^-24 at n = 3, 1.2 and 1.5 at n = 7)."""
    d = R.static_layer_inputs(300, n, C, seed=n)
    ps = [d[k].to(device) for k in ("weight", "H_pre", "H_post", "H_res")]
    out, _, saved = native.mhc_layer_static_fwd(d["x"].to(device), *ps)
    out, coef, x, w = out.cpu().double(), saved[:2 * n + n * n].cpu().double(), d["x"].double(), d["weight"].double()
    hp, h, m = coef[:n], coef[n:2 * n], coef[2 * n:].view(n, n)
    xa = (hp[:, None] * x).sum(1)
    y = xa / torch.sqrt((xa * xa).mean(-1, keepdim=True) + 1e-5) * w
    ref = torch.matmul(m, x) + h[:, None] * y[:, None]
    xa = torch.zeros_like(xa)
    for j in range(n):
        xa = _f32(xa + hp[j] * x[:, j])
    inv = _f32(1 / _f32(torch.sqrt((xa * xa).mean(-1, keepdim=True) + 1e-5)))
    y = _f32(_f32(xa * inv) * w)
    rel = lambda t: float((t - ref).norm() / ref.norm())
    err_last, err_first = rel(_mix32(h, y, m, x, True)), rel(_mix32(h, y, m, x, False))
    assert rel(out) < 0.25 * err_last + 0.75 * err_first, (rel(out), err_last, err_first)
