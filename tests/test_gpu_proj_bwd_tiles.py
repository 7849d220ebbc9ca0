"""The projection backward over one to three output tiles at once (n = 5..8, more
than 1024 tokens; bf16 rows of n = 3): token counts at the edges of its 32-token stages and pairs of
them, widths at the edges of its 32-column waves and 128-column workgroups, both
storage types, and bf16 rows at an unaligned address; against the float64 oracle.

Tolerances as tests/test_gpu_wrapper.py: gradients 1e-3 with 1e-4 max|ref| (one
bf16 rounding, 2^-8, where stored in bf16)."""
import pytest
import torch

import mhc_ascend_amd as mhc
from oracle import reference as R
from tests.conftest import assert_close, grad_atol

pytestmark = pytest.mark.gpu

NAMES = ("rmsnorm_weight", "phi_pre", "phi_post", "phi_res", "alpha_pre", "alpha_post", "alpha_res", "b_pre", "b_post",
         "b_res")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,T,C,shift", [(5, 1025, 32, 0), (6, 1056, 80, 0), (6, 1057, 48, 1), (7, 1087, 32, 0),
                                         (7, 1089, 96, 0), (8, 1151, 20, 0), (8, 1153, 36, 0), (8, 2081, 8, 0), (3, 1, 32, 0),
                                         (3, 65, 160, 0), (3, 700, 128, 0), (3, 33, 128, 1), (3, 4100, 64, 0)])
def test_gradients(device, n, T, C, shift, dtype):
    g = torch.Generator().manual_seed(n * T + C)
    layer = mhc.MHCLayer(C, n)
    with torch.no_grad():
        for nm in NAMES:
            p = getattr(layer, nm)
            if nm.startswith("b_"):
                p.copy_(0.3 * torch.randn(p.shape, generator=g))
            elif nm.startswith("alpha"):
                p.fill_(0.3)
            elif nm.startswith("phi"):
                p.copy_(0.5 / (n * C) ** 0.5 * torch.randn(p.shape, generator=g))
            else:
                p.copy_((1 + 0.1 * torch.randn(p.shape, generator=g)).to(p.dtype))
    x = torch.randn(T, n, C, generator=g).to(dtype)
    cot = torch.randn(T, n, C, generator=g)
    ps = [getattr(layer, nm).detach().double().requires_grad_(True) for nm in NAMES]
    rx = x.double().requires_grad_(True)
    ref = R.mhc_layer_dynamic(rx, *ps, 20, 1e-8, 1e-5, dtype=torch.float64)
    want = torch.autograd.grad(ref, [rx] + ps, cot.double())
    layer = layer.to(device)
    buf = torch.empty(x.numel() + 8, dtype=dtype, device=device)
    xd = buf[shift:shift + x.numel()].view(x.shape)
    xd.copy_(x)
    xd.requires_grad_(True)
    got = torch.autograd.grad(layer(xd), [xd] + [getattr(layer, nm) for nm in NAMES], cot.to(device))
    tag = f"n={n} T={T} C={C} {dtype}"
    rtol, frac = (2.0 ** -8, 1e-3) if dtype == torch.bfloat16 else (1e-3, 1e-5)
    assert_close(got[0], want[0], rtol, grad_atol(want[0], frac), f"{tag} dx")
    for nm, a, e in zip(NAMES, got[1:], want[1:]):
        b = nm == "rmsnorm_weight"
        assert_close(a, e, 2.0 ** -8 if b else 1e-3, grad_atol(e, 1e-3 if b else 1e-4), f"{tag} d{nm}")


@pytest.mark.parametrize("n,T,C", [(3, 300, 256), (3, 40, 1408), (5, 1100, 64)])
def test_dx_is_rounded_once(device, n, T, C):
    """bf16 dx from fp32 sums: the elements that are not the nearest bf16 of the
    float64 gradient are those within fp32's error of a midpoint (some 1e-6 of a
    bf16 step of 2^-8, one in a thousand); a stream part held in 11 bits on the way
    misses one in twenty."""
    d = R.dynamic_layer_inputs(T, n, C, seed=n + T, x_dtype=torch.bfloat16, alpha=0.2, phi_std=0.03, b_std=0.5)
    names = ["weight", "phi_pre", "phi_post", "phi_res", "alpha_pre", "alpha_post", "alpha_res", "b_pre", "b_post",
             "b_res"]
    x = d["x"].to(device).requires_grad_(True)
    out = mhc.mhc_layer_fused_dynamic_training(x, *[d[k].to(device) for k in names])
    gx, = torch.autograd.grad(out, [x], d["grad"].to(device))
    xr = d["x"].double().requires_grad_(True)
    ref = R.mhc_layer_dynamic(xr, *[d[k].double() for k in names], 20, 1e-8, 1e-5, dtype=torch.float64)
    want, = torch.autograd.grad(ref, [xr], d["grad"].double())
    missed = float((gx.cpu() != want.to(torch.bfloat16)).double().mean())
    assert missed < 0.01, (n, T, C, missed)
