"""The projection backward over two or three output tiles at once (n = 5..8, more
than 1024 tokens): token counts at the edges of its 32-token stages and pairs of
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
                                         (7, 1089, 96, 0), (8, 1151, 20, 0), (8, 1153, 36, 0), (8, 2081, 8, 0)])
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
