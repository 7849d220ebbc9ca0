"""The backward row pass with two chunks per lane at n = 5..8 (csrc/layer.hip,
bwd_tiling): widths just past one chunk on 256 lanes, a token count on each side of
the rule's four per CU and one that leaves the last round of tokens ragged, static
H and both storage types; against the float64 oracle (gradients 1e-3 with 1e-4
max|ref|, one bf16 rounding, 2^-8, where stored in bf16)."""
import pytest
import torch

import mhc_ascend_amd as mhc
from oracle import reference as R
from tests.conftest import assert_close, grad_atol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,T,C", [(5, 1024, 1028), (6, 1023, 1040), (7, 1031, 1284), (8, 1300, 1028), (8, 1024, 1532)])
def test_gradients(device, n, T, C, dtype):
    g = torch.Generator().manual_seed(n * T + C)
    layer = mhc.MHCLayer(C, n, use_dynamic_h=False)
    names = ("H_pre", "H_post", "H_res")
    with torch.no_grad():
        for nm in names:
            p = getattr(layer, nm)
            p.copy_(0.3 * torch.randn(p.shape, generator=g))
    x = torch.randn(T, n, C, generator=g).to(dtype)
    cot = torch.randn(T, n, C, generator=g)
    ps = [getattr(layer, nm).detach().double().requires_grad_(True) for nm in ("rmsnorm_weight",) + names]
    rx = x.double().requires_grad_(True)
    want = torch.autograd.grad(R.mhc_layer_static(rx, *ps, 20, 1e-8, 1e-5, dtype=torch.float64), [rx] + ps, cot.double())
    layer = layer.to(device)
    xd = x.to(device).requires_grad_(True)
    params = [getattr(layer, nm) for nm in ("rmsnorm_weight",) + names]
    got = torch.autograd.grad(layer(xd), [xd] + params, cot.to(device))
    for i, (a, e) in enumerate(zip(got, want)):
        b = dtype == torch.bfloat16 if i == 0 else i == 1
        assert_close(a, e, 2.0 ** -8 if b else 1e-3, grad_atol(e, 1e-3 if b else 1e-4), f"n={n} T={T} C={C} {dtype} [{i}]")
