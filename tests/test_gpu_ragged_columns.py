"""Column sums of rows that are not a multiple of four columns, over row counts at
the edges of the partial sum's four-wave, eight-load steps, and the conversions
around an upcast backward at element counts that are not whole pieces: a bf16
layer of odd width against the float64 oracle (the weight gradient is the column
sum; tolerances of one bf16 rounding, 2^-8, and 1e-3 of its largest entry)."""
import pytest
import torch

import mhc_ascend_amd as mhc
from oracle import reference as R
from tests.conftest import assert_close, grad_atol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 33, 513, 700, 2100])
@pytest.mark.parametrize("C", [7, 65, 129])
def test_weight_gradient(device, T, C):
    g = torch.Generator().manual_seed(T + C)
    layer = mhc.MHCLayer(C, 4, use_dynamic_h=False)
    x = torch.randn(T, 4, C, generator=g).to(torch.bfloat16)
    cot = torch.randn(T, 4, C, generator=g)
    names = ("H_pre", "H_post", "H_res")
    w = layer.rmsnorm_weight.detach().double().requires_grad_(True)
    ps = [getattr(layer, k).detach().double() for k in names]
    R.mhc_layer_static(x.double(), w, *ps, 20, 1e-8, 1e-5, dtype=torch.float64).backward(cot.double())
    layer = layer.to(device)
    layer(x.to(device)).backward(cot.to(device))
    assert_close(layer.rmsnorm_weight.grad, w.grad, 2.0 ** -8, grad_atol(w.grad, 1e-3), f"dw T={T} C={C}")
