"""Sinkhorn-Knopp and its adjoint where a matrix is spread over lanes, a wave
or a workgroup (zero-padded to 4, 8, 16 or 32): the padding at every n, the
adjoint's register history and its segments beyond 32 iterations, and the
per-token coefficients over few and many K splits; against the float64 oracle.

Tolerances: fp32 chains of `iters` normalisations of well-conditioned
matrices: 1e-4 / 1e-5 forward, 1e-3 with 1e-5 max|ref| for the adjoint."""
import pytest
import torch

import mhc_ascend_amd as mhc
from oracle import csk
from oracle import reference as R
from tests.conftest import assert_close, grad_atol
from tests.test_gpu_dynamic import _check_dyn, _oracle_dyn, _run_dyn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 11, 16, 17, 31, 32])
@pytest.mark.parametrize("iters,eps", [(31, 1e-8), (32, 0.0), (33, 1e-8), (65, 1e-8)])
def test_sinkhorn_history_segments(device, n, iters, eps):
    g = torch.Generator().manual_seed(1000 * n + iters)
    a = torch.exp(torch.randn(67, n, n, generator=g))
    go = torch.randn(67, n, n, generator=g)
    ad = a.to(device).requires_grad_(True)
    out = mhc.sinkhorn_knopp(ad, iters, eps)
    out.backward(go.to(device))
    ref = torch.from_numpy(csk.sinkhorn_fwd(a.double().numpy(), iters, eps))
    gref = torch.from_numpy(csk.sinkhorn_bwd(go.double().numpy(), a.double().numpy(), iters, eps))
    assert_close(out, ref, 1e-4, 1e-5, f"SK fwd n={n} T={iters}")
    assert_close(ad.grad, gref, 1e-3, max(grad_atol(gref, 1e-5), 1e-6), f"SK bwd n={n} T={iters}")


@pytest.mark.parametrize("n", [5, 8])
@pytest.mark.parametrize("iters", [12, 20])
def test_sinkhorn_large_batch(device, n, iters):
    """Past the batch where the forward takes one row per lane, on both sides
    of that form's 12-iteration register history."""
    g = torch.Generator().manual_seed(n + iters)
    a = torch.exp(torch.randn(16384 + 5, n, n, generator=g))
    go = torch.randn(a.shape, generator=g)
    ad = a.to(device).requires_grad_(True)
    out = mhc.sinkhorn_knopp(ad, iters, 1e-8)
    out.backward(go.to(device))
    idx = torch.cat([torch.arange(200), torch.arange(16384 - 200, 16384 + 5)])
    ref = torch.from_numpy(csk.sinkhorn_fwd(a[idx].double().numpy(), iters, 1e-8))
    gref = torch.from_numpy(csk.sinkhorn_bwd(go[idx].double().numpy(), a[idx].double().numpy(), iters, 1e-8))
    assert_close(out.cpu()[idx], ref, 1e-4, 1e-5, f"SK fwd n={n} T={iters}")
    assert_close(ad.grad.cpu()[idx], gref, 1e-3, max(grad_atol(gref, 1e-5), 1e-6), f"SK bwd n={n} T={iters}")


# (n, tokens, C, iters): 1 to 1025 tokens cross the limit of the split lane
# groups at n <= 4; C = 4096 gives few tokens 64 K splits; iterations 33 / 70
# run the adjoint in segments
@pytest.mark.parametrize("n,B,C,iters", [(3, 1, 4096, 20), (4, 17, 4096, 33), (4, 1024, 64, 20), (4, 1025, 64, 20),
                                         (3, 1027, 32, 33), (5, 3, 1024, 33), (6, 2, 2048, 20), (7, 1030, 32, 20),
                                         (8, 5, 1280, 70), (9, 6, 96, 20), (12, 5, 64, 32), (15, 3, 32, 20),
                                         (16, 7, 256, 20), (16, 3, 32, 33)])
def test_dynamic_coefficients(device, n, B, C, iters):
    d = R.dynamic_layer_inputs(B, n, C, seed=7 * n + B + iters, x_dtype=torch.float32, alpha=0.1, phi_std=0.02,
                               b_std=0.5)
    _check_dyn(_run_dyn(d, device, iters=iters), _oracle_dyn(d, iters=iters), torch.float32,
               f"n={n} B={B} C={C} T={iters}")


# (n, batch, iters): one past the batch (and, backward, below the iterations) up
# to which a matrix is spread over a wave or workgroup, and on it
@pytest.mark.parametrize("n,B,iters", [(9, 2304, 5), (9, 2305, 5), (9, 2881, 5), (16, 4097, 10), (16, 5121, 5),
                                       (17, 817, 5), (17, 1361, 5), (32, 1537, 9), (32, 2561, 5), (5, 4096, 12),
                                       (8, 4097, 12)])
def test_sinkhorn_batches_around_the_forms(device, n, B, iters):
    g = torch.Generator().manual_seed(n + B + iters)
    a = torch.exp(torch.randn(B, n, n, generator=g))
    go = torch.randn(a.shape, generator=g)
    ad = a.to(device).requires_grad_(True)
    out = mhc.sinkhorn_knopp(ad, iters, 1e-8)
    out.backward(go.to(device))
    idx = torch.cat([torch.arange(40), torch.arange(B - 40, B)])
    ref = torch.from_numpy(csk.sinkhorn_fwd(a[idx].double().numpy(), iters, 1e-8))
    gref = torch.from_numpy(csk.sinkhorn_bwd(go[idx].double().numpy(), a[idx].double().numpy(), iters, 1e-8))
    assert_close(out.cpu()[idx], ref, 1e-4, 1e-5, f"SK fwd n={n} B={B} T={iters}")
    assert_close(ad.grad.cpu()[idx], gref, 1e-3, max(grad_atol(gref, 1e-5), 1e-6), f"SK bwd n={n} B={B} T={iters}")


# one past the tokens up to which the coefficients are spread (4096, half of it
# at n = 16), on both sides of the 12 iterations of the row form's history and of
# n iters = 110
@pytest.mark.parametrize("n,B,iters", [(5, 4097, 12), (6, 4097, 10), (7, 4100, 12), (8, 4097, 12), (8, 4097, 13),
                                       (9, 4097, 12), (9, 4097, 13), (16, 2049, 10), (12, 4097, 20)])
def test_dynamic_coefficients_of_many_tokens(device, n, B, iters):
    d = R.dynamic_layer_inputs(B, n, 32, seed=n + B + iters, x_dtype=torch.float32, alpha=0.1, phi_std=0.02, b_std=0.5)
    _check_dyn(_run_dyn(d, device, iters=iters), _oracle_dyn(d, iters=iters), torch.float32, f"n={n} B={B} T={iters}")
