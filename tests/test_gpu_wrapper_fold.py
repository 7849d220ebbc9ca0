"""The wrapper's forward projection folded onto residual and branch
(csrc/wrapper_proj.hip) and the outputs and gradients that rest on it: every
count of residual streams and row tiles, both modes and storage types, token
counts at the edges of the token tiles and of their three sizes, ragged channel
steps, and rows at an unaligned address; against the float64 oracle.

Tolerances as tests/test_gpu_wrapper.py: fp32 outputs 1e-4 / 1e-5, gradients
1e-3 with 1e-4 max|ref| (one bf16 rounding, 2^-8, where stored in bf16)."""
import pytest
import torch

import mhc_ascend_amd as mhc
from oracle import reference as R
from tests.conftest import assert_close, grad_atol

pytestmark = pytest.mark.gpu

NAMES = ("rmsnorm_weight", "phi_pre", "phi_post", "phi_res", "alpha_pre", "alpha_post", "alpha_res", "b_pre", "b_post",
         "b_res")


def _run(device, n, T, C, dtype, mode, seed, shift=0):
    g = torch.Generator().manual_seed(seed)
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
    r, b = torch.randn(T, C, generator=g).to(dtype), torch.randn(T, C, generator=g).to(dtype)
    cot = torch.randn(T, C, generator=g)
    params = [getattr(layer, nm).detach().clone() for nm in NAMES]
    wrap = mhc.MHCResidualWrapper(C, n, residual_mode=mode)
    wrap.mhc = layer
    wrap.to(device)

    def place(t):
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=device)
        v = buf[shift:shift + t.numel()].view(t.shape)
        v.copy_(t)
        return v.requires_grad_(True)

    rd, bd = place(r), place(b)
    out = wrap(rd, bd)
    got = torch.autograd.grad(out, [rd, bd] + [getattr(layer, nm) for nm in NAMES], cot.to(device))

    rr, rb = r.double().requires_grad_(True), b.double().requires_grad_(True)
    ps = [p.double().requires_grad_(True) for p in params]
    ref = R.mhc_residual_wrapper(
        rr, rb, lambda X: R.mhc_layer_dynamic(X, *ps, 20, 1e-8, 1e-5, dtype=torch.float64), n, mode,
        storage_dtype=dtype if dtype == torch.bfloat16 else None)
    want = torch.autograd.grad(ref, [rr, rb] + ps, cot.double())
    tag = f"n={n} T={T} C={C} {dtype} {mode}"
    assert_close(out, ref, 1e-4, 1e-5, f"{tag} out")
    fam = {}
    for nm, e in zip(NAMES, want[2:]):
        k = nm.split("_")[0]
        fam[k] = max(fam.get(k, 0.0), float(e.abs().max()))
    for nm, a, e in zip(("dr", "db"), got[:2], want[:2]):
        rtol, frac = (2.0 ** -8, 1e-3) if dtype == torch.bfloat16 else (1e-3, 1e-5)
        assert_close(a, e, rtol, grad_atol(e, frac), f"{tag} {nm}")
    for nm, a, e in zip(NAMES, got[2:], want[2:]):
        # the H_res gradients vanish: floor against their family's largest
        rtol = 2.0 ** -8 if nm == "rmsnorm_weight" else 1e-3
        floor = max(grad_atol(e, 1e-3 if nm == "rmsnorm_weight" else 1e-4), 1e-5 * fam[nm.split("_")[0]])
        assert_close(a, e, rtol, floor, f"{tag} d{nm}")


@pytest.mark.parametrize("mode", ["decay", "zero"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,C", [(2, 16), (3, 96), (4, 264), (5, 64), (6, 80), (7, 96), (8, 72), (9, 32), (12, 64),
                                 (16, 40), (32, 24)])
def test_every_stream_count(device, n, C, dtype, mode):
    _run(device, n, 37, C, dtype, mode, seed=n + C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,T,C", [(8, 1, 64), (8, 64, 128), (5, 65, 64), (8, 511, 64), (5, 512, 192), (6, 641, 48),
                                   (8, 2047, 64), (8, 2048, 72), (5, 2305, 64), (7, 130, 1056), (3, 20, 2080)])
def test_token_tiles_and_splits(device, n, T, C, dtype):
    _run(device, n, T, C, dtype, "decay", seed=T + C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [5, 8])
def test_unaligned_rows(device, n, dtype):
    _run(device, n, 70, 64, dtype, "decay", seed=n, shift=1)


def _projection_error(device, n, T, C, dtype, mode):
    """|P - float64| / |float64| of the folded P, from the forward's saved state."""
    g = torch.Generator().manual_seed(5)
    r, b = torch.randn(T, C, generator=g).to(dtype), torch.randn(T, C, generator=g).to(dtype)
    layer = mhc.MHCLayer(C, n).to(device)
    with torch.no_grad():  # h_pre = sigmoid(P / r_h): a small weight keeps it linear
        for nm in ("alpha_pre", "alpha_post", "alpha_res"):
            getattr(layer, nm).fill_(1.0)
    from mhc_ascend_amd import native
    ps = [getattr(layer, nm).detach() for nm in NAMES]
    _, saved = native.wrapper_dynamic_fwd(r.to(device), b.to(device), mode, n, *ps)
    np_ = 2 * n + n * n
    off = (C + 63) // 64 * 64 + (T * np_ + 63) // 64 * 64
    P = saved.view(-1)[off:off + T * np_].view(T, np_).double().cpu()
    X = R.build_wrapper_streams(r, b, n, mode).double().reshape(T, -1)
    phi = torch.cat([layer.phi_pre, layer.phi_post, layer.phi_res]).detach().double().cpu()
    ref = X @ phi.t()
    return float((P - ref).norm() / ref.norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_projection_error(device, dtype):
    """The folded P against float64, relative to its norm: 1e-6 (hi / mid / lo
    planes of Phi, residual streams below 2^-24), at n = 8 over a long row."""
    assert _projection_error(device, 8, 96, 4096, dtype, "decay") < 1e-6


@pytest.mark.parametrize("mode", ["decay", "zero"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,T,C", [(3, 700, 512), (5, 700, 512), (8, 300, 64), (12, 300, 64)])
def test_projection_error_of_short_rows(device, n, T, C, dtype, mode):
    """Rows of few steps: three half-ulps of fp32 (3 x 2^-24), which a step's
    products below hi . hi in the large sum's accumulator, or stream 2 of bf16
    'decay' from single bf16 parts, exceed."""
    assert _projection_error(device, n, T, C, dtype, mode) < 3 * 2.0 ** -24
