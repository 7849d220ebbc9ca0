"""Every lane of a row or column scales by the same bits of its sum.

A butterfly's first add that is contracted with the product behind it, or
rotations that leave the lanes of a column with other pairs, give the lanes
sums that differ by a rounding, and the matrix keeps the difference.
Emulated here in fp32 with the sums alike and with a fused first add of the
column: the library's error against float64 is the first one's."""
import pytest
import torch

from mhc_ascend_amd import ops


def _tree(v):
    v = list(v)
    while len(v) > 1:
        v = [v[i] + v[i + 1] if i + 1 < len(v) else v[i] for i in range(0, len(v), 2)]
    return v[0]


def _emulated(x, iters, eps, fused):
    n = x.shape[-1]
    a = x.clone()
    for _ in range(iters):
        rinv = (1 / (_tree(a.unbind(2)) + eps).double()).float()[:, :, None]
        b = a * rinv
        if fused:
            # row r: fma(a_r, rinv_r, b_{r ^ 1}) and the other pairs' sums as they are in its lanes
            part = [(a[:, r].double() * rinv[:, r].double() + (b[:, r ^ 1].double() if (r ^ 1) < n else 0)).float()
                    for r in range(n)]
            col = torch.stack([_tree([part[r if p == r // 2 else 2 * p + (r & 1 if 2 * p + 1 < n else 0)]
                                      for p in range((n + 1) // 2)]) for r in range(n)], 1)
        else:
            col = _tree(b.unbind(1))[:, None]
        a = b * (1 / (col + eps).double()).float()
    return a


@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 12, 16])
def test_sums_alike_model(n):
    """The two emulations are far enough apart to tell (CPU)."""
    same, fused, _ = _errors(n)
    assert fused > 1.05 * same


def _errors(n, iters=20, eps=1e-8):
    g = torch.Generator().manual_seed(n)
    # batches that run with a column's elements in several lanes and tree sums
    x = torch.exp(0.45 * torch.randn(4000 if n <= 8 else 2000, n, n, generator=g))
    e = x.double()
    for _ in range(iters):
        e = e / (e.sum(2, keepdim=True) + eps)
        e = e / (e.sum(1, keepdim=True) + eps)
    err = lambda m: float((m.double() - e).norm() / e.norm())
    return err(_emulated(x, iters, eps, False)), err(_emulated(x, iters, eps, True)), (x, err)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 12, 16])
def test_sums_alike(device, n):
    same, fused, (x, err) = _errors(n)
    got = err(ops.sinkhorn_knopp(x.to(device), 20, 1e-8).cpu())
    assert got <= 0.5 * (same + fused), (got, same, fused)
