"""The adjoint Legendre stage at the edges of its ranges: map counts of one
and two column groups and of several passes, l-ranges of fewer chunks than
segments, ring counts that fill no 16-, 64- or 128-ring unit, both unit
sizes, and units that share a wave (fewer ring groups than units).

Reference: Y^T g from the oracle's Y by the dot-product identity on unit
vectors would be slow; <Y a, g> = <a, Y^T g> is checked instead for several
a per case, each a single coefficient pattern that isolates rows (all l of one
m, one l of all m), so that a row added twice or left out shows.  Both sides
are FP64 sums whose rounding is a few sqrt(npix) 2^-53 of the product of the
norms: 1e-12 of |Y a| |g| bounds it with margin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,M,K", [
    (3, 5, 5, 1), (8, 15, 15, 2), (9, 300, 20, 3), (17, 40, 33, 4), (33, 66, 66, 5),
    (16, 33, 33, 6), (24, 71, 71, 7), (40, 80, 40, 9), (64, 191, 191, 1), (256, 511, 511, 3),
    (300, 650, 800, 2), (512, 1100, 1024, 1)])
def test_adjoint_rows(N, L, M, K):
    import torch
    from wavemoth_amd.torch_sht import DevicePlan
    M = min(M, L)
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    dev = torch.device("cuda:0")
    p = DevicePlan(N, L, M, K)
    gen = torch.Generator(device=dev)
    gen.manual_seed(N + K)
    g = torch.randn((p.npix, K), generator=gen, device=dev, dtype=torch.float64)
    b = torch.full((p.nalm, K), complex(float("nan"), 0.0), device=dev, dtype=torch.complex128)
    p.adjoint_into(g, b)
    ls = np.concatenate([np.arange(m, L + 1) for m in range(M + 1)])
    ms = np.concatenate([np.full(L + 1 - m, m) for m in range(M + 1)])
    picks = [np.ones(len(ls), bool)]
    picks += [ms == m for m in sorted({0, 1, M // 2, M})]
    picks += [ls == l for l in sorted({0, min(17, L), L // 2, L})]
    f = torch.empty_like(g)
    for pick in picks:
        a = torch.randn((p.nalm, K, 2), generator=gen, device=dev, dtype=torch.float64)
        a *= torch.from_numpy(pick.astype(float)).to(dev)[:, None, None]
        a[: L + 1, :, 1] = 0.0
        p.synthesize_into(torch.view_as_complex(a), f)
        lhs = (f * g).sum(0)
        rhs = (a * torch.view_as_real(b)).sum((0, 2))
        scale = torch.linalg.norm(f, dim=0) * torch.linalg.norm(g, dim=0)
        assert bool(((lhs - rhs).abs() <= 1e-12 * scale).all()), (lhs, rhs, scale)
