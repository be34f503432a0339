"""The pair form of the Legendre recurrence (one value per two l) at the edges
of its rule: ring counts with no whole unit in its range, with one, and with
both unit sizes; odd Nside; l-ranges of one chunk and of odd and even length;
mmax below lmax; every map count of a pass.

The synthesis is compared with the oracle, which steps l by l: both sides sum
at most lmax + 1 terms per coefficient in FP64, 1e-12 of the rms as in the other
parity tests.  The adjoint is compared with the synthesis through
<Y a, g> = <a, Y^T g> for several a that each isolate rows; both sides are FP64
sums whose rounding is a few sqrt(npix) 2^-53 of |Y a| |g|: 1e-12 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,M,K", [
    (48, 96, 96, 1), (96, 191, 191, 1), (96, 15, 15, 2), (97, 40, 31, 3), (131, 300, 200, 4),
    (160, 321, 320, 5), (256, 767, 767, 1), (256, 512, 511, 2), (300, 500, 123, 3),
    (512, 1030, 1030, 1), (512, 777, 700, 3)])
def test_pair_form(oracle, N, L, M, K):
    import torch
    import wavemoth_amd as wm
    from wavemoth_amd.torch_sht import DevicePlan
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    dev = torch.device("cuda:0")
    p = DevicePlan(N, L, M, K)
    alm = wm.power_law_alm(L, M, K, 300 + N + K)
    f = torch.empty((p.npix, K), device=dev, dtype=torch.float64)
    p.synthesize_into(torch.from_numpy(alm).to(dev), f)
    ref = oracle.OraclePlan(N, L, M, K).synthesize(alm)
    rms = np.linalg.norm(f.cpu().numpy() - ref, axis=0) / np.linalg.norm(ref, axis=0)
    assert rms.max() <= 1e-12, rms

    gen = torch.Generator(device=dev)
    gen.manual_seed(N + K)
    g = torch.randn((p.npix, K), generator=gen, device=dev, dtype=torch.float64)
    b = torch.full((p.nalm, K), complex(float("nan"), 0.0), device=dev, dtype=torch.complex128)
    p.adjoint_into(g, b)
    ls = np.concatenate([np.arange(m, L + 1) for m in range(M + 1)])
    ms = np.concatenate([np.full(L + 1 - m, m) for m in range(M + 1)])
    picks = [ls >= 0] + [ms == m for m in sorted({0, 1, M // 2, M})]
    picks += [ls == l for l in sorted({0, 1, L // 2, L - 1, L})]
    for pick in picks:
        a = torch.randn((p.nalm, K, 2), generator=gen, device=dev, dtype=torch.float64)
        a *= torch.from_numpy(pick.astype(float)).to(dev)[:, None, None]
        a[: L + 1, :, 1] = 0.0
        p.synthesize_into(torch.view_as_complex(a), f)
        lhs = (f * g).sum(0)
        rhs = (a * torch.view_as_real(b)).sum((0, 2))
        scale = torch.linalg.norm(f, dim=0) * torch.linalg.norm(g, dim=0)
        assert bool(((lhs - rhs).abs() <= 1e-12 * scale).all()), (lhs, rhs, scale)
