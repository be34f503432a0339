"""Power-of-two belts with 2 Nside < mmax < 4 Nside (one conjugate alias per
bin) in the register-FFT kernel and its adjoint: mmax one past the last alias-
free value, at the last value before a wrap, and between; map counts with and
without paired jobs; rings of both phases and with phases off.

Against the oracle (1e-12 of the rms, the bound of the other parity tests) and,
for the adjoint, <Y a, g> = <a, Y^T g> to 1e-12 of the product of the norms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,M,K", [
    (8, 31, 31, 1), (8, 40, 17, 3), (16, 47, 47, 2), (16, 63, 33, 8), (32, 64, 64, 1),
    (64, 191, 191, 4), (64, 255, 255, 5), (256, 600, 513, 1), (256, 767, 767, 2),
    (8, 32, 32, 1)])
def test_belt_alias(oracle, N, L, M, K):
    import torch
    import wavemoth_amd as wm
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    alm = wm.power_law_alm(L, M, K, 31 + N + M)
    op = oracle.OraclePlan(N, L, M, K)
    for phases in (True, False):
        out = np.full((12 * N * N, K), np.nan)
        plan = wm.ShtPlan(N, L, M, alm, out, "mmajor", phase_shifts=phases)
        plan.execute()
        ref = op.synthesize(alm, phase_shifts=phases)
        assert np.linalg.norm(out - ref) <= 1e-12 * np.linalg.norm(ref)
    info = plan.info()
    assert info["rings_belt"] == (N + 1 if 4 * N > M else 0), info


@pytest.mark.parametrize("N,L,M,K", [(8, 31, 31, 2), (16, 50, 33, 1), (64, 255, 255, 3),
                                     (256, 767, 700, 1), (64, 128, 128, 4)])
def test_belt_alias_adjoint(N, L, M, K):
    import torch
    from wavemoth_amd.torch_sht import DevicePlan, random_alm
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    dev = torch.device("cuda:0")
    p = DevicePlan(N, L, M, K)
    a = random_alm(L, M, K, 5, dev, flat=True)
    g = torch.randn((p.npix, K), device=dev, dtype=torch.float64,
                    generator=torch.Generator(device=dev).manual_seed(6))
    f, b = torch.empty_like(g), torch.empty_like(a)
    p.synthesize_into(a, f)
    p.adjoint_into(g, b)
    lhs = (f * g).sum(0)
    rhs = (torch.view_as_real(a) * torch.view_as_real(b)).sum((0, 2))
    scale = torch.linalg.norm(f, dim=0) * torch.linalg.norm(g, dim=0)
    assert bool(((lhs - rhs).abs() <= 1e-12 * scale).all()), (lhs, rhs)
