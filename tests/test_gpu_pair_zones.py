"""The pair-form sweep (one value per two l) where the plan's rule takes it: odd
Nside, mmax far below lmax, l-ranges of one to a few chunks, every map count.

1. Its map against the oracle, 1e-12 of the rms as in the other parity tests.
2. Its even and odd sums against those of the one-step form (a plan of four
   maps, matrix-core sweep; same rings, seeds and a_lm), zone by zone of latitude.
   A rounding of 2^-53 in one step shifts later values by up to 2^-53 / (sin theta)
   in the one-step form and 2^-53 / (sin 2 theta) in steps of 2 theta; L of them
   add up as sqrt(L), and the rounding of x^2 less the zone's centre, the same in
   every step, is below L 2^-53 / 32 of the same response.  Two forms, two
   roundings a step and a factor of two for the rest: 8 sqrt(L) 2^-53 / (sin theta
   cos theta) of the rms, at the worst ring of the zone (L <= 1030 here).
3. The adjoint of 2, 4 and 7 maps in units of 128 rings, which the sweeps of
   other map counts do not share, through <Y a, g> = <a, Y^T g>: each of the two
   transforms is off by at most sqrt(L) 2^-53 / 0.12 of its rms (as in 2.), the
   dot products by less; 16 sqrt(L) 2^-53 / 0.12 of the norms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ZONES = np.sqrt([0.125 ** 2, 0.125, 0.28125, 0.5, 0.75, 0.99 ** 2])  # of z


def _z(N):
    i = 2 * N - np.arange(2 * N)
    return np.where(i <= N, 1 - i * i / (3.0 * N * N), 4 / 3.0 - 2 * i / (3.0 * N))


def _assert_pair_form(N, L, M, K):
    """The sweep takes K maps a pass on the vector units, with whole units of
    128 rings in 1/8 <= z <= 0.99."""
    from wavemoth_amd import BatchPlan
    info = BatchPlan([(N, L, M, K)]).request_info(0)
    assert info["maps_per_pass"] == K and info["rings_per_lane"] == 2
    z = _z(N)
    units = [u for u in range(2 * N // 128)
             if z[128 * u] >= 0.125 and z[128 * u + 127] <= 0.99]
    assert units and (K < 3 or (M + 1) * -(-2 * N // 128) >= 16384)


def _flat_alm(L, M, K, seed):
    import wavemoth_amd as wm
    a = np.random.default_rng(seed).standard_normal((wm.nalm(L, M), K, 2))
    a[: L + 1, :, 1] = 0.0
    return a.view(np.complex128)[..., 0].copy()


def _work(N, L, M, alm):
    import wavemoth_amd as wm
    out = np.zeros((12 * N * N, alm.shape[1]))
    p = wm.ShtPlan(N, L, M, alm, out, "mmajor")
    p.perform_legendre_transform()
    return p.get_work()


@pytest.mark.parametrize("N,L,M,K", [
    (257, 511, 511, 1), (300, 230, 210, 2), (512, 777, 127, 1), (512, 130, 128, 2)])
def test_map(oracle, N, L, M, K):
    import wavemoth_amd as wm
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    _assert_pair_form(N, L, M, K)
    alm = wm.power_law_alm(L, M, K, N + K)
    got = np.full((12 * N * N, K), np.nan)
    wm.ShtPlan(N, L, M, alm, got, "mmajor").execute()
    ref = oracle.OraclePlan(N, L, M, K).synthesize(alm)
    rms = np.linalg.norm(got - ref, axis=0) / np.linalg.norm(ref, axis=0)
    assert rms.max() <= 1e-12, rms


@pytest.mark.parametrize("N,L,M,K", [
    (257, 511, 511, 1), (300, 230, 210, 2), (512, 777, 127, 1), (512, 130, 128, 2),
    (512, 1030, 1030, 1), (1025, 1030, 1023, 3)])
def test_sums_by_zone(N, L, M, K):
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    _assert_pair_form(N, L, M, K)
    alm = _flat_alm(L, M, K, N + K)
    got = _work(N, L, M, alm)
    ref = _work(N, L, M, np.concatenate([alm] * 4, axis=1)[:, :4].copy())[..., :K]
    z = _z(N)
    for lo, hi in zip(ZONES[:-1], ZONES[1:]):
        r = np.flatnonzero((z >= lo) & (z < hi))
        sc = (z[r] * np.sqrt(1 - z[r] ** 2)).min()
        err = np.linalg.norm(got[:, :, r] - ref[:, :, r]) / np.linalg.norm(ref[:, :, r])
        bound = 8 * np.sqrt(L) * 2.0 ** -53 / sc
        print("z %.3f .. %.3f: error %.2e, bound %.2e" % (lo, hi, err, bound), flush=True)
        assert err <= bound


@pytest.mark.parametrize("N,L,M,K", [(512, 520, 511, 2), (512, 600, 515, 4), (513, 530, 520, 7)])
def test_adjoint(N, L, M, K):
    import torch
    from wavemoth_amd.torch_sht import DevicePlan
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    assert (M + 1) * -(-2 * N // 128) >= 4096
    dev = torch.device("cuda:0")
    p = DevicePlan(N, L, M, K)
    assert p.info()["adjoint_groups"] > 1  # one group would take one-step units only
    gen = torch.Generator(device=dev)
    gen.manual_seed(N + K)
    g = torch.randn((p.npix, K), generator=gen, device=dev, dtype=torch.float64)
    b = torch.full((p.nalm, K), complex(float("nan"), 0.0), device=dev, dtype=torch.complex128)
    p.adjoint_into(g, b)
    ls = np.concatenate([np.arange(m, L + 1) for m in range(M + 1)])
    ms = np.concatenate([np.full(L + 1 - m, m) for m in range(M + 1)])
    picks = [ls >= 0] + [ms == m for m in (0, 1, M // 2, M)]
    picks += [ls == l for l in (0, 1, L // 2, L - 1, L)]
    f = torch.empty_like(g)
    for pick in picks:
        a = torch.randn((p.nalm, K, 2), generator=gen, device=dev, dtype=torch.float64)
        a *= torch.from_numpy(pick.astype(float)).to(dev)[:, None, None]
        a[: L + 1, :, 1] = 0.0
        p.synthesize_into(torch.view_as_complex(a), f)
        lhs = (f * g).sum(0)
        rhs = (a * torch.view_as_real(b)).sum((0, 2))
        scale = torch.linalg.norm(f, dim=0) * torch.linalg.norm(g, dim=0)
        assert bool(((lhs - rhs).abs() <= 16 * L ** 0.5 * 2.0 ** -53 / 0.12 * scale).all()), \
            (lhs, rhs, scale)
