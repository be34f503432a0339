"""The Legendre sweep's shapes at the edges of their ranges, against the
oracle: map counts at every pass size of the matrix-core sweep (4 .. 16 maps,
one to three passes, map counts that leave columns or a whole pass partly
empty), l-ranges of fewer chunks than segments, ring counts that fill no
16-, 64- or 128-ring group, both sides of the wave-count rule, seeds made
per execute, and a batch whose requests take different shapes.

Both sides sum at most lmax + 1 terms per coefficient in FP64; their
difference is a few sqrt(lmax) 2^-53 of the rms: 1e-12 is the bound the other
parity tests use for the same comparison."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gpu(N, L, M, K, alm, flags=0):
    import wavemoth_amd as wm
    out = np.full((12 * N * N, K), np.nan)
    wm.ShtPlan(N, L, M, alm, out, "mmajor", flags=flags).execute()
    return out


@pytest.mark.parametrize("N,L,M,K", [
    (5, 9, 9, 4), (8, 15, 15, 5), (8, 16, 16, 6), (9, 300, 20, 7), (20, 61, 61, 8),
    (33, 66, 50, 9), (12, 30, 30, 11), (16, 47, 47, 12), (17, 40, 40, 14), (24, 63, 63, 16),
    (32, 64, 64, 17), (7, 129, 64, 33), (64, 191, 191, 1), (64, 128, 128, 2), (70, 140, 140, 3),
    (256, 200, 200, 4), (129, 257, 257, 6)])
def test_sweep_shapes(oracle, N, L, M, K):
    import wavemoth_amd as wm
    print("case N=%d L=%d M=%d K=%d" % (N, L, M, K), flush=True)
    alm = wm.power_law_alm(L, M, K, 900 + N + K)
    ref = oracle.OraclePlan(N, L, M, K).synthesize(alm)
    got = _gpu(N, L, M, K, alm)
    rms = np.linalg.norm(got - ref, axis=0) / np.linalg.norm(ref, axis=0)
    assert rms.max() <= 1e-12, rms


@pytest.mark.parametrize("K,M", [(3, 1534), (3, 1536), (2, 254), (2, 256)])
def test_wave_count_rule(K, M):
    """One map repeated: the vector sweep (a plan of one map at mmax 4096 / few
    maps past the rule's line) and the matrix sweep give the same map."""
    import wavemoth_amd as wm
    N = 256
    print("case K=%d M=%d" % (K, M), flush=True)
    one = wm.power_law_alm(M, M, 1, 77)
    got = _gpu(N, M, M, K, np.repeat(one, K, axis=1))
    many = _gpu(N, M, M, 8, np.repeat(one, 8, axis=1))
    for k in range(K):
        assert np.linalg.norm(got[:, k] - many[:, 0]) <= 1e-12 * np.linalg.norm(many[:, 0])


def test_seeds_per_execute_match():
    import wavemoth_amd as wm
    N, L, K = 48, 143, 6
    alm = wm.power_law_alm(L, L, K, 5)
    a = _gpu(N, L, L, K, alm)
    b = _gpu(N, L, L, K, alm, flags=wm.WAVEMOTH_SEEDS_ON_THE_FLY)
    assert np.array_equal(a, b)


def test_batch_of_all_shapes():
    import wavemoth_amd as wm
    reqs = [(16, 33, 33, K) for K in (1, 2, 3, 4, 6, 7, 10, 11, 13, 16, 20)]
    alms = [wm.power_law_alm(L, M, K, 60 + K) for _, L, M, K in reqs]
    outs = [np.full((12 * N * N, K), np.nan) for N, _, _, K in reqs]
    wm.BatchPlan(reqs).execute(alms, outs)
    for (N, L, M, K), alm, out in zip(reqs, alms, outs):
        assert np.array_equal(out, _gpu(N, L, M, K, alm)), K
