"""WAVEMOTH_MEASURE batches at sizes whose sweep has the pair form of the
recurrence, and on both sides of its rule for three maps: a measured sweep
shape gives the single plan's map bit for bit.  In these geometries no ring
wraps or the wrapping rings' kernel is the single plan's, which the test
checks before it compares."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,M,K", [
    (256, 512, 512, 1), (257, 600, 600, 2), (512, 1024, 1024, 1), (512, 1024, 1024, 2),
    (512, 1024, 1024, 3), (512, 1024, 700, 3), (1024, 2048, 2048, 1), (1024, 2048, 2048, 3)])
def test_measured_shape_keeps_the_map(N, L, M, K):
    import torch
    from wavemoth_amd import WAVEMOTH_MEASURE, BatchPlan
    from wavemoth_amd.torch_sht import DevicePlan, random_alm
    dev = torch.device("cuda:0")
    b = BatchPlan([(N, L, M, K)], WAVEMOTH_MEASURE)
    info = b.request_info(0)
    print("case N=%d L=%d M=%d K=%d: RL %d KB %d" % (N, L, M, K, info["rings_per_lane"],
                                                     info["maps_per_pass"]), flush=True)
    assert info["measured"] == 1
    alm = random_alm(L, M, K, 11, dev)
    got = torch.full((12 * N * N, K), float("nan"), dtype=torch.float64, device=dev)
    want = torch.empty_like(got)
    b.synthesize_into([alm], [got])
    DevicePlan(N, L, M, K).synthesize_into(alm, want)
    torch.cuda.synchronize()
    if info["wrap_register"]:
        pytest.skip("the tuner took the other kernel for the wrapping rings")
    assert torch.equal(got, want)
