"""The host-array calls at sizes on both sides of the split of large copies
(2 MiB) and at sizes that leave an uneven last part: bit for bit what the
device call gives on the same a_lm (the same kernels run on copies), forward
and adjoint, repeated, after the arrays changed, and from two threads with a
plan each."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _device_map(N, L, K, alm):
    import torch
    from wavemoth_amd.torch_sht import DevicePlan
    out = torch.empty((12 * N * N, K), dtype=torch.float64, device="cuda:0")
    DevicePlan(N, L, L, K).synthesize_into(torch.from_numpy(alm).to("cuda:0"), out)
    return out.cpu().numpy()


@pytest.mark.parametrize("N,L,K", [(104, 60, 2), (105, 60, 2), (128, 255, 3), (256, 600, 2),
                                   (333, 700, 1)])
def test_execute_equals_device(N, L, K):
    import wavemoth_amd as wm
    print("case N=%d L=%d K=%d" % (N, L, K), flush=True)
    alm = wm.power_law_alm(L, L, K, 8)
    out = np.full((12 * N * N, K), np.nan)
    plan = wm.ShtPlan(N, L, L, alm, out, "mmajor")
    for rep in range(2):
        alm *= 1.0 + rep
        out[:] = np.nan
        plan.execute()
        assert np.array_equal(out, _device_map(N, L, K, alm))


def test_adjoint_equals_device():
    import torch
    import wavemoth_amd as wm
    from wavemoth_amd.torch_sht import DevicePlan
    N, L, K = 200, 450, 2
    g = np.random.default_rng(4).standard_normal((12 * N * N, K))
    alm = np.zeros((wm.nalm(L, L), K), complex)
    wm.ShtPlan(N, L, L, alm, g.copy(), "mmajor").execute_adjoint()
    ref = torch.empty(alm.shape, dtype=torch.complex128, device="cuda:0")
    DevicePlan(N, L, L, K).adjoint_into(torch.from_numpy(g).to("cuda:0"), ref)
    assert np.array_equal(alm, ref.cpu().numpy())


def test_two_threads():
    import wavemoth_amd as wm
    N, L = 256, 511
    alms = [wm.power_law_alm(L, L, 1, s) for s in (1, 2)]
    outs = [np.full((12 * N * N, 1), np.nan) for _ in alms]
    plans = [wm.ShtPlan(N, L, L, a, o, "mmajor") for a, o in zip(alms, outs)]
    workers = [threading.Thread(target=p.execute, kwargs={"repeat": 5}) for p in plans]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    for a, o in zip(alms, outs):
        assert np.array_equal(o, _device_map(N, L, 1, a))
