"""What WAVEMOTH_SEEDS_ON_THE_FLY adds to an execute, as launches of a captured
execute: the seeds and the wave bounds, and recurrence checkpoints only where
the sweep of that plan starts from them (the FP64 matrix-core sweep, the
register-Lambda FP16 contraction)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _launches(plan, alm, out):
    import torch
    from wavemoth_amd import _native
    hip = ctypes.CDLL(_native.LIB_PATH)  # symbols of the runtime it is linked to
    s = torch.cuda.Stream()
    stream, graph, n = ctypes.c_void_p(s.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t()
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
    plan(alm, out, s.cuda_stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return n.value


@pytest.mark.parametrize("N,L,K,mixed,extra", [
    (256, 256, 1, 0, 2), (256, 511, 2, 0, 2), (64, 128, 1, 0, 3), (48, 96, 6, 0, 3),
    (64, 128, 16, 0x1000, 2), (64, 128, 16, 0x8000, 3)])
def test_launches_of_seeds_per_execute(N, L, K, mixed, extra):
    import torch
    import wavemoth_amd as wm
    from wavemoth_amd.torch_sht import DevicePlan, random_alm
    print("case N=%d L=%d K=%d mixed=%#x" % (N, L, K, mixed), flush=True)
    dev = torch.device("cuda:0")
    alm = random_alm(L, L, K, 3, dev)
    out = torch.empty((12 * N * N, K), dtype=torch.float64, device=dev)
    plans = [DevicePlan(N, L, L, K, mixed | f) for f in (0, wm.WAVEMOTH_SEEDS_ON_THE_FLY)]
    counts = [_launches(p.synthesize_into, alm, out) for p in plans]
    assert counts[1] - counts[0] == extra, counts


def test_launches_of_seeds_per_execute_with_a_resource(tmp_path):
    import numpy as np
    import torch
    import wavemoth_amd as wm
    from wavemoth_amd import _native
    from wavemoth_amd.resource import write_resource
    N, L, K = 16, 32, 5
    fn = str(tmp_path / "r.dat")
    write_resource(fn, N, L, L)
    host = np.zeros((wm.nalm(L, L), K), np.complex128), np.zeros((12 * N * N, K))
    dev = torch.device("cuda:0")
    alm, out = (torch.from_numpy(x).to(dev) for x in host)
    counts = []
    for f in (0, wm.WAVEMOTH_SEEDS_ON_THE_FLY):
        p = wm.ShtPlan(N, L, L, host[0], host[1], "mmajor", matrix_data_filename=fn,
                       flags=_native.WAVEMOTH_RESOURCE_APPLY | f)
        counts.append(_launches(
            lambda a, o, s, p=p: p.execute_device(a.data_ptr(), o.data_ptr(), s), alm, out))
    assert counts[1] - counts[0] == 2, counts
