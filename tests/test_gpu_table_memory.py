"""Device memory of the sweep's tables: plans and batches hold the recurrence
checkpoints (48 bytes per m and ring) only for a matrix-core sweep or the
adjoint, so a plan of one map (vector sweep) without an adjoint, or such a
batch, is smaller by them than one of 4 maps, besides 3 maps' a_lm and q."""
import pytest

pytestmark = pytest.mark.gpu


def _per_map(N, L):
    padded = sum((L - m) // 16 * 16 + 16 for m in range(L + 1))
    return 16 * padded + 16 * 2 * (2 * N) * (L + 1)


def _bytes(kind, N, L, K):
    import wavemoth_amd as wm
    from wavemoth_amd.torch_sht import DevicePlan
    if kind == "batch":
        b = wm.BatchPlan([(N, L, L, K)])
        assert (b.request_info(0)["maps_per_pass"] > 3) == (K == 4)
        return b.info()["device_bytes"]
    p = DevicePlan(N, L, L, K)
    assert p.info()["adjoint_groups"] == 0
    return p.info()["device_bytes"]


@pytest.mark.parametrize("kind,N,L", [("plan", 2304, 300), ("batch", 96, 511), ("batch", 512, 512)])
def test_checkpoints_only_where_read(kind, N, L):
    one, four = _bytes(kind, N, L, 1), _bytes(kind, N, L, 4)
    ckpt = 48 * (L + 1) * 2 * N
    print("case %s N=%d L=%d: %d %d bytes, checkpoints %d" % (kind, N, L, one, four, ckpt),
          flush=True)
    assert four - one - 3 * _per_map(N, L) >= 0.5 * ckpt


def test_mixed_plan_without_adjoint():
    """Neither table in a mixed plan without an adjoint: an FP64 plan of the same
    4 maps holds the checkpoints (133 MB) and 64 bytes of a_lm per padded (l, m);
    the FP32 one the B operand of 32 columns and two tables, 144 bytes (27 MB)."""
    import wavemoth_amd as wm
    from wavemoth_amd.torch_sht import DevicePlan
    N, L, K = 2304, 600, 4
    fp64, mixed = (DevicePlan(N, L, L, K, f).info()["device_bytes"]
                   for f in (0, wm.WAVEMOTH_MIXED_F32))
    ckpt = 48 * (L + 1) * 2 * N
    print("fp64 %d mixed %d checkpoints %d" % (fp64, mixed, ckpt), flush=True)
    assert fp64 - mixed >= 0.5 * ckpt
