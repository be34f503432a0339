"""The adjoint's partial sums past 2^32 doubles per m: lmax 32767 with 70000 maps
at Nside 1, mmax 0 (2 maps lmax = 4.6e9), some maps against plans of one map.
The same sums in another grouping of maps: 1e-12 of the rms as elsewhere.  The
plan, its partial sums and the result take 37 GB each."""
import pytest

pytestmark = pytest.mark.gpu


def test_rows_past_32_bits():
    import torch
    from wavemoth_amd.torch_sht import DevicePlan
    dev = torch.device("cuda:0")
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info(dev)[0] < 130e9:
        pytest.skip("needs 130 GB of free device memory")
    N, L, K = 1, 32767, 70000
    gen = torch.Generator(device=dev)
    gen.manual_seed(5)
    g = torch.randn((12, K), generator=gen, device=dev, dtype=torch.float64)
    print("case N=%d L=%d K=%d" % (N, L, K), flush=True)
    p = DevicePlan(N, L, 0, K)
    b = torch.empty((L + 1, K), device=dev, dtype=torch.complex128)
    p.adjoint_into(g, b)
    one = DevicePlan(N, L, 0, 1)
    ref = torch.empty((L + 1, 1), device=dev, dtype=torch.complex128)
    for k in (0, 1, 3, 34567, K - 1):
        one.adjoint_into(g[:, k:k + 1].contiguous(), ref)
        err = float(torch.linalg.norm(b[:, k] - ref[:, 0]) / torch.linalg.norm(ref))
        print("map %d: %.2e" % (k, err), flush=True)
        assert err <= 1e-12
    del p, b
    torch.cuda.empty_cache()
