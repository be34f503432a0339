"""Host-array calls of many plans at once: the helper streams of the large
copies are shared by all plans of a device and destroyed with the last of them,
so plans come and go in several threads while others are copying (every map of
a thread bit for bit the first plan's), and again after all have gone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _map(N, L, K, alm):
    import wavemoth_amd as wm
    out = np.full((12 * N * N, K), np.nan)
    wm.ShtPlan(N, L, L, alm, out, "mmajor").execute()
    return out


def test_plans_come_and_go_while_others_copy():
    import wavemoth_amd as wm
    N, L, K = 150, 210, 1
    alms = [wm.power_law_alm(L, L, K, s) for s in range(4)]
    assert 12 * N * N * K * 8 >= 2 << 20  # copies of this size are cut
    refs = [_map(N, L, K, a) for a in alms]  # each plan the only one
    bad = []

    def work(i):
        for rep in range(6):
            if not np.array_equal(_map(N, L, K, alms[i]), refs[i]):
                bad.append((i, rep))

    for rnd in range(2):
        print("round", rnd, flush=True)
        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not bad, bad


def test_live_plans_share():
    import wavemoth_amd as wm
    N, L = 170, 220
    alm = wm.power_law_alm(L, L, 1, 9)
    outs = [np.full((12 * N * N, 1), np.nan) for _ in range(8)]
    plans = [wm.ShtPlan(N, L, L, alm, o, "mmajor") for o in outs]
    for p in plans:
        p.execute()
    del plans[::2], p
    ref = outs[0].copy()
    assert np.isfinite(ref).all()
    for o in outs:
        assert np.array_equal(o, ref)
        o[:] = np.nan
    for p in plans:
        p.execute()
    assert all(np.array_equal(o, ref) for o in outs[1::2])
