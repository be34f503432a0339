"""The work that users of this package have it do, as cases to be timed: a_lm -> HEALPix
synthesis of one map or many, its adjoint, the gradient of a map-domain loss, batches of uneven
requests, and the host-array call.  Sizes are the repository's own (tests, benchmark) or generic
ones: lmax = 2 Nside is the usual band limit, 3 Nside - 1 the other common choice.

A case is a dict of plain values:
  kind   "synth"    DevicePlan.synthesize_into on tensors in GPU memory
         "adjoint"  DevicePlan.adjoint_into
         "grad"     torch_sht.synthesis with autograd: map, weighted residual, gradient
         "batch"    BatchPlan.synthesize_into over `nreq` requests
         "host"     ShtPlan.execute on numpy arrays
  N, L, M, K   Nside, lmax, mmax, number of maps (batch: N is the largest Nside)
  scheme       "fp64", or a mixed-precision contraction: "f16x3", "f32", "bf16x6"
"""
import math
import random

import numpy as np
import torch

import wavemoth_amd as wm
from wavemoth_amd import torch_sht

FLAGS = {"fp64": 0, "f32": wm.WAVEMOTH_MIXED_F32, "f16x3": wm.WAVEMOTH_MIXED_F16X3,
         "bf16x6": wm.WAVEMOTH_MIXED_BF16X6}
DEV = torch.device("cuda:0") if torch.cuda.is_available() else torch.device("cpu")


def _case(kind, N, L, K, M=None, scheme="fp64", **more):
    return dict(kind=kind, N=N, L=L, M=L if M is None else M, K=K, scheme=scheme, **more)


def listed():
    return [
        # one low-resolution map inside a sampler or an interactive session: latency
        dict(_case("synth", 64, 128, 1), name="synth_n64"),
        # intensity and polarisation-like triplet at the band limit 3 Nside - 1
        dict(_case("synth", 256, 767, 3), name="synth_n256_l767_k3"),
        # sizes that are no powers of two, mmax < lmax, a map count that fills no block
        dict(_case("synth", 300, 700, 5, M=500), name="synth_n300_ragged_k5"),
        # the package's metric: one full-resolution FP64 map
        dict(_case("synth", 2048, 4096, 1), name="synth_n2048"),
        # the largest map in use
        dict(_case("synth", 4096, 8192, 1), name="synth_n4096"),
        # an ensemble of simulations in double precision
        dict(_case("synth", 1024, 2048, 64), name="synth_n1024_k64"),
        # the benchmark's default: many maps, mixed-precision contraction
        dict(_case("synth", 2048, 4096, 64, scheme="f16x3"), name="mixed_f16x3_n2048_k64"),
        # a mid-size ensemble with the FP32 contraction
        dict(_case("synth", 512, 1024, 32, scheme="f32"), name="mixed_f32_n512_k32"),
        # differentiable synthesis: forward, weighted least squares, backward
        dict(_case("grad", 512, 1024, 3), name="grad_n512_k3"),
        # analysis of one full-resolution map
        dict(_case("adjoint", 2048, 4096, 1), name="adjoint_n2048"),
        # uneven requests of several users served together
        dict(_case("batch", 2048, 4096, 8, nreq=24, mix=3), name="batch_24"),
        # the drop-in call on numpy arrays: copies to and from the GPU included
        dict(_case("host", 1024, 2048, 1), name="host_n1024"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _nside(rng, lo, hi):
    """Two thirds of the time a power of two, as HEALPix maps mostly are; else any value."""
    N = _log_int(rng, lo, hi)
    if rng.random() < 2.0 / 3.0:
        N = 1 << int(round(math.log2(N)))
    return min(hi, max(lo, N))


def _band(rng, N):
    """(lmax, mmax): 2 Nside, 3 Nside - 1 or anything between Nside and 3 Nside - 1; mmax is
    lmax, or now and then less."""
    L = rng.choice([2 * N, 2 * N, 3 * N - 1, rng.randint(N, 3 * N - 1)])
    M = L if rng.random() < 0.75 else rng.randint(L // 2, L)
    return L, M


def draw(rng):
    kind = rng.choice(["synth"] * 5 + ["mixed", "mixed", "grad", "adjoint", "adjoint", "batch",
                                       "host"])
    if kind == "batch":
        return _case("batch", 2048, 4096, 8, nreq=rng.randint(4, 16), mix=rng.randint(0, 1 << 30))
    # triples (l, m, ring pair) times maps bound the cost: no more than the listed cases'
    cap = {"synth": 2.0e11, "mixed": 1.5e12, "grad": 2.0e10, "adjoint": 7.0e10, "host": 2.0e10}[kind]
    while True:
        if kind == "mixed":
            N, K = _nside(rng, 64, 2048), _log_int(rng, 16, 64)
        elif kind == "synth":
            N, K = _nside(rng, 32, 4096), rng.choice([1, 1, 1, 2, 3, 4, 5, 8, _log_int(rng, 8, 64)])
        else:
            N, K = _nside(rng, 64, 2048), rng.choice([1, 1, 2, 3, 4, 8])
        L, M = _band(rng, N)
        if L * (M + 1.0) * 2 * N * K <= 2 * cap:
            break
    if kind == "mixed":
        return _case("synth", N, L, K, M=M, scheme=rng.choice(["f16x3", "f16x3", "f32", "bf16x6"]))
    return _case(kind, N, L, K, M=M)


# ------------------------------------------------------------------ inputs

def _requests(case):
    """(Nside, lmax, mmax, nmaps) of a batch: Nside over {128 .. 2048}, 1, 3 or 8 maps."""
    r = random.Random(case["mix"])
    sides = [n for n in (128, 256, 512, 1024, 2048) if n <= case["N"]]
    got = []
    for _ in range(case["nreq"]):
        N = r.choice(sides)
        got.append((N, 2 * N, 2 * N, r.choice([1, 3, 8])))
    return got


def _nalm(L, M):
    return (M + 1) * (L + 1) - M * (M + 1) // 2


def _alm(L, M, K, g):
    """m-major a_lm with the power-law spectrum C_l = (l + 1)^-2; a_l0 real."""
    m = torch.arange(M + 1, device=DEV)
    first = m * (2 * L - m + 3) // 2
    l_of = torch.arange(_nalm(L, M), device=DEV) - torch.repeat_interleave(first - m, L + 1 - m)
    a = torch.randn((_nalm(L, M), K, 2), generator=g, device=DEV, dtype=torch.float64)
    a.mul_((math.sqrt(0.5) / (l_of + 1.0)).double()[:, None, None])
    a[: L + 1, :, 0] *= math.sqrt(2.0)
    a[: L + 1, :, 1] = 0.0
    return torch.view_as_complex(a)


def _sky(N, K, g):
    """A map of unit variance."""
    return torch.randn((12 * N * N, K), generator=g, device=DEV, dtype=torch.float64)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _inputs(case, seed):
    kind, N, L, M, K = (case[k] for k in ("kind", "N", "L", "M", "K"))
    g = _generator(seed)
    if kind == "batch":
        return {"alms": [_alm(l, m, k, g) for _, l, m, k in _requests(case)]}
    if kind == "adjoint":
        return {"map": _sky(N, K, g)}
    got = {"alm": _alm(L, M, K, g)}
    if kind == "grad":
        got["data"] = _sky(N, K, g)
        # an equatorial cut (|z| < 0.2) masked out, inverse noise elsewhere
        w = torch.empty((12 * N * N, 1), device=DEV, dtype=torch.float64)
        w.uniform_(0.5, 2.0, generator=g)
        count, z = _rings(N)[:2]
        z = torch.from_numpy(np.repeat(np.concatenate([z, -z[-2::-1]]),
                                       np.concatenate([count, count[-2::-1]]))).to(DEV)
        got["weight"] = torch.where(z.abs() < 0.2, 0.0, w[:, 0])[:, None].contiguous()
    return got


def prepare(case, seed):
    kind, N, L, M, K = (case[k] for k in ("kind", "N", "L", "M", "K"))
    state = dict(_inputs(case, seed), kind=kind)
    if kind == "batch":
        reqs = _requests(case)
        state["plan"] = wm.BatchPlan(reqs)
        state["outs"] = [torch.empty((12 * n * n, k), device=DEV, dtype=torch.float64)
                         for n, _, _, k in reqs]
    elif kind == "host":
        alm = state.pop("alm").cpu().numpy()
        state["plan"] = wm.ShtPlan(N, L, M, alm, np.zeros((12 * N * N, K)), "mmajor")
    elif kind == "grad":
        state["size"] = (N, L, M)
        torch_sht.get_plan(N, L, M, K, DEV)
        state["alm"].requires_grad_(True)
    else:
        state["plan"] = torch_sht.DevicePlan(N, L, M, K, FLAGS[case["scheme"]])
        state["out"] = (torch.empty((_nalm(L, M), K), device=DEV, dtype=torch.complex128)
                        if kind == "adjoint" else
                        torch.empty((12 * N * N, K), device=DEV, dtype=torch.float64))
    return state


def run(state):
    kind = state["kind"]
    if kind == "synth":
        return state["plan"].synthesize_into(state["alm"], state["out"])
    if kind == "adjoint":
        return state["plan"].adjoint_into(state["map"], state["out"])
    if kind == "batch":
        return state["plan"].synthesize_into(state["alms"], state["outs"])
    if kind == "host":
        return state["plan"].execute()
    sky = torch_sht.synthesis(state["alm"], *state["size"])
    res = sky - state["data"]
    loss = 0.5 * (state["weight"] * res * res).sum()
    return {"map": sky.detach(), "grad": torch.autograd.grad(loss, state["alm"])[0]}


# ------------------------------------------------------------- work counts

def _transform_work(N, L, M, K):
    """One synthesis or adjoint.  Bytes: a_lm and map once each.  Flops: per (l, m, ring pair)
    with l sin(theta) >= m (elsewhere Lambda_lm is negligible) 4 for the recurrence and 4 per map,
    and 2.5 n log2 n per ring FFT."""
    count, z = _rings(N)[:2]
    s = np.sqrt((1 - z) * (1 + z))
    m = np.minimum(M, L * s)
    triples = float(np.sum(L * m - m * m / (2 * s)))
    fft = float(np.sum(2 * 2.5 * count * np.log2(count)))
    return 16 * _nalm(L, M) * K + 8 * 12 * N * N * K, triples * (4 + 4 * K) + K * fft


def work(case):
    sizes = (_requests(case) if case["kind"] == "batch"
             else [tuple(case[k] for k in ("N", "L", "M", "K"))])
    got = [_transform_work(*s) for s in sizes]
    b, f = sum(g[0] for g in got), sum(g[1] for g in got)
    if case["kind"] == "grad":  # both directions; data and weights are read too
        b, f = 2 * b + 8 * 12 * case["N"] ** 2 * (case["K"] + 1), 2 * f
    return {"bytes": b, "flops": f}


# ----------------------------------------- the same in 64 bits, without the package

def _rings(N):
    """Northern rings and the equator, from the pole: pixel count, z, phi0 * n / pi (as the
    package defines it, also for odd Nside: both rings of a pair have the southern one's)."""
    i = np.arange(1, 2 * N + 1)
    cap = i < N
    count = np.where(cap, 4 * i, 4 * N)
    z = np.where(cap, 1 - i ** 2 / (3.0 * N * N), 4.0 / 3.0 - 2 * i / (3.0 * N))
    return count, z, np.where(cap, 1, (i - 1) % 2)


def _lambda_blocks(N, L, M, block=32):
    """Yields (l0, lam): normalised associated Legendre functions lam[l - l0, m, ring] for the
    l of one block, from the three-term recurrence with a binary exponent kept apart."""
    theta = torch.from_numpy(np.arccos(_rings(N)[1])).to(DEV)
    x, ls = torch.cos(theta), torch.log2(torch.sin(theta))
    m = torch.arange(M + 1, device=DEV, dtype=torch.float64)
    k = torch.arange(1, M + 1, device=DEV, dtype=torch.float64)
    norm = torch.cat([torch.zeros(1, device=DEV, dtype=torch.float64),
                      torch.cumsum(0.5 * torch.log2((2 * k + 1) / (2 * k)), 0)])
    e0 = norm - 0.5 * math.log2(4 * math.pi)
    log_mm = e0[:, None] + m[:, None] * ls[None, :]
    start_e = torch.floor(log_mm)
    start = torch.exp2(log_mm - start_e) * torch.where(m % 2 == 1, -1.0, 1.0)[:, None]
    prev, cur = torch.zeros_like(start), torch.zeros_like(start)
    expo = start_e
    scale = torch.exp2(expo.clamp(min=-1100.0))
    for l0 in range(0, L + 1, block):
        n = min(block, L + 1 - l0)
        top = min(M, l0 + n - 1) + 1
        lam = torch.zeros((n, top, 2 * N), device=DEV, dtype=torch.float64)
        for j in range(n):
            l = l0 + j
            if l <= M:
                cur[l] = start[l]
                prev[l] = 0
            t = min(M, l) + 1
            torch.mul(cur[:t], scale[:t], out=lam[j, :t])
            mm = m[:t] ** 2
            a = torch.sqrt((4.0 * (l + 1) ** 2 - 1) / ((l + 1.0) ** 2 - mm))[:, None]
            b = torch.sqrt((l * l - mm) / (4.0 * l * l - 1)) if l else torch.zeros_like(mm)
            prev[:t].mul_(-(a * b[:, None])).addcmul_(a * cur[:t], x[None, :])
            prev, cur = cur, prev
            # rows that have not started keep zeros in both
        big = torch.maximum(cur[:top].abs(), prev[:top].abs())
        far = big > 2.0 ** 200
        cur[:top] = torch.where(far, cur[:top] * 2.0 ** -200, cur[:top])
        prev[:top] = torch.where(far, prev[:top] * 2.0 ** -200, prev[:top])
        expo[:top] = torch.where(far, expo[:top] + 200.0, expo[:top])
        scale[:top] = torch.exp2(expo[:top].clamp(min=-1100.0))
        yield l0, lam


def _rows(L, M, l0, n, top):
    """Index of a_lm (l, m) for l in the block, m < top; and where l >= m."""
    l = torch.arange(l0, l0 + n, device=DEV)[:, None]
    m = torch.arange(top, device=DEV)[None, :]
    return (m * (2 * L - m + 3) // 2 + (l - m).clamp(min=0)), l >= m


def _ring_dft(spec, n):
    """sum_b spec[v, b] e^(2 pi i b j / n[v]) for j < n[v] (spec and result zero past n[v]):
    Bluestein's chirp transform over a power of two, all vectors at once."""
    width = spec.shape[1]
    P = 1 << (2 * width - 1).bit_length()
    j = torch.arange(width, device=DEV)[None, :]
    sq = (j * j) % (2 * n[:, None])
    chirp = torch.polar(torch.ones((), device=DEV, dtype=torch.float64),
                        math.pi * sq.double() / n[:, None])
    live = j < n[:, None]
    chirp = torch.where(live, chirp, torch.zeros((), device=DEV, dtype=torch.complex128))
    ker = torch.zeros((spec.shape[0], P), device=DEV, dtype=torch.complex128)
    ker[:, :width] = chirp.conj()
    ker[:, P - width + 1:] = chirp.conj()[:, 1:].flip(1)
    conv = torch.fft.ifft(torch.fft.fft(spec * chirp, n=P) * torch.fft.fft(ker))
    return conv[:, :width] * chirp


def _ring_groups(N):
    """Ring indices (0 = the northernmost pair) in groups of similar length, few at a time."""
    count = _rings(N)[0]
    width = 1 << np.ceil(np.log2(count)).astype(int)
    for w in np.unique(width):
        ids = np.nonzero(width == w)[0]
        step = max(1, (1 << 24) // int(w))
        for i in range(0, len(ids), step):
            yield ids[i:i + step]


def _exact_synthesis(alm, N, L, M, K):
    count, _, s = _rings(N)
    q = torch.zeros((2, M + 1, 2 * N, 2 * K), device=DEV, dtype=torch.float64)
    a2 = torch.view_as_real(alm).reshape(-1, 2 * K)
    for l0, lam in _lambda_blocks(N, L, M):
        n, top = lam.shape[:2]
        idx, live = _rows(L, M, l0, n, top)
        a = a2[idx.reshape(-1)].reshape(n, top, 2 * K) * live[:, :, None]
        par = (torch.arange(l0, l0 + n, device=DEV)[:, None] -
               torch.arange(top, device=DEV)[None, :]) % 2
        if K == 1:
            for j in range(n):
                for p in range(2):
                    v = a[j] * (par[j] == p)[:, None]
                    for c in range(2):
                        q[p, :top, :, c].addcmul_(lam[j], v[:, c, None])
        else:
            w = lam.permute(1, 2, 0).contiguous()
            for p in range(2):
                v = (a * (par == p)[:, :, None]).permute(1, 0, 2).contiguous()
                q[p, :top] += torch.bmm(w, v)
    q = torch.view_as_complex(q.reshape(2, M + 1, 2 * N, K, 2))
    m = torch.arange(M + 1, device=DEV)
    c_m = torch.where(m == 0, 1.0, 2.0).double()
    out = torch.empty((12 * N * N, K), device=DEV, dtype=torch.float64)
    first = np.concatenate([[0], np.cumsum(count)])
    for ids in _ring_groups(N):
        nn = torch.from_numpy(count[ids]).to(DEV)
        phase = math.pi * ((m[None, :] * torch.from_numpy(s[ids]).to(DEV)[:, None]) %
                           (2 * nn[:, None])).double() / nn[:, None]
        ph = torch.polar(c_m.expand_as(phase).contiguous(), phase)
        at = (m[None, :] % nn[:, None])
        width = int(count[ids].max())
        for k in range(K):
            e, o = (q[p, :, torch.from_numpy(ids).to(DEV), k].transpose(0, 1) for p in (0, 1))
            for south in (False, True):
                g = torch.view_as_real(((e - o) if south else (e + o)) * ph)
                spec = torch.zeros((len(ids), width, 2), device=DEV, dtype=torch.float64)
                for c in range(2):
                    spec[:, :, c].scatter_add_(1, at, g[:, :, c])
                f = _ring_dft(torch.view_as_complex(spec), nn).real
                for v, i in enumerate(ids):
                    if south and i == 2 * N - 1:
                        continue
                    b = 12 * N * N - first[i] - count[i] if south else first[i]
                    out[b:b + count[i], k] = f[v, : count[i]]
    return out


def _exact_adjoint(sky, N, L, M, K):
    count, _, s = _rings(N)
    first = np.concatenate([[0], np.cumsum(count)])
    m = torch.arange(M + 1, device=DEV)
    q = torch.zeros((2, M + 1, 2 * N, K), device=DEV, dtype=torch.complex128)
    for ids in _ring_groups(N):
        nn = torch.from_numpy(count[ids]).to(DEV)
        at_ring = torch.from_numpy(ids).to(DEV)
        phase = math.pi * ((m[None, :] * torch.from_numpy(s[ids]).to(DEV)[:, None]) %
                           (2 * nn[:, None])).double() / nn[:, None]
        ph = torch.polar(torch.ones_like(phase), -phase)
        at = (m[None, :] % nn[:, None])
        width = int(count[ids].max())
        for k in range(K):
            for south in (False, True):
                f = torch.zeros((len(ids), width), device=DEV, dtype=torch.complex128)
                for v, i in enumerate(ids):
                    if south and i == 2 * N - 1:
                        continue
                    b = 12 * N * N - first[i] - count[i] if south else first[i]
                    f[v, : count[i]] = sky[b:b + count[i], k].to(torch.complex128)
                g = torch.gather(_ring_dft(f, nn).conj(), 1, at) * ph
                q[0, :, at_ring, k] += g.transpose(0, 1)
                q[1, :, at_ring, k] += (-g if south else g).transpose(0, 1)
    q = torch.view_as_real(q).reshape(2, M + 1, 2 * N, 2 * K)
    out = torch.zeros((_nalm(L, M), 2 * K), device=DEV, dtype=torch.float64)
    for l0, lam in _lambda_blocks(N, L, M):
        n, top = lam.shape[:2]
        idx, live = _rows(L, M, l0, n, top)
        par = (torch.arange(l0, l0 + n, device=DEV)[:, None] -
               torch.arange(top, device=DEV)[None, :]) % 2
        w = lam.transpose(0, 1).contiguous()
        b = [torch.bmm(w, q[p, :top].contiguous()).transpose(0, 1) for p in (0, 1)]
        b = torch.where((par == 1)[:, :, None], b[1], b[0])
        out[idx[live]] = b[live]
    out[L + 1:] *= 2.0
    return torch.view_as_complex(out.reshape(-1, K, 2))


def _too_long(N, L, M, K):
    """Whether the 64-bit computation takes more than some 20 seconds or 100 GB."""
    return L * (M + 1.0) * 2 * N > 8.0e10 or (M + 1.0) * 2 * N * K * 32 > 3.0e10


def exact(case, seed):
    if case["kind"] == "batch":
        alms = _inputs(case, seed)["alms"]
        # the large requests would take long: the others stand for them
        return [None if n > 512 else _exact_synthesis(a, n, l, m, k)
                for a, (n, l, m, k) in zip(alms, _requests(case))]
    N, L, M, K = (case[k] for k in ("N", "L", "M", "K"))
    if _too_long(N, L, M, K):
        return None
    x = _inputs(case, seed)
    if case["kind"] == "adjoint":
        return _exact_adjoint(x["map"], N, L, M, K)
    sky = _exact_synthesis(x["alm"], N, L, M, K)
    if case["kind"] == "grad":
        return {"map": sky, "grad": _exact_adjoint(x["weight"] * (sky - x["data"]), N, L, M, K)}
    return sky.cpu().numpy() if case["kind"] == "host" else sky
