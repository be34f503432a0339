// Adjoint of the synthesis (map -> a_lm): b = Y^T g.
//
// The synthesis evaluates, exactly at every pixel (the aliased c2r of the
// ring stage is an exact trigonometric-polynomial evaluation),
//   f(theta_p, phi_p) = sum_{l, m} c_m Re(a_lm Lambda_l^m(theta_p) e^{i m phi_p}),
// c_0 = 1, c_m = 2 (m > 0).  With the real inner products <f, g> = sum f g and
// <a, b> = sum Re(conj(a) b), its adjoint is
//   b_lm = c_m sum_p g_p Lambda_l^m(theta_p) e^{-i m phi_p},
// the unweighted analysis.  b is also the gradient d<f, g>/dRe(a) +
// i d<f, g>/dIm(a) (torch's convention for complex leaves).  The reference's
// only GPU code computes the transposed Legendre stage of this direction
// (wavemoth/cuda/legendre_transform.cu.in:297-679).
//
// Stages:
//  1. k_ring_adjoint: per ring pair, F_m(ring) = e^{-i m phi0} G^[m mod n]
//     with G^ the forward real DFT of the ring (conjugate-symmetric for
//     bins past n/2), then q_even = F_north + F_south, q_odd = F_north -
//     F_south (the equator ring feeds both), into the [R][2][M+1][K] buffer.
//  2. k_legendre_adj: b~_l = sum_rings L~_l(x_r) q_{parity(l-m)}(r) with the
//     same recurrences, seeds and l-segments as the synthesis, the sum over
//     rings on the matrix cores.
//  3. k_adj_finish: b_lm = c_m A_l sum_groups b~ into the m-major layout.
#include <cmath>
#include <mutex>

#include "wm_fft16.h"
#include "wm_host.h"

namespace wm {

using namespace fft;

// One block per (ring pair, map), the maps of a q group on one XCD.  MAXP: the
// plan's longest transform (Bluestein length, or twice a power-of-two ring's
// h); the per-thread loops and FFT passes are sized for it.
template <int MAXP>
__global__ __launch_bounds__(NT) void k_ring_adjoint(LegTables t, RingTables rt, int first,
                                                     int count, int lds_slots,
                                                     const double *__restrict__ map) {
  constexpr int kHalf = (MAXP / 2 + 1 + NT - 1) / NT;  // h-range entries per thread
  constexpr int kFull = (MAXP + NT - 1) / NT;          // P-range entries per thread
  extern __shared__ double2 lds[];
  double2 *twl = lds + lds_slots - kTwSlots;
  int pi, k;
  if (!ring16_job(blockIdx.x, 1, 0, t.K, count, &pi, &k)) return;
  const RingPair rp = rt.pairs[rt.order[first + pi]];
  const int n = rp.n, h = n / 2, K = t.K, M = t.M, P = rp.P;
  const bool south = rp.pix_s >= 0;
  const double2 *chirp = rt.chirp + rp.chirp_off;
  const double2 *vhat = rt.vhat + rp.vhat_off;
  load_twiddles(twl, rt.twiddle);
  const int nhemi = south ? 2 : 1;
  {
    double2 *qe = t.qbuf + q_index(rp.r, 0, k, 0, K, M + 1);  // element m at [m * G]
    double2 *qo = t.qbuf + q_index(rp.r, 1, k, 0, K, M + 1);
    for (int hemi = 0; hemi < nhemi; ++hemi) {
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const double *g = map + (hemi ? rp.pix_s : rp.pix_n) * K;
      // z_p = g_{2p} + i g_{2p+1}; Z = DFT_h(z), computed as conj(IDFT(conj z))
      // for Bluestein lengths
#pragma unroll
      for (int i = 0; i < kHalf; ++i) {
        const int p = tid + NT * i;
        if (p < h) {
          const double2 z = make_double2(g[(int64_t)(2 * p) * K + k], g[(int64_t)(2 * p + 1) * K + k]);
          lds[pidx(p)] = (P == 0) ? z : cmul(cconj(z), chirp[p]);
        }
      }
      if (P == 0) {
        __syncthreads();
        lds_fft<false, MAXP>(lds, h, twl);
      } else {
#pragma unroll
        for (int i = 0; i < kFull; ++i) {
          const int a = h + tid + NT * i;
          if (a < P) lds[pidx(a)] = make_double2(0.0, 0.0);
        }
        __syncthreads();
        lds_fft<false, MAXP>(lds, P, twl);
#pragma unroll
        for (int i = 0; i < kFull; ++i) {
          const int a = tid + NT * i;
          if (a < P) lds[pidx(a)] = cmul(lds[pidx(a)], vhat[a]);
        }
        __syncthreads();
        lds_fft<true, MAXP>(lds, P, twl);
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
          const int p = tid + NT * i;
          if (p < h) lds[pidx(p)] = cconj(cmul(lds[pidx(p)], chirp[p]));
        }
        __syncthreads();
      }
      // real-DFT split: G^_k = (Z_k + conj Z_{h-k})/2 - (i/2) e^{-2 pi i k/n}
      // (Z_k - conj Z_{h-k}), k in [0, h], Z_h = Z_0.  Each thread reads and
      // rewrites only its own pair (a, h - a), so the split runs in place.
      {
        const double2 step = expipi(-2 * NT, n);
        double2 om = expipi(-2 * (int64_t)tid, n);
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
          const int a = tid + NT * i;
          if (a <= h / 2) {
            const int c = h - a;
            const double2 za = lds[pidx(a)], zc = lds[pidx(c % h)];
            const double2 e = cadd(za, cconj(zc)), d = csub(za, cconj(zc));
            // -(i/2) om d
            const double2 od = cmul(om, d);
            const double2 ga = make_double2(0.5 * (e.x + od.y), 0.5 * (e.y - od.x));
            // partner: e' = conj(e), d' = -conj(d), om' = e^{-2 pi i c/n} = -conj(om)
            const double2 oc = make_double2(-om.x, om.y);
            const double2 dc = make_double2(-d.x, d.y);
            const double2 odc = cmul(oc, dc);
            const double2 gc = make_double2(0.5 * (e.x + odc.y), 0.5 * (-e.y - odc.x));
            lds[pidx(a)] = ga;
            lds[pidx(c)] = gc;
          }
          om = cmul(om, step);
        }
      }
      __syncthreads();
      // F_m = e^{-i pi s m / n} G^[m mod n] (conjugate past n/2), into q
      {
        const double2 step = expipi(-(int64_t)rp.s * NT, n);
        double2 w = expipi(-(int64_t)rp.s * tid, n);
        for (int m0 = 0; m0 <= M; m0 += NT * kHalf) {
#pragma unroll
          for (int i = 0; i < kHalf; ++i) {
            const int m = m0 + tid + NT * i;
            if (m <= M) {
              if (i == 0 && m0 > 0) w = expipi(-(int64_t)rp.s * m, n);
              const int kk = m % n;
              const double2 v = (kk <= h) ? lds[pidx(kk)] : cconj(lds[pidx(n - kk)]);
              const double2 f = cmul(v, w);
              const int64_t o = (int64_t)m * q_group(K);
              if (hemi == 0) {
                qe[o] = f;
                qo[o] = f;
              } else {
                qe[o] = cadd(qe[o], f);
                qo[o] = csub(qo[o], f);
              }
            }
            w = cmul(w, step);
          }
        }
      }
      __syncthreads();
    }
  }
}

// The ring adjoint of power-of-two rings with mmax < n (the forward belt
// kernel's rings) on the register FFT: a job of T = h/16 threads per (ring
// pair, map).  Per hemisphere: z_p = g_{2p} + i g_{2p+1}
// for p = j + T rho, Z = DFT_h(z) in registers (canonical layout), Z into the
// job's buffer and back for the partner Z_{h-k}, then for the thread's own
// k = j + T rho
//   G^_k = (Z_k + conj Z_{h-k})/2 - (i/2) e^{-2 pi i k/n} (Z_k - conj Z_{h-k})
// (Z_h = Z_0; thread 0 also forms G^_h), F_m = e^{-i pi s m/n} G^_m for
// m = k <= mmax, and q_e = F_N + F_S, q_o = F_N - F_S (the southern pass
// adds to what the same thread wrote for the northern ring).
// Blocks hold at least one wave and `maps` jobs where they fit in 512 threads,
// so that a few rings still reach many CUs and several blocks share one.  The
// belt takes all maps of a q group (they share lines of q and of the map:
// 3 maps at Nside 512 64 us, 79 with one job per block), the caps, whose time
// is in their transforms, one job (52 us, 60 with the group's).
constexpr int kAdjRB = 2 * fft16::kThreads;  // most threads per block
inline int adj16_threads(int P, int maps) {
  int n = P / 16;
  while (n < kAdjRB && (n < 64 || n / (P / 16) < maps)) n *= 2;
  return n;
}
constexpr size_t adj16_bytes(int P, int threads) {
  return (size_t)(kTwSlots + threads / (P / 16) * fft16::job_slots(P)) * sizeof(double2);
}

template <int P>
__global__ __launch_bounds__(kAdjRB) void k_ring_adjoint16(LegTables t, RingTables rt, int first,
                                                           int count,
                                                           const double *__restrict__ map) {
  using fft16::pad;
  constexpr int T = P / 16;
  const int J = blockDim.x / T;
  extern __shared__ double2 lds[];
  double2 *twl = lds;
  for (int u = threadIdx.x; u < kTwSlots; u += blockDim.x)  // read after the FFT's first barrier
    twl[u] = (u < kTwC) ? rt.twiddle[u * 64] : rt.twiddle[u - kTwC];
  const int jb = threadIdx.x / T;
  int j = threadIdx.x - jb * T;
  double2 *buf = lds + kTwSlots + jb * fft16::job_slots(P);
  const int K = t.K, M = t.M;
  int pi, k;
  // a job is padding only if every later one of its block is
  if (!ring16_job(blockIdx.x, J, 0, K, count, &pi, &k)) return;
  const bool act = ring16_job(blockIdx.x, J, jb, K, count, &pi, &k);
  if (!act) pi = k = 0;
  const RingPair rp = rt.pairs[rt.order[first + pi]];
  const int n = rp.n;
  const bool south = rp.pix_s >= 0;
  double2 *qe = t.qbuf + q_index(rp.r, 0, k, 0, K, M + 1);
  double2 *qo = t.qbuf + q_index(rp.r, 1, k, 0, K, M + 1);
  const int64_t qs = q_group(K);
  auto put = [&](int m, double2 f, int hemi) {
    const int64_t o = (int64_t)m * qs;
    if (hemi == 0) {
      qe[o] = f;
      qo[o] = f;
    } else {
      qe[o] = cadd(qe[o], f);
      qo[o] = csub(qo[o], f);
    }
  };
#pragma unroll 1
  for (int hemi = 0; hemi < 2; ++hemi) {  // every job takes both passes (block barriers)
    const bool on = act && (hemi == 0 || south);
    const double *gp = map + (int64_t)(hemi && south ? rp.pix_s : rp.pix_n) * K + k;
    double2 v[16];
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) {
      const int64_t p = j + T * rho;
      v[rho] = on ? make_double2(gp[2 * p * K], gp[(2 * p + 1) * K]) : make_double2(0.0, 0.0);
    }
    fft16::fft<P, false>(v, buf, twl, j);
    asm volatile("" : "+v"(j));
    __syncthreads();  // the transform's last reads of buf done
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) buf[pad(j + T * rho)] = v[rho];
    __syncthreads();
    const double2 wstep = expipi(-(int64_t)rp.s * T, n), ostep = expipi(-2 * (int64_t)T, n);
    double2 w = expipi(-(int64_t)rp.s * j, n), om = expipi(-2 * (int64_t)j, n);
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) {
      const int kk = j + T * rho;
      const double2 za = v[rho], zc = buf[pad((P - kk) & (P - 1))];
      const double2 e = cadd(za, cconj(zc)), d = csub(za, cconj(zc));
      const double2 od = cmul(om, d);
      const double2 gk = make_double2(0.5 * (e.x + od.y), 0.5 * (e.y - od.x));
      if (on && kk <= M) put(kk, cmul(gk, w), hemi);
      // m = n - k past h: G^_m = conj G^_k, e^{-i pi s m/n} = (-1)^s conj w
      if (on && kk > 0 && n - kk <= M) {
        const double2 f = cconj(cmul(gk, w));
        put(n - kk, rp.s ? make_double2(-f.x, -f.y) : f, hemi);
      }
      w = cmul(w, wstep);
      om = cmul(om, ostep);
    }
    if (j == 0 && on && P <= M) {
      // G^_h from Z_0 (partner of k = 0): e^{-2 pi i h/n} = -1
      const double2 z0 = v[0];
      const double2 e = cadd(z0, cconj(z0)), d = csub(z0, cconj(z0));
      const double2 gh = make_double2(0.5 * (e.x - d.y), 0.5 * (e.y + d.x));
      put(P, cmul(gh, expipi(-(int64_t)rp.s * P, n)), hemi);
    }
  }
}

#define WM_ADJ16_SIZES(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)

// The ring adjoint of the forward cap kernel's rings (h = n/2 not a power
// of two, n > mmax) on the register FFT: Z = DFT_h(z) as conj(IDFT(conj z))
// by Bluestein's chirp z-transform of length P = next_pow2(2h - 1) (the
// plan's non-split chirp and vhat), u_a = conj(z_a) chirp_a (a < h), then
// FFT_P, times vhat, inverse FFT_P, Z_p = conj(chirp_p u_p); the split of
// k_ring_adjoint16 for G^_0 .. G^_h into the job's buffer, and F_m =
// e^{-i pi s m/n} G^[m] (m <= h) or conj G^[n - m] (h < m <= mmax < n).
template <int P>
__global__ __launch_bounds__(kAdjRB) void k_ring_adjoint_cap16(LegTables t, RingTables rt,
                                                               int first, int count,
                                                               const double *__restrict__ map) {
  using fft16::pad;
  constexpr int T = P / 16;
  const int J = blockDim.x / T;
  extern __shared__ double2 lds[];
  double2 *twl = lds;
  for (int u = threadIdx.x; u < kTwSlots; u += blockDim.x)  // read after the FFT's first barrier
    twl[u] = (u < kTwC) ? rt.twiddle[u * 64] : rt.twiddle[u - kTwC];
  const int jb = threadIdx.x / T;
  int j = threadIdx.x - jb * T;
  double2 *buf = lds + kTwSlots + jb * fft16::job_slots(P);
  const int K = t.K, M = t.M;
  int pi, k;
  // a job is padding only if every later one of its block is
  if (!ring16_job(blockIdx.x, J, 0, K, count, &pi, &k)) return;
  const bool act = ring16_job(blockIdx.x, J, jb, K, count, &pi, &k);
  if (!act) pi = k = 0;
  const RingPair rp = rt.pairs[rt.order[first + pi]];
  const int n = rp.n, h = n / 2;
  const bool south = rp.pix_s >= 0;
  const double2 *chirp = rt.chirp + rp.chirp_off;  // [h]
  const double2 *vhat = rt.vhat + rp.vhat_off;     // [P]
  double2 *qe = t.qbuf + q_index(rp.r, 0, k, 0, K, M + 1);
  double2 *qo = t.qbuf + q_index(rp.r, 1, k, 0, K, M + 1);
  const int64_t qs = q_group(K);
#pragma unroll 1
  for (int hemi = 0; hemi < 2; ++hemi) {  // every job takes both passes (block barriers)
    const bool on = act && (hemi == 0 || south);
    const double *gp = map + (int64_t)(hemi && south ? rp.pix_s : rp.pix_n) * K + k;
    double2 v[16];
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) {
      const int a = j + T * rho;
      double2 x = make_double2(0.0, 0.0);
      if (on && a < h) {
        const double2 z = make_double2(gp[2 * (int64_t)a * K], gp[(2 * (int64_t)a + 1) * K]);
        x = cmul(cconj(z), chirp[a]);
      }
      v[rho] = x;
    }
    fft16::fft<P, false>(v, buf, twl, j);
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) v[rho] = cmul(v[rho], vhat[j + T * rho]);
    fft16::fft<P, true>(v, buf, twl, j);
    asm volatile("" : "+v"(j));
    __syncthreads();  // the transform's last reads of buf done
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) {
      const int p = j + T * rho;
      if (p < h) buf[pad(p)] = cconj(cmul(v[rho], chirp[p]));  // Z_p
    }
    __syncthreads();
    // G^_k, k = j + T rho <= h (k = h from Z_0), kept in registers until
    // every partner read is done, then into buf
    double2 gk[16];
    {
      const double2 ostep = expipi(-2 * (int64_t)T, n);
      double2 om = expipi(-2 * (int64_t)j, n);
#pragma unroll
      for (int rho = 0; rho < 16; ++rho) {
        const int kk = j + T * rho;
        double2 gv = make_double2(0.0, 0.0);
        if (kk <= h) {
          const double2 za = buf[pad(kk < h ? kk : 0)], zc = buf[pad(kk == 0 || kk == h ? 0 : h - kk)];
          const double2 e = cadd(za, cconj(zc)), d = csub(za, cconj(zc));
          const double2 od = cmul(om, d);
          gv = make_double2(0.5 * (e.x + od.y), 0.5 * (e.y - od.x));
        }
        gk[rho] = gv;
        om = cmul(om, ostep);
      }
    }
    __syncthreads();  // partner reads done
#pragma unroll
    for (int rho = 0; rho < 16; ++rho) {
      const int kk = j + T * rho;
      if (kk <= h) buf[pad(kk)] = gk[rho];
    }
    __syncthreads();
    if (on) {
      for (int m = j; m <= M; m += T) {
        const double2 gv = m <= h ? buf[pad(m)] : cconj(buf[pad(n - m)]);
        const double2 f = cmul(gv, expipi(-(int64_t)rp.s * m, n));
        const int64_t o = (int64_t)m * qs;
        if (hemi == 0) {
          qe[o] = f;
          qo[o] = f;
        } else {
          qe[o] = cadd(qe[o], f);
          qo[o] = csub(qo[o], f);
        }
      }
    }
    __syncthreads();  // F reads of buf done before the next pass writes it
  }
}

#define WM_ADJ_CAP_SIZES(X) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)


__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x from the lane that DPP control C names.
template <int C>
__device__ __forceinline__ double dpp_move(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, C, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), C, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (unsigned long long)lo | (unsigned long long)hi << 32);
}
// x of lane ^ 8 (row_ror:8) and of lane ^ 4 (row_half_mirror, then the four
// lanes of a quad reversed).
__device__ __forceinline__ double lane_xor8(double x) { return dpp_move<0x128>(x); }
__device__ __forceinline__ double lane_xor4(double x) { return dpp_move<0x1b>(dpp_move<0x141>(x)); }

// b~ partial sums on the FP64 matrix cores.  A wave is one work item (m, ring
// group g): units of 16 GR rings one after the other, for each the whole
// l-range of the unit's rings in four segments, as in the matrix-core
// synthesis sweep (the same segments and checkpoints).  Lane 4 i + u steps
// segment u of ring i of every 16-ring group: with A[row][k] on lane row +
// 4 block + 16 k that is a product, in each of the 4 blocks of
// v_mfma_f64_4x4x4f64, of 4 l (one per segment) with 4 rings as it stands, and
// B has q of the same ring on lane 4 i + column: 16 distinct rings in 64 lanes.
// The GR products of a step add up in one accumulator; the 4 blocks of 4
// steps are then summed by two exchange-and-add stages that leave step b in
// block b, one row of 4 columns per lane quad.
//
// FP64 matrix and vector instructions share one pipe, and a product takes four
// times a vector instruction.  Units in the middle latitudes run in the pair
// form (legendre.hip): a step of two l costs 2 vector instructions and one
// product per map, whose 4 columns are the real and imaginary parts of the
// even and, times x, the odd sums.  The other units step l by l: 2 vector
// instructions and, for every 2 maps, one product of which one parity's
// columns are wanted; per two l and 16 rings 4 + 8 against 2 + 4 instruction
// times at 1 map, 4 + 16 against 2 + 12 at 3 (this kernel with one-step units
// only / as it is: Nside 2048, lmax 4096, 1 map 6.46 / 4.40 ms; Nside 512, lmax
// 1024, 3 maps 0.282 / 0.247 ms).  A group's units are all of one form: its
// rows of partial sums are b~_l or the sums of p_k.

// The units c = c0, c0 + step, ... of `units` one-step units (those below ua,
// then those from ub on).
template <int KN, int GR>
__device__ __forceinline__ void adj_units(const LegTables &t, int c0, int step, int units, int ua,
                                          int ub, int m, int kb, double *prow, int lane,
                                          double2 *seeds) {
  constexpr int ST = 4, RU = 16 * GR, CG = (KN + 1) / 2, kn = KN;
  const int L = t.L, R = t.R, M = t.M, K = t.K;
  const int u = lane & 3, ring = lane >> 2;  // segment (and column of B), ring in a group
  const int b = ring & 3, ds = lane >> 4;    // block, segment of the result rows
  const int64_t offm = t.off[m];
  const double *ct0 = t.ctil + (offm - m);
  const double *cs0 = t.cscale + offm / kChunk;
  const int64_t rstride = 2 * (int64_t)K;  // doubles per row of the partial sums (times lmax past 2^32)
  bool first = true;
  for (int ci = c0; ci < units; ci += step) {
    const int c = ci < ua ? ci : ci - ua + ub;
    const int l0 = __builtin_amdgcn_readfirstlane(
        t.seg_l0[(int64_t)m * t.SW + c * RU / kSegRings]);
    if (l0 > L) continue;
    if (first) {  // rows no unit has written yet
      for (int j = lane; j < (l0 - m) * 2 * kn; j += 64) {
        const int l = j / (2 * kn);
        prow[(int64_t)l * rstride + (j - l * 2 * kn)] = 0.0;
      }
    }
    const int nc = (L - l0) / kChunk + 1, ns = (nc + 3) / 4;
    const int cb = u * ns;
#pragma unroll
    for (int i = 0; i < RU / 64; ++i) {
      const int r = c * RU + 64 * i + lane;
      if (r < R) seeds[64 * i + lane] = t.seed_v[(int64_t)m * R + r];
    }
    double x[GR], prev[GR], cur[GR], bq[2][CG][GR];
    int sl[GR];
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      const int r = c * RU + 16 * i + ring;
      const bool ok = r < R;
      x[i] = ok ? t.ring_x[r] : 0.0;
      sl[i] = ok ? t.seed_l[(int64_t)m * R + r] : kSeedNone;
      double2 v = make_double2(0.0, 0.0);
      if (ok && u > 0 && cb < nc) v = t.ckpt[((int64_t)m * 3 + u - 1) * R + r];
      prev[i] = v.x;
      cur[i] = v.y;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
          const int k = 2 * cg + (u >> 1);
          bq[p][cg][i] = ok && k < kn
                             ? ((const double *)t.qbuf)[2 * q_index(r, p, kb + k, m, K, M + 1) + (u & 1)]
                             : 0.0;
        }
    }
    const double *ct = ct0 + l0, *cs = cs0 + (l0 - m) / kChunk;
    double *pr = prow + (int64_t)(l0 - m) * rstride + u;
    unsigned e = kChunk * (unsigned)(cb < nc ? cb : nc - 1);
    double cc[ST], S = cs[e / kChunk], old[CG];
#pragma unroll
    for (int s = 0; s < ST; ++s) cc[s] = ct[e + s];
    // row of the lane's results: segment ds, step b of a 4-step block; what
    // earlier units left there is read one block ahead
    const int drow0 = kChunk * ds * ns + b;
    auto load_old = [&](int blk, double (&o)[CG]) {
      const int dr = drow0 + ST * blk;
      const bool rok = !first && ds * ns + blk / (kChunk / ST) < nc && l0 + dr <= L &&
                       blk < ns * (kChunk / ST);
#pragma unroll
      for (int cg = 0; cg < CG; ++cg)
        o[cg] = rok && 4 * cg + u < 2 * kn ? pr[dr * rstride + 4 * cg] : 0.0;
    };
    wave_sync_lds();
    load_old(0, old);
    for (int j = 0; j < ns; ++j) {
      const int ls = l0 + kChunk * (cb + j);
      bool hit = false;
#pragma unroll
      for (int i = 0; i < GR; ++i) hit |= sl[i] == ls;
      if (__any(hit)) {
#pragma unroll
        for (int i = 0; i < GR; ++i)
          if (sl[i] == ls) {
            const double2 v = seeds[16 * i + ring];
            prev[i] = v.x;
            cur[i] = v.y;
          }
      }
      if (3 * ns + j >= nc) {  // past the rows of some segments
        asm volatile("");  // stays a branch: as selects 4 GR instructions a chunk, 4.51 / 4.40 ms
        const bool past = cb + j >= nc;
#pragma unroll
        for (int i = 0; i < GR; ++i) {
          prev[i] = past ? 0.0 : prev[i];
          cur[i] = past ? 0.0 : cur[i];
        }
      }
      const unsigned en = kChunk * (unsigned)(cb + j + 1 < nc ? cb + j + 1 : nc - 1);
      double Sn = S;
      const int drow = drow0 + kChunk * j;
      const bool dok = ds * ns + j < nc;
#pragma unroll
      for (int s0 = 0; s0 < kChunk; s0 += ST) {
        double cn[ST], on[CG];
#pragma unroll
        for (int s = 0; s < ST; ++s) cn[s] = ct[(s0 + ST < kChunk ? e + s0 + ST : en) + s];
        if (s0 + ST == kChunk) Sn = cs[en / kChunk];
        const bool rok = dok && l0 + drow + s0 <= L;
        const int64_t ro = (drow + s0) * rstride;
        load_old(j * (kChunk / ST) + s0 / ST + 1, on);
        __builtin_amdgcn_sched_barrier(0);
        double d[ST][CG];
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) d[s][cg] = 0.0;
        // two steps of a group at a time: their products go to two accumulators
#pragma unroll
        for (int s = 0; s < ST; s += 2)
#pragma unroll
          for (int i = 0; i < GR; ++i) {
            const double nx = fma(x[i], cur[i], -(cc[s] * prev[i]));
#pragma unroll
            for (int cg = 0; cg < CG; ++cg) {
              d[s][cg] =
                  __builtin_amdgcn_mfma_f64_4x4x4f64(cur[i], bq[0][cg][i], d[s][cg], 0, 0, 0);
              d[s + 1][cg] =
                  __builtin_amdgcn_mfma_f64_4x4x4f64(nx, bq[1][cg][i], d[s + 1][cg], 0, 0, 0);
            }
            prev[i] = nx;
            cur[i] = fma(x[i], nx, -(cc[s + 1] * cur[i]));
          }
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
          const bool b2 = b & 2, b1 = b & 1;
          const double e0 = (b2 ? d[2][cg] : d[0][cg]) + lane_xor8(b2 ? d[0][cg] : d[2][cg]);
          const double e1 = (b2 ? d[3][cg] : d[1][cg]) + lane_xor8(b2 ? d[1][cg] : d[3][cg]);
          const double f = (b1 ? e1 : e0) + lane_xor4(b1 ? e0 : e1);
          if (rok && 4 * cg + u < 2 * kn) pr[ro + 4 * cg] = old[cg] + f;
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) cc[s] = cn[s];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) old[cg] = on[cg];
      }
#pragma unroll
      for (int i = 0; i < GR; ++i) {
        prev[i] *= S;
        cur[i] *= S;
      }
      S = Sn;
      e = en;
    }
    // the next unit's segments give these rows to other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    first = false;
  }
  if (first)
    for (int j = lane; j < (L - m + 1) * 2 * kn; j += 64) {
      const int l = j / (2 * kn);
      prow[(int64_t)l * rstride + (j - l * 2 * kn)] = 0.0;
    }
}


// The pair-form units c = c0, c0 + step, ... < ub: row k of the partial sums
// takes the places of the rows l = m + 2 k (sums of p_k q_even) and l + 1
// (p_k x q_odd).  Seeds and checkpoints are the one-step form's, converted.
template <int KN, int GR>
__device__ __forceinline__ void adj_pair_units(const LegTables &t, int c0, int step, int ub, int m,
                                               int kb, double *prow, int lane, double2 *seeds) {
  constexpr int ST = 4, RU = 16 * GR, KC = kChunk / 2;  // steps of a chunk
  const int L = t.L, M = t.M, K = t.K;
  const int u = lane & 3, ring = lane >> 2;  // segment (and column of B), ring in a group
  const int b = ring & 3, ds = lane >> 4;    // block, segment of the result rows
  const int64_t offm = t.off[m];
  const double *ct0 = t.ctil + (offm - m);
  const double2 *h0 = t.pair_h + offm / kChunk;
  const int64_t rstride = 2 * (int64_t)K;  // doubles per row of the partial sums (times lmax past 2^32)
  bool first = true;
  for (int c = c0; c < ub; c += step) {
    const int l0 = __builtin_amdgcn_readfirstlane(
        t.seg_l0[(int64_t)m * t.SW + c * RU / kSegRings]);
    if (l0 > L) continue;
    if (first) {  // rows no unit has written yet
      for (int j = lane; j < (l0 - m) * 2 * KN; j += 64) {
        const int l = j / (2 * KN);
        prow[(int64_t)l * rstride + (j - l * 2 * KN)] = 0.0;
      }
    }
    const int nc = (L - l0) / kChunk + 1, ns = (nc + 3) / 4;
    const int cb = u * ns;
    // (L~_{l-1}, L~_l) at the start of a chunk -> (p_{k-1}, p_k)
    auto to_pair = [&](double2 v, double x, int l) {
      const double2 h = h0[(l - m) / kChunk];
      const double rx = 1.0 / x;
      return make_double2(v.x * h.y * rx, fma(x, v.y, -(ct0[l] * v.x)) * h.x * rx);
    };
#pragma unroll
    for (int i = 0; i < RU / 64; ++i) {
      const int r = c * RU + 64 * i + lane;
      const int s = t.seed_l[(int64_t)m * t.R + r];
      if (s <= L) seeds[64 * i + lane] = to_pair(t.seed_v[(int64_t)m * t.R + r], t.ring_x[r], s);
    }
    const int zone = __builtin_amdgcn_readfirstlane(pair_zone(t.ring_x[c * RU + RU / 2]));
    double y[GR], prev[GR], cur[GR], bq[KN][GR];
    int sl[GR];
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      const int r = c * RU + 16 * i + ring;
      const double x = t.ring_x[r];
      y[i] = fma(x, x, -pair_centre(zone));
      sl[i] = t.seed_l[(int64_t)m * t.R + r];
      double2 v = make_double2(0.0, 0.0);
      if (u > 0 && cb < nc)
        v = to_pair(t.ckpt[((int64_t)m * 3 + u - 1) * t.R + r], x, l0 + kChunk * cb);
      prev[i] = v.x;
      cur[i] = v.y;
#pragma unroll
      for (int k = 0; k < KN; ++k) {
        const double q =
            ((const double *)t.qbuf)[2 * q_index(r, u >> 1, kb + k, m, K, M + 1) + (u & 1)];
        bq[k][i] = u >= 2 ? q * x : q;
      }
    }
    const double2 *pc = t.pair_t + (t.nlpad * zone + offm + l0 - m) / 2;
    double *pr = prow + (int64_t)(l0 - m + (u >> 1)) * rstride + (u & 1);
    unsigned e = KC * (unsigned)(cb < nc ? cb : nc - 1);
    double2 cc[ST];
    double old[KN];
#pragma unroll
    for (int s = 0; s < ST; ++s) cc[s] = pc[e + s];
    // row of the lane's results: segment ds, step b of a 4-step block; what
    // earlier units left there is read one block ahead
    const int drow0 = KC * ds * ns + b;
    auto load_old = [&](int blk, double (&o)[KN]) {
      const int dr = drow0 + ST * blk;
      const bool rok = !first && ds * ns + blk / (KC / ST) < nc && l0 + 2 * dr <= L &&
                       blk < ns * (KC / ST);
#pragma unroll
      for (int k = 0; k < KN; ++k) o[k] = rok ? pr[2 * dr * rstride + 2 * k] : 0.0;
    };
    wave_sync_lds();
    load_old(0, old);
    for (int j = 0; j < ns; ++j) {
      const int ls = l0 + kChunk * (cb + j);
      bool hit = false;
#pragma unroll
      for (int i = 0; i < GR; ++i) hit |= sl[i] == ls;
      if (__any(hit)) {
#pragma unroll
        for (int i = 0; i < GR; ++i)
          if (sl[i] == ls) {
            const double2 v = seeds[16 * i + ring];
            prev[i] = v.x;
            cur[i] = v.y;
          }
      }
      if (3 * ns + j >= nc) {  // past the rows of some segments
        asm volatile("");  // stays a branch: as selects 4 GR instructions a chunk, 4.51 / 4.40 ms
        const bool past = cb + j >= nc;
#pragma unroll
        for (int i = 0; i < GR; ++i) {
          prev[i] = past ? 0.0 : prev[i];
          cur[i] = past ? 0.0 : cur[i];
        }
      }
      const unsigned en = KC * (unsigned)(cb + j + 1 < nc ? cb + j + 1 : nc - 1);
      const int drow = drow0 + KC * j;
      const bool dok = ds * ns + j < nc;
#pragma unroll
      for (int s0 = 0; s0 < KC; s0 += ST) {
        double2 cn[ST];
        double on[KN];
#pragma unroll
        for (int s = 0; s < ST; ++s) cn[s] = pc[(s0 + ST < KC ? e + s0 + ST : en) + s];
        const bool rok = dok && l0 + 2 * (drow + s0) <= L;
        const int64_t ro = 2 * (drow + s0) * rstride;
        load_old(j * (KC / ST) + s0 / ST + 1, on);
        __builtin_amdgcn_sched_barrier(0);
        double d[ST][KN];
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
          for (int k = 0; k < KN; ++k) d[s][k] = 0.0;
        // two steps of a group at a time: their products go to two accumulators
#pragma unroll
        for (int s = 0; s < ST; s += 2)
#pragma unroll
          for (int i = 0; i < GR; ++i) {
            const double nx = fma(fma(cc[s].x, y[i], cc[s].y), cur[i], -prev[i]);
#pragma unroll
            for (int k = 0; k < KN; ++k) {
              d[s][k] = __builtin_amdgcn_mfma_f64_4x4x4f64(cur[i], bq[k][i], d[s][k], 0, 0, 0);
              d[s + 1][k] =
                  __builtin_amdgcn_mfma_f64_4x4x4f64(nx, bq[k][i], d[s + 1][k], 0, 0, 0);
            }
            prev[i] = nx;
            cur[i] = fma(fma(cc[s + 1].x, y[i], cc[s + 1].y), nx, -cur[i]);
          }
#pragma unroll
        for (int k = 0; k < KN; ++k) {
          const bool b2 = b & 2, b1 = b & 1;
          const double e0 = (b2 ? d[2][k] : d[0][k]) + lane_xor8(b2 ? d[0][k] : d[2][k]);
          const double e1 = (b2 ? d[3][k] : d[1][k]) + lane_xor8(b2 ? d[1][k] : d[3][k]);
          const double f = (b1 ? e1 : e0) + lane_xor4(b1 ? e0 : e1);
          if (rok) pr[ro + 2 * k] = old[k] + f;
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) cc[s] = cn[s];
#pragma unroll
        for (int k = 0; k < KN; ++k) old[k] = on[k];
      }
      e = en;
    }
    // the next unit's segments give these rows to other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    first = false;
  }
  if (first)
    for (int j = lane; j < (L - m + 1) * 2 * KN; j += 64) {
      const int l = j / (2 * KN);
      prow[(int64_t)l * rstride + (j - l * 2 * KN)] = 0.0;
    }
}

// Groups g < G1 take the one-step units, the others the pair-form units.
template <int KN, int GR>
__global__ __launch_bounds__(64, KN <= 2 ? 3 : 2) void k_legendre_adj(LegTables t, int G, int G1,
                                                                      int kb, double2 *partial) {
  constexpr int RU = 16 * GR;
  __shared__ double2 seeds[RU];  // of the unit's rings: a load where one joins would stall
  // block b runs on XCD b % 8; runs of 8 consecutive m share an XCD, since 8
  // entries of q (at one map) share a line
  const int xi = blockIdx.x >> 3, g = xi % G, mi = xi / G;
  const int m = ((mi >> 3) * 8 + (blockIdx.x & 7)) * 8 + (mi & 7);
  if (m > t.M) return;
  double *prow = (double *)(partial + ((int64_t)g * t.nlpad + t.off[m]) * t.K + kb);
  const int all = (t.R + RU - 1) / RU;
  int ua = all, ub = all;
  if (G1 < G) pair_units(t, RU, &ua, &ub);
  if (g < G1)
    adj_units<KN, GR>(t, g, G1, all - (ub - ua), ua, ub, m, kb, prow, threadIdx.x, seeds);
  else
    adj_pair_units<KN, GR>(t, ua + g - G1, G - G1, ub, m, kb, prow, threadIdx.x, seeds);
}

// b_lm = c_m sum_g, from b~ (times A_l) of the one-step groups and from the
// sums S_k of the pair-form groups: Lambda_{l+1} = x P_k, Lambda_l = A_{l+1} P_k
// + A_l P_{k-1}, P_k = s_k p_k.  Into the m-major complex layout; one thread
// per (row, map), so that each group's partial sums are read contiguously
// across the threads.
__global__ __launch_bounds__(256) void k_adj_finish(LegTables t, int G, int G1,
                                                    const double2 *__restrict__ partial,
                                                    double2 *__restrict__ alm) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int K = t.K;
  if (u >= t.nlpad * K) return;
  const int64_t j = u / K;
  const int k = (int)(u - j * K);
  const int m = t.chunk_m[j / kChunk];
  const int64_t jj = j - t.off[m];
  const int l = m + (int)jj;
  if (l > t.L) return;
  const int64_t rows = t.nlpad * K;
  const int64_t idx = (int64_t)m * (2 * t.L - m + 3) / 2 + jj;
  double2 acc = make_double2(0.0, 0.0);
  for (int g = 0; g < G1; ++g) acc = cadd(acc, partial[g * rows + u]);
  const double s = t.ascale[j];
  acc.x *= s;
  acc.y *= s;
  if (G1 < G) {
    double2 pk = make_double2(0.0, 0.0), pp = make_double2(0.0, 0.0);
    const bool two = !(jj & 1) && jj > 0;
    for (int g = G1; g < G; ++g) {
      pk = cadd(pk, partial[g * rows + u]);
      if (two) pp = cadd(pp, partial[g * rows + u - 2 * K]);
    }
    double w = t.pair_w[j / 2], wp = 0.0;
    if (!(jj & 1)) {
      w *= sqrt(t.ctil[j + 1]);
      if (two) wp = t.pair_w[j / 2 - 1] * sqrt(t.ctil[j]);
    }
    acc.x += fma(w, pk.x, wp * pp.x);
    acc.y += fma(w, pk.y, wp * pp.y);
  }
  const double cm = m == 0 ? 1.0 : 2.0;
  acc.x *= cm;
  acc.y = m == 0 ? 0.0 : acc.y * cm;
  alm[idx * K + k] = acc;
}

// Rings of a work unit: 8 groups of 16 while such units fill the chip's
// 1024 SIMDs a few times over, 4 groups below that.
static int adjoint_unit(const LegTables &t) {
  return (int64_t)(t.M + 1) * ((t.R + 127) / 128) >= 4096 ? 128 : 64;
}

int adjoint_groups(const LegTables &t) {
  // one wave per (m, group): groups up to one per unit, while the waves stay
  // below 20 per SIMD (more only add partial sums to write and read) and the
  // partial sums below 2 GiB
  const int units = (t.R + adjoint_unit(t) - 1) / adjoint_unit(t);
  const double row_bytes = (double)t.nlpad * t.K * sizeof(double2);
  int G = 1;
  while (2 * G <= units && (int64_t)(t.M + 1) * 2 * G <= 20480 &&
         row_bytes * 2 * G <= 2.0 * 1024 * 1024 * 1024)
    G *= 2;
  return G;
}

// Partial sums of the adjoint entry that allocates nothing
// (wavemoth_execute_adjoint_device_noalloc): a fixed array in device
// memory, held by each GPU the library runs on until the process ends.
// Every call on a GPU writes its rows before reading them (each wave of
// k_legendre_adj writes all of its own rows), so the contents left by an
// earlier call never matter; calls that overlap on one GPU race on it.
constexpr size_t kAdjScratchBytes = (size_t)256 << 20;
static __device__ __align__(256) double2 scratch[kAdjScratchBytes / sizeof(double2)];

size_t adjoint_scratch_elems() { return kAdjScratchBytes / sizeof(double2); }

// Device address of `scratch` on the current device (which must be
// `device`), looked up once per device; nullptr with the error set on
// failure.
double2 *adjoint_scratch(int device) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static double2 *addr[kMaxDevices] = {nullptr};
  if (device < 0 || device >= kMaxDevices) {
    set_err("adjoint scratch: device index out of range");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_err(std::string("adjoint scratch: hipGetSymbolAddress: ") + hipGetErrorString(e));
      return nullptr;
    }
    addr[device] = (double2 *)ptr;
  }
  return addr[device];
}

// Ring groups for partial sums that must fit `cap` complex entries: the
// largest power of two G <= adjoint_groups(t) with G nlpad nmaps <= cap, or
// 0 when one group does not fit.
int adjoint_groups_within(const LegTables &t, size_t cap) {
  const size_t per = (size_t)t.nlpad * (size_t)t.K;
  int G = adjoint_groups(t);
  while (G > 0 && (size_t)G * per > cap) G /= 2;
  return G;
}

// Of G ring groups, those that take the one-step units: their share of the
// instruction times (above), each unit weighed by sin(theta) (the l > m part of
// the l, m triangle that its rings reach), at least one; all where the range of
// the pair form holds no whole unit or there is one group only.  A pass of 4
// maps is what is priced: the actual passes (3 maps at 5, 6 and 9) give no better
// split (5 .. 9 maps within 2 %; Nside 300, lmax 899: 13 maps 1.42 ms so, 1.53
// with the actual ones).
static int adjoint_one_step_groups(const LegTables &t, int G) {
  const int ru = adjoint_unit(t);
  int ua, ub;
  pair_units(t, ru, &ua, &ub);
  if (G < 2 || ua >= ub) return G;
  const int units = (t.R + ru - 1) / ru, kn = std::min(t.K, 4);
  double one = 0.0, pair = 0.0;
  for (int c = 0; c < units; ++c) {
    const double z = ring_z(t.N, std::min(c * ru + ru / 2, t.R - 1)), w = std::sqrt(1.0 - z * z);
    if (c >= ua && c < ub) pair += w * (2 + 4 * kn);
    else one += w * (4 + 8 * ((kn + 1) / 2));
  }
  const int g1 = (int)std::lround(G * one / (one + pair));
  return std::max(std::max(1, G - (ub - ua)), std::min(g1, std::min(G - 1, units - (ub - ua))));
}

hipError_t launch_adjoint(const LegTables &t, const RingTables &rt, const double *map,
                          double2 *alm, double2 *partial, int G, hipStream_t s) {
  for (int i = 0; i < rt.nlaunch; ++i) {
    if (rt.count[i] == 0) continue;
    if (rt.kind[i] == kRingBelt16 && rt.fftP[i] <= 4096) {
      // the forward belt kernel's rings: the register-FFT adjoint
      const int P = rt.fftP[i], nthr = adj16_threads(P, pow2_ceil(q_group(t.K)));
      const unsigned nb = (unsigned)ring16_job_blocks(nthr / (P / 16), t.K, rt.count[i]);
      switch (P) {
#define WM_ADJ16_CASE(PP)                                                                   \
  case PP:                                                                                  \
    hipLaunchKernelGGL(k_ring_adjoint16<PP>, dim3(nb), dim3(nthr), adj16_bytes(PP, nthr), s, t,  \
                       rt, rt.first[i], rt.count[i], map);                                  \
    break;
        WM_ADJ16_SIZES(WM_ADJ16_CASE)
#undef WM_ADJ16_CASE
        default:
          return hipErrorInvalidValue;
      }
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      continue;
    }
    if (rt.kind[i] == kRingCap16 && 2 * rt.fftP[i] >= 32 && 2 * rt.fftP[i] <= 8192) {
      // the cap kernel's rings: Bluestein of length P = 2 P2 on the register FFT
      const int P = 2 * rt.fftP[i], nthr = adj16_threads(P, 1);
      const unsigned nb = (unsigned)ring16_job_blocks(nthr / (P / 16), t.K, rt.count[i]);
      switch (P) {
#define WM_ADJCAP_CASE(PP)                                                                  \
  case PP:                                                                                  \
    hipLaunchKernelGGL(k_ring_adjoint_cap16<PP>, dim3(nb), dim3(nthr), adj16_bytes(PP, nthr), s, \
                       t, rt, rt.first[i], rt.count[i], map);                               \
    break;
        WM_ADJ_CAP_SIZES(WM_ADJCAP_CASE)
#undef WM_ADJCAP_CASE
        default:
          return hipErrorInvalidValue;
      }
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      continue;
    }
    // every pair of the group fits: adj_lds[i] >= ring_lds_slots of each
    const size_t lds = (size_t)rt.adj_lds[i] * sizeof(double2);
    switch (rt.adj_maxp) {
#define WM_RADJ(MP)                                                                         \
  case MP:                                                                                  \
    hipLaunchKernelGGL(k_ring_adjoint<MP>,                                                  \
                       dim3((unsigned)ring16_job_blocks(1, t.K, rt.count[i])), dim3(NT),    \
                       lds, s, t, rt, rt.first[i], rt.count[i], rt.adj_lds[i], map);        \
    break;
      WM_RADJ(1024) WM_RADJ(2048) WM_RADJ(4096) WM_RADJ(8192)
#undef WM_RADJ
      default:
        return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const int G1 = adjoint_one_step_groups(t, G);
  const unsigned nblk = (unsigned)((t.M + 64) / 64 * 64 * G);
  // passes of up to 4 maps: 8 in one pass leave registers for half the rings
  // only, and with them twice the partial sums to read and write (Nside 1024,
  // 8 maps: 4.2 ms in one pass, 3.6 in two)
  const int passes = (t.K + 3) / 4, per = (t.K + passes - 1) / passes;
  for (int kb = 0; kb < t.K; kb += per) {
    const int kn = std::min(per, t.K - kb);
    const bool big = adjoint_unit(t) == 128;
#define WM_ADJ(KN, GR)                                                                    \
  hipLaunchKernelGGL((k_legendre_adj<KN, GR>), dim3(nblk), dim3(64), 0, s, t, G, G1, kb,  \
                     partial)
    switch (kn) {
      case 1: if (big) WM_ADJ(1, 8); else WM_ADJ(1, 4); break;
      case 2: if (big) WM_ADJ(2, 8); else WM_ADJ(2, 4); break;
      case 3: if (big) WM_ADJ(3, 8); else WM_ADJ(3, 4); break;
      default: if (big) WM_ADJ(4, 8); else WM_ADJ(4, 4);
    }
#undef WM_ADJ
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_adj_finish, dim3((unsigned)((t.nlpad * t.K + 255) / 256)), dim3(256), 0,
                     s, t, G, G1, partial, alm);
  return hipGetLastError();
}

hipError_t adjoint_set_lds_limit(int slots) {
  // The limit only grows, so plans made earlier keep a valid launch size.
  static std::mutex mu;
  static int cur = 0;
  std::lock_guard<std::mutex> lock(mu);
  if (slots <= cur) return hipSuccess;
  hipError_t e = hipSuccess;
  for (const void *f : {(const void *)k_ring_adjoint<1024>, (const void *)k_ring_adjoint<2048>,
                        (const void *)k_ring_adjoint<4096>, (const void *)k_ring_adjoint<8192>})
    if (e == hipSuccess)
      e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)((size_t)slots * sizeof(double2)));
  // the register-FFT adjoint's fixed sizes (set once; they do not grow)
#define WM_ADJ16_SET(PP)                                                                    \
  if (e == hipSuccess)                                                                      \
    e = hipFuncSetAttribute((const void *)k_ring_adjoint16<PP>,                             \
                            hipFuncAttributeMaxDynamicSharedMemorySize,             \
                            (int)adj16_bytes(PP, kAdjRB));
  WM_ADJ16_SIZES(WM_ADJ16_SET)
#undef WM_ADJ16_SET
#define WM_ADJCAP_SET(PP)                                                                   \
  if (e == hipSuccess)                                                                      \
    e = hipFuncSetAttribute((const void *)k_ring_adjoint_cap16<PP>,                         \
                            hipFuncAttributeMaxDynamicSharedMemorySize,             \
                            (int)adj16_bytes(PP, kAdjRB));
  WM_ADJ_CAP_SIZES(WM_ADJCAP_SET)
#undef WM_ADJCAP_SET
  if (e == hipSuccess) cur = slots;
  return e;
}

}  // namespace wm
