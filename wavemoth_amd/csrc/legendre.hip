// Legendre stage of the a_lm -> map synthesis on gfx950, in FP64.
//
// For every (m, ring pair r) the engine needs the even and odd partial sums
//   E[r][m] = sum_{l-m even} Lambda_l^m(x_r) a_lm,
//   O[r][m] = sum_{l-m odd}  Lambda_l^m(x_r) a_lm,
// which the reference computes per (m, parity) with the x^2 two-step
// recurrence from stored seeds (src/legendre_transform.c.in:680-747,
// src/wavemoth.c:958-1028) and keeps in work_q[m][odd][ring].
//
// Here Lambda is generated on the fly with the one-step recurrence written
// in monic form.  With Lambda_{l+1} = a_l x Lambda_l - b_l Lambda_{l-1}
// (the normalised recurrence of libpshtlight/ylmgen_c.c:604-619, 643-732)
// and Lambda_l = A_l L~_l, A_{l+1} = a_l A_l, the scaled values obey
//   L~_{l+1} = x L~_l - c~_l L~_{l-1},   c~_l = (l^2 - m^2) / (4 l^2 - 1),
// i.e. one multiply and one FMA per (l, ring) instead of three operations.
// A_l is reset to 1 at the start of every kChunk-long l-chunk; the state
// is multiplied by the chunk's end product once per chunk and the
// contraction uses a~_lm = A_l a_lm, prescaled once per execute.
// Both parities come out of the same sweep (odd and even l alternate).
//
// Seeds: Lambda_mm = (-1)^m sqrt(prod (2i+1)/(2i)) / sqrt(4 pi) sin^m theta
// underflows FP64 for large m near the poles, so the seed kernel carries a
// separate binary exponent, runs the recurrence through the negligible
// region and records, per (m, ring), the chunk-aligned l where |Lambda|
// first reaches 2^-107 together with the two recurrence states there.  This
// is the GPU form of Ylmgen's firstl and the reference's stripify start
// rows (wavemoth/lib.pyx:301-368, 397-487); terms skipped before that
// point are below 1e-32 in magnitude.
#include "wm_host.h"

namespace wm {

// Up to this many maps the sweep's contraction runs on the vector units.
constexpr int kMapsVector = 3;

// -------------------------------------------------------------- seeds

// One thread per (m, ring).  Writes seed_l / seed_v.
__global__ __launch_bounds__(256) void k_seeds(LegTables t) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int R = t.R, L = t.L;
  if (gid >= (int64_t)(t.M + 1) * R) return;
  const int m = (int)(gid / R), r = (int)(gid - (int64_t)m * R);
  const double x = t.ring_x[r];

  // log2 |Lambda_mm| = mfac[m] + m log2 sin(theta), in double-double so
  // the seed is good to ~1 ulp even when the exponent is ~ -10^4.
  const double2 mf = t.mfac[m];
  const double2 ls = t.ring_ls[r];
  const double dm = (double)m;
  double p = dm * ls.x;
  double pe = fma(dm, ls.x, -p) + dm * ls.y;
  double hi = mf.x + p;
  double bb = hi - mf.x;
  double lo = (mf.x - (hi - bb)) + (p - bb) + mf.y + pe;
  double E = floor(hi);
  double frac = (hi - E) + lo;
  if (frac >= 1.0) { E += 1.0; frac -= 1.0; }
  if (frac < 0.0) { E -= 1.0; frac += 1.0; }
  int iE = (int)E;
  double cur = exp2(frac);
  if (m & 1) cur = -cur;
  double prev = 0.0;

  const int64_t offm = t.off[m];
  const double *ct = t.ctil + (offm - m);
  const double *cs = t.cscale + offm / kChunk;
  int found = kSeedNone;
  double sp = 0.0, sc = 0.0;
  int c = 0;
  for (int l0 = m; l0 <= L; l0 += kChunk, ++c) {
    const double cp = prev, cc = cur;
    const int cE = iE;
#pragma unroll
    for (int j = 0; j < kChunk; ++j) {
      const double nx = fma(x, cur, -ct[l0 + j] * prev);
      prev = cur;
      cur = nx;
    }
    const double S = cs[c];
    prev *= S;
    cur *= S;
    const double big = fmax(fabs(prev), fabs(cur));
    if (!(big > 0.0)) break;
    const int e = ilogb(big);
    if (e + iE >= -107) {
      found = l0;
      sp = ldexp(cp, cE);
      sc = ldexp(cc, cE);
      break;
    }
    prev = ldexp(prev, -e);
    cur = ldexp(cur, -e);
    iE += e;
  }
  t.seed_l[gid] = found;
  t.seed_v[gid] = make_double2(sp, sc);
}

// One thread per (m, wave): the wave-uniform first l and the last l at
// which some lane of the wave still has to pick up its seed.
__global__ __launch_bounds__(256) void k_wave_bounds(LegTables t) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (int64_t)(t.M + 1) * t.W) return;
  const int m = (int)(gid / t.W), w = (int)(gid - (int64_t)m * t.W);
  int lo = kSeedNone, hi = -1;
  const int rings = 64 * t.RL;
  for (int i = 0; i < rings; ++i) {
    const int r = w * rings + i;
    if (r >= t.R) break;
    const int s = t.seed_l[(int64_t)m * t.R + r];
    if (s < lo) lo = s;
    if (s <= t.L && s > hi) hi = s;
  }
  t.wstart[gid] = lo;
  t.wseedmax[gid] = hi;
}

// The first l of each (m, chunk of kSegRings rings) and the recurrence
// states (L~_{l-1}, L~_l) of its rings at the starts of l-segments 1 .. 3
// (zero before a ring's seed), with the same steps and chunk rescale as the
// sweep: ckpt[(3 m + s - 1) R + r].  A segment is ns = ceil(nc / 4) of the nc
// l-chunks from the first one.  One block per (m, chunk), a thread per ring.
__global__ __launch_bounds__(kSegRings) void k_checkpoints(LegTables t) {
  __shared__ int wmin[kSegRings / 64];
  const int m = blockIdx.x / t.SW, sc = blockIdx.x - m * t.SW;
  const int r = sc * kSegRings + threadIdx.x, R = t.R, L = t.L;
  const int sl = r < R ? t.seed_l[(int64_t)m * R + r] : kSeedNone;
  int lo = sl;
  for (int d = 32; d >= 1; d >>= 1) {
    const int o = __shfl_xor(lo, d);
    lo = o < lo ? o : lo;
  }
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = lo;
  __syncthreads();
  int l0 = wmin[0];
  for (int i = 1; i < kSegRings / 64; ++i) l0 = wmin[i] < l0 ? wmin[i] : l0;
  l0 = __builtin_amdgcn_readfirstlane(l0);
  if (threadIdx.x == 0) t.seg_l0[blockIdx.x] = l0;
  if (l0 > L) return;
  const int nc = (L - l0) / kChunk + 1, ns = (nc + 3) / 4;
  const int64_t offm = t.off[m];
  const double *ct = t.ctil + (offm - m), *cs = t.cscale + (offm + l0 - m) / kChunk;
  const double x = r < R ? t.ring_x[r] : 0.0;
  const double2 sv = sl <= L ? t.seed_v[(int64_t)m * R + r] : make_double2(0.0, 0.0);
  double prev = 0.0, cur = 0.0;
  for (int s = 1; s <= 3 && s * ns < nc; ++s) {
    for (int ch = (s - 1) * ns; ch < s * ns; ++ch) {
      const int l = l0 + kChunk * ch;
      if (sl == l) {
        prev = sv.x;
        cur = sv.y;
      }
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        const double nx = fma(x, cur, -(ct[l + j] * prev));
        prev = cur;
        cur = nx;
      }
      prev *= cs[ch];
      cur *= cs[ch];
    }
    if (r < R) t.ckpt[((int64_t)m * 3 + s - 1) * R + r] = make_double2(prev, cur);
  }
}

// ----------------------------------------------------------- pair form
//
// With A_l^2 = (l^2 - m^2) / (4 l^2 - 1), x Lambda_l = A_{l+1} Lambda_{l+1} +
// A_l Lambda_{l-1}.  Take P_k = Lambda_{l+1} / x at l = m + 2 k.  Then
//   Lambda_{l+1} = x P_k,   Lambda_l = A_{l+1} P_k + A_l P_{k-1},
// and, applying the relation twice,
//   A_{l+2} A_{l+3} P_{k+1} = (x^2 - A_{l+1}^2 - A_{l+2}^2) P_k - A_l A_{l+1} P_{k-1}:
// one value serves two l.  (K. Ishioka, J. Meteorol. Soc. Japan 96, 2018,
// computes the transform with such a function.)  Scaled, P_k = s_k p_k with
// s_{k+1} / s_{k-1} = A_l A_{l+1} / (A_{l+2} A_{l+3}), s_0 = s_1 = 1:
//   p_{k+1} = (alpha_k y + beta_k) p_k - p_{k-1},
// two FMAs per two l where the one-step form has four operations.  The rounding
// of y shifts the angle of all steps alike, so y is x^2 less the middle of its
// zone of latitude, one rounding of a small number, and beta_k differs by zone.
// (With y = x^2 or x^2 - 1 the error of E and O is 1.2 .. 1.5 times the one-step
// form's, with five zones 0.9.)
//
// The tables, one wave per m: s_k is a product of k ratios, so all of it is
// computed in double-double and rounded once.
// No contraction here: a product fused into one use of it and rounded in
// another would count its rounding error twice.
#pragma clang fp contract(off)
__device__ __forceinline__ double2 dd_quick(double a, double b) {
  const double s = a + b;
  return make_double2(s, b - (s - a));
}
__device__ __forceinline__ double2 dd_sum(double a, double b) {
  const double s = a + b, t = s - a;
  return make_double2(s, (a - (s - t)) + (b - t));
}
__device__ __forceinline__ double2 dd_add(double2 a, double2 b) {
  const double2 s = dd_sum(a.x, b.x);
  return dd_quick(s.x, s.y + a.y + b.y);
}
__device__ __forceinline__ double2 dd_mul(double2 a, double2 b) {
  const double p = a.x * b.x;
  return dd_quick(p, fma(a.x, b.x, -p) + (a.x * b.y + a.y * b.x));
}
__device__ __forceinline__ double2 dd_div(double2 a, double2 b) {
  const double q = a.x / b.x;
  const double r = fma(-q, b.x, a.x) + (a.y - q * b.y);
  return dd_quick(q, r / b.x);
}
__device__ __forceinline__ double2 dd_sqrt(double2 a) {
  const double s = sqrt(a.x);
  return dd_quick(s, (fma(-s, s, a.x) + a.y) / (2.0 * s));
}
// A_l^2; both products are exact
__device__ __forceinline__ double2 dd_a2(double l, double m) {
  return dd_div(make_double2((l - m) * (l + m), 0.0),
                make_double2((2.0 * l - 1.0) * (2.0 * l + 1.0), 0.0));
}

// s_{k+1}^2 / s_{k-1}^2 of every second k multiply up; a lane takes a run of k,
// and the products of the runs before it come by a scan over the wave.
__global__ __launch_bounds__(64) void k_pair_tables(LegTables t) {
  const int m = blockIdx.x, lane = threadIdx.x;
  const double dm = (double)m;
  const int64_t o = t.off[m] / 2;
  const int n = (t.L - m + kChunk) / kChunk * (kChunk / 2);
  const int len = (n + 127) / 128 * 2;
  const int ka = lane * len < n ? lane * len : n, ke = ka + len < n ? ka + len : n;
  const double2 one = make_double2(1.0, 0.0);
  const double la = dm + 2.0 * (double)ka;
  double2 tp = one, tk = one;  // products of even, of odd k
  {
    double2 g0 = dd_mul(dd_a2(la, dm), dd_a2(la + 1.0, dm));
    for (int k = ka; k < ke; ++k) {
      const double l = dm + 2.0 * (double)k;
      const double2 g1 = dd_mul(dd_a2(l + 2.0, dm), dd_a2(l + 3.0, dm));
      const double2 r = k == 0 ? one : dd_div(g0, g1);
      if (k & 1) tk = dd_mul(tk, r);
      else tp = dd_mul(tp, r);
      g0 = g1;
    }
  }
  for (int d = 1; d <= 32; d *= 2) {
    const double2 p = make_double2(__shfl_up(tp.x, d), __shfl_up(tp.y, d));
    const double2 q = make_double2(__shfl_up(tk.x, d), __shfl_up(tk.y, d));
    if (lane >= d) {
      tp = dd_mul(tp, p);
      tk = dd_mul(tk, q);
    }
  }
  tp = make_double2(__shfl_up(tp.x, 1), __shfl_up(tp.y, 1));
  tk = make_double2(__shfl_up(tk.x, 1), __shfl_up(tk.y, 1));
  if (lane == 0) tp = tk = one;
  // tp = s_{k-1}^2, tk = s_k^2
  double2 c0 = dd_a2(la, dm), c1 = dd_a2(la + 1.0, dm);  // A_l^2, A_{l+1}^2
  for (int k = ka; k < ke; ++k) {
    const double l = dm + 2.0 * (double)k;
    const double2 c2 = dd_a2(l + 2.0, dm), c3 = dd_a2(l + 3.0, dm);
    const double2 g1 = dd_mul(c2, c3);
    const double2 tn = k == 0 ? one : dd_mul(tp, dd_div(dd_mul(c0, c1), g1));
    const double2 al = dd_sqrt(dd_div(tk, dd_mul(tn, g1)));
    const double2 u = dd_add(c1, c2);
    for (int z = 0; z < kPairZones; ++z) {
      const double2 d = dd_add(make_double2(pair_centre(z), 0.0), make_double2(-u.x, -u.y));
      t.pair_t[t.nlpad / 2 * z + o + k] = make_double2(al.x, dd_mul(al, d).x);
    }
    t.pair_w[o + k] = dd_sqrt(tk).x;
    if (k % (kChunk / 2) == 0)
      // L~_{l+1} = A_{l+1} Lambda_{l+1} and L~_{l-1} = Lambda_{l-1} / A_l there
      t.pair_h[(o + k) / (kChunk / 2)] = make_double2(
          dd_sqrt(dd_div(one, dd_mul(c1, tk))).x, k == 0 ? 0.0 : dd_sqrt(dd_div(c0, tp)).x);
    tp = tk;
    tk = tn;
    c0 = c2;
    c1 = c3;
  }
}
#pragma clang fp contract(fast)

// ------------------------------------------------------- a_lm prescale

// map slots of atil: nmaps rounded up to whole blocks of KB
__host__ __device__ inline int legendre_padded_maps_of(int K, int KB) {
  return (K + KB - 1) / KB * KB;
}

// atil[kb][j][k'] = A_l * a_{l m}[kb*KB + k'] on the padded l-grid, zero
// past lmax and for map slots past nmaps: map-block-major so that a wave
// of map block kb reads KB consecutive complex values per l.  One entry:
// padded l-entry j, map slot kk < KB nkb.
__device__ __forceinline__ void prep_entry(const LegTables &t, const double2 *__restrict__ alm,
                                           int64_t j, int kk, int KB) {
  const int K = t.K, L = t.L;
  const int m = t.chunk_m[j / kChunk];
  const int64_t jj = j - t.off[m];
  const int l = m + (int)jj;
  const bool live = l <= L && kk < K;
  const double sc = t.ascale[j];
  const int64_t idx = (int64_t)m * (2 * L - m + 3) / 2 + (l <= L ? jj : 0);
  const double2 a = alm[idx * K + (kk < K ? kk : K - 1)];
  const int kb = kk / KB;
  t.atil[((int64_t)kb * t.nlpad + j) * KB + (kk - kb * KB)] =
      live ? make_double2(a.x * sc, a.y * sc) : make_double2(0.0, 0.0);
  if (t.ptil) {
    // the coefficients of p_k in E and of x p_k in O (pair form): s_k (A_{l+1}
    // a_l + A_{l+2} a_{l+2}) and s_k a_{l+1}, side by side
    double2 v = make_double2(0.0, 0.0);
    if (live) {
      const double w = t.pair_w[j / 2];
      if (jj & 1) {
        v = make_double2(w * a.x, w * a.y);
      } else {
        const double f = w * sqrt(t.ctil[j + 1]);
        v = make_double2(f * a.x, f * a.y);
        if (l + 2 <= L) {  // then the padded range has l + 2
          const double h = w * sqrt(t.ctil[j + 2]);
          const double2 b = alm[(idx + 2) * K + kk];
          v = make_double2(fma(h, b.x, v.x), fma(h, b.y, v.y));
        }
      }
    }
    t.ptil[((int64_t)kb * t.nlpad + (j - (jj & 1))) * KB + 2 * (kk - kb * KB) + (jj & 1)] = v;
  }
}

// The single-plan prescale: one thread per (padded l-entry j, map slot kk),
// maps fastest, so that a wave reads the consecutive a_lm of one l (and of
// JB = 256 / Kp consecutive l) and writes KB-map runs of atil.
__global__ __launch_bounds__(256) void k_prep_alm(LegTables t, const double2 *__restrict__ alm,
                                                  int KB, int nkb) {
  const int Kp = KB * nkb;
  const int JB = Kp >= 256 ? 1 : 256 / Kp;
  const int64_t j0 = (int64_t)blockIdx.x * JB;
  for (int u = threadIdx.x; u < JB * Kp; u += blockDim.x) {
    const int jl = u / Kp, kk = u - jl * Kp;
    const int64_t j = j0 + jl;
    if (j >= t.nlpad) break;  // jl only grows with u
    prep_entry(t, alm, j, kk, KB);
  }
}

// One wave's share of the sweep: ring chunk w (rings w*64*RL + lane + 64*i,
// i < RL) of m, maps kb*KB .. kb*KB+KB-1.  Used by the grid kernel below
// and by the batched work-queue kernel (batch.hip).
// Tables the sweep only reads are accessed through constant-address-space
// views: their loads are then known not to be clobbered by the q stores
// (which matters inside the persistent loop of the batched kernel), and
// wave-uniform ones go through the scalar unit.
#define WM_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const WM_CONST T *const_view(const T *p) {
  return (const WM_CONST T *)p;
}

// Brings the coefficient rows of a later chunk into the XCD's L2.  A scalar
// load that misses it waits for memory, all waves of an m wait with the first
// one, and the scalar registers hold one step ahead at most: a SIMD's waves
// together did not have enough arithmetic to cover that (vector units busy 65
// .. 78 % of the time; one-step sweep at lmax 4096, 1 map without / with this
// 3.96 / 3.75 ms, lmax 2048 0.576 / 0.541, lmax 1024, 3 maps 0.191 / 0.175).
// Lane 0 touches the chunk's line of c~_l (or alpha_k, beta_k), lane 1 + i line
// i of its a~ rows; take() marks where the value has long arrived.
template <int KB>
struct RowTouch {
  const double *p;
  unsigned stride;  // doubles per chunk
  double v;
  __device__ __forceinline__ RowTouch(const double *c, const double *a, int lane) {
    const int line = lane < 2 * KB ? lane : 2 * KB;
    p = line == 0 ? c : a + 16 * (line - 1);
    stride = line == 0 ? kChunk : 2 * KB * kChunk;
    v = 0.0;
  }
  __device__ __forceinline__ void touch(int chunk) { v = p[(unsigned)chunk * stride]; }
  __device__ __forceinline__ void take() { asm volatile("" ::"v"(v)); }
};
constexpr int kTouchAhead = 1;  // chunks: a chunk takes longer than memory; 2 and 4 are no better

// The sweep of up to 3 maps on the vector units: 2 + 2 KB FP64 instructions
// per (l, ring), their coefficients (c~_l and KB complex a~_l) wave-uniform
// SGPR operands.  The scalar loads of a step of ST l are issued one step
// ahead: scalar loads return out of order, so a wait for one is a wait for
// all, and a step that loads what it uses itself stalls for the whole L2
// latency.  The empty asm marks where the step's own values must have
// arrived; the next step's loads follow it and have the step's arithmetic
// (ST RL (2 + 2 KB) instructions) to arrive.
template <int RL, int KB>
__device__ __forceinline__ void legendre_sweep(
    int L, int R, int Mp1, int K, int m, int w, int kbase, int lane, int l0, int lsmax,
    const WM_CONST double *ct, const WM_CONST double *at,
    const WM_CONST double *cs, const double *__restrict__ ring_x,
    const int *__restrict__ seed_l, const double2 *__restrict__ seed_v,
    double2 *__restrict__ qbuf) {
  constexpr int ST = KB <= 2 ? 4 : 2;  // l per step: both steps' values fit the SGPRs
  double x[RL], prev[RL], cur[RL];
  double2 sv[RL];
  int sl[RL], rr[RL];
  double acc[RL][2][KB][2];
#pragma unroll
  for (int i = 0; i < RL; ++i) {
    rr[i] = w * 64 * RL + lane + 64 * i;
    const bool ok = rr[i] < R;
    x[i] = ok ? ring_x[rr[i]] : 0.0;
    sl[i] = ok ? seed_l[(int64_t)m * R + rr[i]] : kSeedNone;
    sv[i] = ok ? seed_v[(int64_t)m * R + rr[i]] : make_double2(0.0, 0.0);
    prev[i] = 0.0;
    cur[i] = 0.0;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int k = 0; k < KB; ++k) acc[i][p][k][0] = acc[i][p][k][1] = 0.0;
  }

  if (l0 <= L) {
    double c[ST], a[ST][2 * KB], S;
    const int last = m + (L - m) / kChunk * kChunk + kChunk - ST;  // start of the last step
#pragma unroll
    for (int j = 0; j < ST; ++j) {
      c[j] = ct[l0 + j];
#pragma unroll
      for (int u = 0; u < 2 * KB; ++u) a[j][u] = at[2 * (int64_t)KB * (l0 + j) + u];
    }
    S = cs[(l0 - m) / kChunk];
    RowTouch<KB> ahead((const double *)ct + m, (const double *)at + 2 * KB * (int64_t)m, lane);
    const int lastc = (L - m) / kChunk;
    for (; l0 <= L; l0 += kChunk) {
      const int far = (l0 - m) / kChunk + kTouchAhead;
      ahead.take();
      ahead.touch(far < lastc ? far : lastc);
      if (l0 <= lsmax) {
#pragma unroll
        for (int i = 0; i < RL; ++i) {
          prev[i] = sl[i] == l0 ? sv[i].x : prev[i];
          cur[i] = sl[i] == l0 ? sv[i].y : cur[i];
        }
      }
      double Sn = S;
#pragma unroll
      for (int j0 = 0; j0 < kChunk; j0 += ST) {
        const int ln = l0 + j0 < last ? l0 + j0 + ST : last;
        asm volatile("" ::"s"(a[ST - 1][2 * KB - 1]), "s"(c[ST - 1]), "s"(S));
        __builtin_amdgcn_sched_barrier(0);
        double cn[ST], an[ST][2 * KB];
#pragma unroll
        for (int j = 0; j < ST; ++j) {
          cn[j] = ct[ln + j];
#pragma unroll
          for (int u = 0; u < 2 * KB; ++u) an[j][u] = at[2 * (int64_t)KB * (ln + j) + u];
        }
        if (j0 == kChunk - ST) Sn = cs[(ln - m) / kChunk];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < RL; ++i) {
#pragma unroll
          for (int j = 0; j < ST; ++j) {
#pragma unroll
            for (int k = 0; k < KB; ++k) {
              acc[i][j & 1][k][0] = fma(cur[i], a[j][2 * k], acc[i][j & 1][k][0]);
              acc[i][j & 1][k][1] = fma(cur[i], a[j][2 * k + 1], acc[i][j & 1][k][1]);
            }
            const double nx = fma(x[i], cur[i], -(c[j] * prev[i]));
            prev[i] = cur[i];
            cur[i] = nx;
          }
          if (j0 == kChunk - ST) {
            prev[i] *= S;
            cur[i] *= S;
          }
        }
#pragma unroll
        for (int j = 0; j < ST; ++j) {
          c[j] = cn[j];
#pragma unroll
          for (int u = 0; u < 2 * KB; ++u) a[j][u] = an[j][u];
        }
      }
      S = Sn;
    }
  }

#pragma unroll
  for (int i = 0; i < RL; ++i) {
    if (rr[i] < R) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int k = 0; k < KB; ++k)
          if (kbase + k < K)
            qbuf[q_index(rr[i], p, kbase + k, m, K, Mp1)] =
                make_double2(acc[i][p][k][0], acc[i][p][k][1]);
      }
    }
  }
}

// The same in the pair form: 2 + 4 KB FP64 instructions per two l and ring
// where the one-step form has 4 + 4 KB, and one move of beta_k for all rings
// of a lane (a vector instruction reads one scalar operand).  Bound by the
// vector units: 2.6 ms of 3.4 at lmax 4096, 1 map, where the one-step form
// takes 3.75; lmax 2048, 2 maps 0.74 / 0.79 ms, lmax 4096, 3 maps 6.6 / 7.2.  pc:
// (alpha_k, beta_k), at: the KB (E, O) coefficient pairs of p_k.
template <int RL, int KB>
__device__ __forceinline__ void legendre_pair_sweep(
    const LegTables &t, int m, int w, int kbase, int lane, int l0, int lsmax,
    const WM_CONST double *pc, const WM_CONST double *at, int zone) {
  constexpr int ST = KB <= 2 ? 2 : 1, KC = kChunk / 2;
  const int L = t.L, K = t.K;
  double y[RL], prev[RL], cur[RL];
  double2 sv[RL];
  int sl[RL];
  double acc[RL][2][KB][2];
#pragma unroll
  for (int i = 0; i < RL; ++i) {
    const int r = w * 64 * RL + lane + 64 * i;
    const double x = t.ring_x[r];
    y[i] = fma(x, x, -pair_centre(zone));
    sl[i] = t.seed_l[(int64_t)m * t.R + r];
    sv[i] = make_double2(0.0, 0.0);
    if (sl[i] <= L) {
      // (L~_{l-1}, L~_l) -> (p_{k-1}, p_k)
      const double2 v = t.seed_v[(int64_t)m * t.R + r];
      const int64_t j = t.off[m] + sl[i] - m;
      const double2 h = t.pair_h[j / kChunk];
      const double rx = 1.0 / x;
      sv[i] = make_double2(v.x * h.y * rx, fma(x, v.y, -(t.ctil[j] * v.x)) * h.x * rx);
    }
    prev[i] = 0.0;
    cur[i] = 0.0;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int k = 0; k < KB; ++k) acc[i][p][k][0] = acc[i][p][k][1] = 0.0;
  }

  if (l0 <= L) {
    double al[ST], be[ST], a[ST][4 * KB];
    const int last = ((L - m) / kChunk + 1) * KC - ST;  // start of the last step
    int k0 = (l0 - m) / 2;
#pragma unroll
    for (int j = 0; j < ST; ++j) {
      al[j] = pc[2 * (k0 + j)];
      be[j] = pc[2 * (k0 + j) + 1];
#pragma unroll
      for (int u = 0; u < 4 * KB; ++u) a[j][u] = at[4 * (int64_t)KB * (k0 + j) + u];
    }
    RowTouch<KB> ahead((const double *)pc, (const double *)at, lane);
    const int lastc = (L - m) / kChunk;
    for (; l0 <= L; l0 += kChunk) {
      const int far = (l0 - m) / kChunk + kTouchAhead;
      ahead.take();
      ahead.touch(far < lastc ? far : lastc);
      if (l0 <= lsmax) {
#pragma unroll
        for (int i = 0; i < RL; ++i) {
          prev[i] = sl[i] == l0 ? sv[i].x : prev[i];
          cur[i] = sl[i] == l0 ? sv[i].y : cur[i];
        }
      }
#pragma unroll
      for (int s0 = 0; s0 < KC; s0 += ST) {
        k0 = k0 < last ? k0 + ST : last;
        asm volatile("" ::"s"(a[ST - 1][4 * KB - 1]), "s"(al[ST - 1]), "s"(be[ST - 1]));
        __builtin_amdgcn_sched_barrier(0);
        double aln[ST], ben[ST], an[ST][4 * KB];
#pragma unroll
        for (int j = 0; j < ST; ++j) {
          aln[j] = pc[2 * (k0 + j)];
          ben[j] = pc[2 * (k0 + j) + 1];
#pragma unroll
          for (int u = 0; u < 4 * KB; ++u) an[j][u] = at[4 * (int64_t)KB * (k0 + j) + u];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < ST; ++j) {
#pragma unroll
          for (int i = 0; i < RL; ++i) {
#pragma unroll
            for (int k = 0; k < KB; ++k)
#pragma unroll
              for (int u = 0; u < 4; ++u)
                acc[i][u >> 1][k][u & 1] =
                    fma(cur[i], a[j][4 * k + u], acc[i][u >> 1][k][u & 1]);
            const double nx = fma(fma(al[j], y[i], be[j]), cur[i], -prev[i]);
            prev[i] = cur[i];
            cur[i] = nx;
          }
        }
#pragma unroll
        for (int j = 0; j < ST; ++j) {
          al[j] = aln[j];
          be[j] = ben[j];
#pragma unroll
          for (int u = 0; u < 4 * KB; ++u) a[j][u] = an[j][u];
        }
      }
    }
  }

#pragma unroll
  for (int i = 0; i < RL; ++i) {
    const int r = w * 64 * RL + lane + 64 * i;
    const double x = t.ring_x[r];
#pragma unroll
    for (int k = 0; k < KB; ++k)
      if (kbase + k < K) {
        t.qbuf[q_index(r, 0, kbase + k, m, K, t.M + 1)] =
            make_double2(acc[i][0][k][0], acc[i][0][k][1]);
        t.qbuf[q_index(r, 1, kbase + k, m, K, t.M + 1)] =
            make_double2(x * acc[i][1][k][0], x * acc[i][1][k][1]);
      }
  }
}

typedef double leg_d4 __attribute__((ext_vector_type(4)));

// Seeds of a wave's rings in LDS (matrix-core sweep).
__host__ __device__ constexpr int sweep_lds(int RL, int KB) {
  return KB > kMapsVector ? 64 * RL : 1;
}

// The sweep of KB maps (even, 2 .. 16) with the contraction on the FP64
// matrix cores.  The chunk's l-range is cut into four segments and the four
// 16-lane rows of the wave step one segment each, all for the same rings:
// lane 16 g + i holds Lambda_{l_g}(ring 16 j + i), l_g = step s of segment g,
// which is the A operand of a product of 16 rings x 4 l as it stands
// (a product only needs A and B to agree on the l of each k).  Columns are
// the real and imaginary parts of the pass's maps: v_mfma_f64_16x16x4f64 for
// every 8 maps, v_mfma_f64_4x4x4f64 (4 blocks of 4 rings, the same 4 columns)
// for every further 2.  Segments 1 .. 3 start from checkpoints of the
// recurrence (k_checkpoints), made once per geometry.
//
// Why so: an FP64 matrix instruction keeps its SIMD's whole vector unit busy
// (measured: any vector instruction of another wave adds to its time), so
// the time is the sum 4 RL (2 + 2) FP64 instructions of the recurrence and
// 4 RL KB / 2 quarter products per step, and nothing may be added to it.  A
// wave that steps one l-range per lane has to transpose Lambda first: 16
// lane swaps per 8 l and 64 rings (8.5 cycles each, +30 % at 16 maps) or an
// LDS round trip (LDS-bound below 8 maps).  The coefficients and the a~ rows
// differ by segment and come by vector loads, four steps ahead; in order,
// unlike scalar loads.
template <int RL, int KB>
__device__ __forceinline__ void legendre_sweep_mm(
    int L, int R, int Mp1, int K, int m, int w, int kbase, int lane, int l0,
    const double *__restrict__ ct, const double *__restrict__ at,
    const double *__restrict__ cs, const double *__restrict__ ring_x,
    const int *__restrict__ seed_l, const double2 *__restrict__ seed_v,
    const double2 *__restrict__ ckpt, double2 *__restrict__ qbuf, double2 *seeds) {
  constexpr int GR = 4 * RL;                      // 16-ring groups
  constexpr int C16 = KB / 8, C4 = (KB % 8) / 2;  // 16-column tiles, 4-column groups
  constexpr int B16 = C16 > 0 ? C16 : 1, B4 = C4 > 0 ? C4 : 1;
  constexpr int ST = KB <= 6 ? 4 : 2;             // steps per load block
  const int kq = lane >> 4, col = lane & 15, rbase = w * 64 * RL + col;
  double x[GR], prev[GR], cur[GR];
  int sl[GR];
  leg_d4 acc16[GR][2][B16];
  double acc4[GR][2][B4];
#pragma unroll
  for (int i = 0; i < GR; ++i)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int c = 0; c < B16; ++c) acc16[i][p][c] = leg_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int c = 0; c < B4; ++c) acc4[i][p][c] = 0.0;
    }

  if (l0 <= L) {
    const int nc = (L - l0) / kChunk + 1, ns = (nc + 3) / 4;  // chunks, chunks per segment
    const int cb = kq * ns;                                   // the lane's first chunk
    // the rings' seeds wait in LDS: a load where a ring joins would stall the wave
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const int r = w * 64 * RL + 64 * i + lane;
      if (r < R) seeds[64 * i + lane] = seed_v[(int64_t)m * R + r];
    }
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      const int r = rbase + 16 * i;
      const bool ok = r < R;
      x[i] = ok ? ring_x[r] : 0.0;
      sl[i] = ok ? seed_l[(int64_t)m * R + r] : kSeedNone;
      double2 v = make_double2(0.0, 0.0);
      if (ok && kq > 0 && cb < nc) v = ckpt[((int64_t)m * 3 + kq - 1) * R + r];
      prev[i] = v.x;
      cur[i] = v.y;
    }
    ct += l0;
    at += 2 * (int64_t)KB * l0;
    cs += (l0 - m) / kChunk;
    // row e of the lane's segment: c~ at ct[e], a~ at at[2 KB e + column]
    unsigned e = kChunk * (unsigned)(cb < nc ? cb : nc - 1);
    double c[ST], S, b16[ST][B16], b4[ST][B4];
    auto load = [&](unsigned el, double (&cc)[ST], double (&v16)[ST][B16], double (&v4)[ST][B4]) {
      const unsigned o16 = 2 * KB * el + col, o4 = 2 * KB * el + 16 * C16 + (lane & 3);
#pragma unroll
      for (int j = 0; j < ST; ++j) {
        cc[j] = ct[el + j];
#pragma unroll
        for (int u = 0; u < C16; ++u) v16[j][u] = at[o16 + 2 * KB * j + 16 * u];
#pragma unroll
        for (int u = 0; u < C4; ++u) v4[j][u] = at[o4 + 2 * KB * j + 4 * u];
      }
    };
    load(e, c, b16, b4);
    S = cs[e / kChunk];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int j = 0; j < ns; ++j) {
      const int ls = l0 + kChunk * (cb + j);
      bool hit = false;
#pragma unroll
      for (int i = 0; i < GR; ++i) hit |= sl[i] == ls;
      if (__any(hit)) {
#pragma unroll
        for (int i = 0; i < GR; ++i)
          if (sl[i] == ls) {
            const double2 v = seeds[16 * i + col];
            prev[i] = v.x;
            cur[i] = v.y;
          }
      }
      if (3 * ns + j >= nc && cb + j >= nc) {  // past the segment's rows
#pragma unroll
        for (int i = 0; i < GR; ++i) prev[i] = cur[i] = 0.0;
      }
      const unsigned en = kChunk * (unsigned)(cb + j + 1 < nc ? cb + j + 1 : nc - 1);
      double Sn = S;
#pragma unroll
      for (int s0 = 0; s0 < kChunk; s0 += ST) {
        double cn[ST], bn16[ST][B16], bn4[ST][B4];
        load(s0 + ST < kChunk ? e + s0 + ST : en, cn, bn16, bn4);
        if (s0 + ST == kChunk) Sn = cs[en / kChunk];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
          for (int i = 0; i < GR; ++i) {
#pragma unroll
            for (int u = 0; u < C16; ++u)
              acc16[i][s & 1][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                  cur[i], b16[s][u], acc16[i][s & 1][u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < C4; ++u)
              acc4[i][s & 1][u] = __builtin_amdgcn_mfma_f64_4x4x4f64(
                  cur[i], b4[s][u], acc4[i][s & 1][u], 0, 0, 0);
            const double nx = fma(x[i], cur[i], -(c[s] * prev[i]));
            prev[i] = cur[i];
            cur[i] = nx;
          }
#pragma unroll
        for (int s = 0; s < ST; ++s) {
          c[s] = cn[s];
#pragma unroll
          for (int u = 0; u < C16; ++u) b16[s][u] = bn16[s][u];
#pragma unroll
          for (int u = 0; u < C4; ++u) b4[s][u] = bn4[s][u];
        }
      }
#pragma unroll
      for (int i = 0; i < GR; ++i) {
        prev[i] *= S;
        cur[i] *= S;
      }
      S = Sn;
      e = en;
    }
  }

  // D of a 16-column tile: ring 16 i + kq + 4 j in register j, column col; of
  // a 4-column group: ring 16 i + 4 (col / 4) + kq, column col % 4.  Rows of
  // q (ring, parity) are `row` doubles apart.
  const int G = q_group(K);
  const int64_t row = 2 * (int64_t)q_groups(K) * Mp1 * G;
#pragma unroll
  for (int u = 0; u < C16 + C4; ++u) {
    const bool wide = u < C16;
    const int k = kbase + (wide ? 8 * u + (col >> 1) : 8 * C16 + 2 * (u - C16) + ((col & 3) >> 1));
    const int rl = w * 64 * RL + kq + (wide ? 0 : (col & 12));  // the lane's first ring
    if (k >= K) continue;
    double *q = (double *)qbuf + 2 * q_index(rl, 0, k, m, K, Mp1) + (col & 1);
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      const int ro = 16 * i;
      if (wide) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (rl + ro + 4 * j < R) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
              q[(2 * (ro + 4 * j) + p) * row] = acc16[i][p][wide ? u : 0][j];
          }
      } else if (rl + ro < R) {
#pragma unroll
        for (int p = 0; p < 2; ++p) q[(2 * ro + p) * row] = acc4[i][p][wide ? 0 : u - C16];
      }
    }
  }
}

// One wave's share of the sweep: ring chunk w (rings w*64*RL + lane + 64*i,
// i < RL) of m, maps kb*KB .. kb*KB+KB-1; wb: the entry of the wave bounds.
// Used by the grid kernel below and by the batched work-queue kernel.
template <int RL, int KB>
__device__ __forceinline__ void legendre_item(const LegTables &t, int m, int w, int kb,
                                              int wb, int lane, double2 *seeds) {
  const int64_t offm = t.off[m];
  const double *at = (const double *)(t.atil + ((int64_t)kb * t.nlpad + offm - m) * KB);
  if constexpr (KB <= kMapsVector) {
    const int l0 = __builtin_amdgcn_readfirstlane(t.wstart[(int64_t)m * t.W + wb]);
    const int lsmax = __builtin_amdgcn_readfirstlane(t.wseedmax[(int64_t)m * t.W + wb]);
    // Form and zone go by the unit of kSegRings rings: a wave of two units has
    // them in common, or takes its units in turn (sweep_items).
    if constexpr (64 * RL >= kSegRings) {
      if (t.ptil && w * 64 * RL >= t.pair_r0 && (w + 1) * 64 * RL <= t.pair_r1) {
        const int zone =
            __builtin_amdgcn_readfirstlane(pair_zone(t.ring_x[w * 64 * RL + kSegRings / 2]));
        const double2 *pc = t.pair_t + (t.nlpad * zone + offm) / 2;
        const double2 *pt = t.ptil + ((int64_t)kb * t.nlpad + offm) * KB;
        legendre_pair_sweep<RL, KB>(t, m, w, kb * KB, lane, l0, lsmax,
                                    const_view((const double *)pc),
                                    const_view((const double *)pt), zone);
        return;
      }
    }
    legendre_sweep<RL, KB>(t.L, t.R, t.M + 1, t.K, m, w, kb * KB, lane, l0, lsmax,
                           const_view(t.ctil + (offm - m)), const_view(at),
                           const_view(t.cscale + offm / kChunk), t.ring_x, t.seed_l, t.seed_v,
                           t.qbuf);
  } else {
    const int sc = w * RL * 64 / kSegRings;
    const int l0 = __builtin_amdgcn_readfirstlane(t.seg_l0[(int64_t)m * t.SW + sc]);
    legendre_sweep_mm<RL, KB>(t.L, t.R, t.M + 1, t.K, m, w, kb * KB, lane, l0,
                              t.ctil + (offm - m), at, t.cscale + offm / kChunk, t.ring_x,
                              t.seed_l, t.seed_v, t.ckpt, t.qbuf, seeds);
  }
}

// One wave per block: waves of one m run for different times (a ring near
// the pole joins late or never), and a block's slots are only refilled
// together.  Block b runs on XCD b % 8; every m's blocks are kept on one XCD
// (m = xcd + 8 * i) so the per-m coefficient rows are fetched into one L2
// only, and each XCD walks its m's from cheap-to-start (small m, long
// l-range) to short ones, within an m from the equator to the pole, the map
// blocks of a ring chunk side by side.
template <int RL, int KB>
__global__ __launch_bounds__(64) void k_legendre(LegTables t, int nkb, int bpm) {
  const int b = blockIdx.x;
  const int s = b >> 3;
  const int m = (b & 7) + 8 * (s / bpm);
  if (m > t.M) return;
  const int item = s % bpm;
  const int w = item / nkb, kb = item - w * nkb;
  __shared__ double2 seeds[sweep_lds(RL, KB)];
  legendre_item<RL, KB>(t, m, w, kb, w, threadIdx.x, seeds);
}

// ------------------------------------------------------------ launchers

static inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t launch_seeds(const LegTables &t, hipStream_t s) {
  const int64_t n = (int64_t)(t.M + 1) * t.R;
  hipLaunchKernelGGL(k_seeds, dim3(nblocks(n, 256)), dim3(256), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_checkpoints(const LegTables &t, hipStream_t s) {
  hipLaunchKernelGGL(k_checkpoints, dim3((unsigned)((t.M + 1) * t.SW)), dim3(kSegRings), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_pair_tables(const LegTables &t, hipStream_t s) {
  hipLaunchKernelGGL(k_pair_tables, dim3((unsigned)(t.M + 1)), dim3(64), 0, s, t);
  return hipGetLastError();
}

hipError_t launch_wave_bounds(const LegTables &t, hipStream_t s) {
  const int64_t n = (int64_t)(t.M + 1) * t.W;
  hipLaunchKernelGGL(k_wave_bounds, dim3(nblocks(n, 256)), dim3(256), 0, s, t);
  return hipGetLastError();
}

// Maps per pass (KB) of the sweep: up to kMapsVector maps in one pass on the
// vector units, more in passes of at most 16 on the matrix cores, all of one
// even size.  Measured, ms of one sweep at lmax = 2 Nside = 2048 (vector with
// four maps a pass / vector of this form / matrix cores): 1 map 0.64 / 0.60 /
// 1.35, 2 maps 0.91 / 0.81 / 0.95, 3 maps 1.24 / 1.23 / 1.40, 4 maps 1.53 / - /
// 1.40, 6 maps 2.97 / - / 1.87, 8 maps 2.92 / - / 2.02, 64 maps 23.2 / - / 14.2.
// Geometries of few waves are bound by the length of a wave, not by the
// chip's rate; the matrix form's four segments make it four times shorter.
// Waves of the vector form at which the two are even: 3 maps between 3072
// (Nside 256, lmax 767: 114 / 79 us) and 8200 (Nside 512: 207 / 250 us),
// fewer maps between 514 (Nside 128: 23 / 17 us) and 2052 (Nside 256: 44 / 45).
int legendre_map_block(int K, int L, int M, int R) {
  if (K <= kMapsVector) {
    const int64_t waves = (int64_t)(M + 1) * ((R + 127) / 128);
    return waves < (K < 3 ? 1024 : 6144) ? kMapsVector + 1 : K;
  }
  // the matrix form's row offsets are 32 bits: 2 KB (lmax + kChunk) below 2^32
  const int most = L < (1 << 27) - kChunk ? 16 : 6;
  const int passes = (K + most - 1) / most, kb = (K + passes - 1) / passes;
  return (kb + 1) / 2 * 2;
}
bool legendre_matrix(int KB) { return KB > kMapsVector; }
// Rings per wave / 64: two on the vector units (each coefficient row then
// serves twice the rings; one: 0.87 ms where two take 0.60), two on the matrix
// cores while the accumulators leave two waves per SIMD and the waves fill
// the chip (6 maps: 1.87 ms, with one 2.01; 8 maps: 2.08, with one 2.02).
int legendre_default_rl(int K, int L, int M, int R) {
  const int KB = legendre_map_block(K, L, M, R);
  if (!legendre_matrix(KB)) return 2;
  return KB <= 6 && (int64_t)(M + 1) * ((R + 127) / 128) >= 2048 ? 2 : 1;
}
// The pair form of 3 maps a pass holds 76 registers, 6 waves a SIMD where the
// one-step form has 8, so it needs more waves than are resident at once: at
// 8200 waves (Nside 512, lmax 1024) it takes 0.183 ms where the one-step form
// takes 0.175, at 32784 (Nside 1024, lmax 2048) and more it is 5 .. 8 % faster.
// Fewer maps gain at every size (lmax 1024, 1 map 86 / 88 us, 2 maps 126 / 130).
// A ring's sums differ in the last bits between the forms, so the answer goes
// by the geometry and the map count alone, not by the rings per wave.
bool legendre_pairs(const LegTables &t) {
  int a, b;
  pair_units(t, kSegRings, &a, &b);
  return !legendre_matrix(t.KB) && a < b &&
         (t.KB < 3 || (int64_t)(t.M + 1) * ((t.R + kSegRings - 1) / kSegRings) >= 16384);
}
int legendre_unit_form(const LegTables &t, int u) {
  if (!legendre_pairs(t) || u * kSegRings < t.pair_r0 || (u + 1) * kSegRings > t.pair_r1) return -1;
  return pair_zone(ring_z(t.N, u * kSegRings + kSegRings / 2));
}
int legendre_padded_maps(int K, int KB) {
  return ((K + KB - 1) / KB) * KB;
}

hipError_t launch_prep_alm(const LegTables &t, const double2 *alm, hipStream_t s) {
  const int KB = t.KB;
  const int nkb = (t.K + KB - 1) / KB, Kp = KB * nkb;
  const int JB = Kp >= 256 ? 1 : 256 / Kp;
  hipLaunchKernelGGL(k_prep_alm, dim3((unsigned)((t.nlpad + JB - 1) / JB)), dim3(256), 0, s, t,
                     alm, KB, nkb);
  return hipGetLastError();
}

template <int RL, int KB>
static hipError_t launch_leg_t(const LegTables &t, hipStream_t s) {
  const int nkb = (t.K + KB - 1) / KB;
  const int bpm = t.W * nkb;
  const int mgroups = (t.M + 1 + 7) / 8;
  const unsigned grid = (unsigned)(8 * mgroups * bpm);
  hipLaunchKernelGGL((k_legendre<RL, KB>), dim3(grid), dim3(64), 0, s, t, nkb, bpm);
  return hipGetLastError();
}

// ---------------------------------------------------------------- batch

__global__ void k_batch_reset(int *counters) {
  if (threadIdx.x < kBatchCounters) counters[threadIdx.x] = 0;
}

// Prescale of every request's a_lm: thread g owns entry u = g - prep_off[r]
// of request r, u = j Kp + kk (padded l-entry j, map slot kk of Kp = KB nkb
// slots; maps fastest, as the single-plan prescale).
__global__ __launch_bounds__(256) void k_batch_prep(BatchDev b) {
  __shared__ int s_r0;
  const int64_t g0 = (int64_t)blockIdx.x * blockDim.x;
  if (threadIdx.x == 0) {
    int lo = 0, hi = b.nreq - 1;  // prep_off[lo] <= g0 < prep_off[lo + 1]
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (b.prep_off[mid] <= g0) lo = mid; else hi = mid - 1;
    }
    s_r0 = lo;
  }
  __syncthreads();
  const int64_t g = g0 + threadIdx.x;
  if (g >= b.prep_total) return;
  int lo = s_r0;  // the block's first request; few blocks span more than one
  while (g >= b.prep_off[lo + 1]) ++lo;
  const LegTables &t = b.tabs[lo];
  const int Kp = legendre_padded_maps_of(t.K, t.KB);
  const int64_t u = g - b.prep_off[lo];
  const int64_t j = u / Kp;
  prep_entry(t, b.alm[lo], j, (int)(u - j * Kp), t.KB);
}

// (RL, KB) shapes of the single-plan sweep (those of legendre_default_rl and
// legendre_map_block) and the further ones of a measured batch
#define WM_PLAN_SHAPES(X)                                                     \
  X(2, 1) X(2, 2) X(2, 3) X(1, 4) X(2, 4) X(1, 6) X(2, 6) X(1, 8)             \
  X(1, 10) X(1, 12) X(1, 14) X(1, 16)
#define WM_SWEEP_SHAPES(X)                                                    \
  WM_PLAN_SHAPES(X) X(1, 1) X(1, 2) X(1, 3) X(4, 1) X(4, 2) X(4, 3) X(2, 8)

bool batch_shape_supported(int RL, int KB) { return batch_shape_index(RL, KB) >= 0; }

int batch_shape_index(int RL, int KB) {
  int i = 0;
#define WM_IDX(R_, K_)                     \
  if (RL == R_ && KB == K_) return i;      \
  ++i;
  WM_SWEEP_SHAPES(WM_IDX)
#undef WM_IDX
  return -1;
}

// Persistent sweep of one shape: each wave takes items (request, m, ring
// chunk, map block) of the shape's queue until it runs dry; the host
// orders each queue costliest request first.  One kernel per shape, so
// each has the registers of its own shape (as the single-plan sweep).
template <int R_, int K_>
__global__ __launch_bounds__(256) void k_batch_legendre(BatchDev b, int first, int count,
                                                        int ctr) {
  __shared__ double2 seeds[4][sweep_lds(R_, K_)];
  const int lane = threadIdx.x & 63;
  for (;;) {
    int it = 0;
    if (lane == 0) it = atomicAdd(&b.counters[ctr], 1);
    it = __builtin_amdgcn_readfirstlane(__shfl(it, 0));
    if (it >= count) break;
    const WM_CONST BatchLegItem *ip = const_view(b.litems + first + it);
    const int req = ip->req, m = ip->m, w = ip->w, kb = ip->kb;
    const WM_CONST LegTables *tp = const_view(b.tabs + req);
    LegTables t;
    t.L = tp->L;
    t.M = tp->M;
    t.K = tp->K;
    t.R = tp->R;
    t.W = tp->W;
    t.nlpad = tp->nlpad;
    t.off = tp->off;
    t.ctil = tp->ctil;
    t.cscale = tp->cscale;
    t.ring_x = tp->ring_x;
    t.seed_l = tp->seed_l;
    t.seed_v = tp->seed_v;
    t.wstart = tp->wstart;
    t.wseedmax = tp->wseedmax;
    t.SW = tp->SW;
    t.seg_l0 = tp->seg_l0;
    t.ckpt = tp->ckpt;
    t.atil = tp->atil;
    t.ptil = tp->ptil;
    t.pair_r0 = tp->pair_r0;
    t.pair_r1 = tp->pair_r1;
    t.pair_t = tp->pair_t;
    t.pair_h = tp->pair_h;
    t.qbuf = tp->qbuf;
    if constexpr (R_ == 4 && K_ <= kMapsVector) {
      if (w < 0) {  // the wave's two units differ in form
#pragma unroll 1
        for (int u = 2 * (-1 - w); u < 2 * -w && u * kSegRings < t.R; ++u)
          legendre_item<2, K_>(t, m, u, kb, -1 - w, lane, seeds[threadIdx.x >> 6]);
        continue;
      }
    }
    legendre_item<R_, K_>(t, m, w, kb, w, lane, seeds[threadIdx.x >> 6]);
  }
}

hipError_t launch_batch_reset(const BatchDev &b, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3(64), 0, s, b.counters);
  return hipGetLastError();
}

hipError_t launch_batch_prep(const BatchDev &b, hipStream_t s) {
  if (b.prep_total == 0) return hipSuccess;
  hipLaunchKernelGGL(k_batch_prep, dim3(nblocks(b.prep_total, 256)), dim3(256), 0, s, b);
  return hipGetLastError();
}

hipError_t batch_legendre_occupancy(int RL, int KB, int *blocks_per_cu) {
#define WM_OCC(R_, K_)                                                                   \
  if (RL == R_ && KB == K_)                                                              \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu,                   \
                                                        k_batch_legendre<R_, K_>, 256, 0);
  WM_SWEEP_SHAPES(WM_OCC)
#undef WM_OCC
  return hipErrorInvalidValue;
}

hipError_t launch_batch_legendre(const BatchDev &b, int RL, int KB, int first, int count,
                                 int nb, hipStream_t s) {
  const int ctr = kBatchSweepCtr + batch_shape_index(RL, KB);
#define WM_LAUNCH(R_, K_)                                                                \
  if (RL == R_ && KB == K_) {                                                            \
    hipLaunchKernelGGL((k_batch_legendre<R_, K_>), dim3(nb), dim3(256), 0, s, b, first,  \
                       count, ctr);                                                      \
    return hipGetLastError();                                                            \
  }
  WM_SWEEP_SHAPES(WM_LAUNCH)
#undef WM_LAUNCH
  return hipErrorInvalidValue;
}

hipError_t launch_legendre(const LegTables &t, hipStream_t s) {
#define WM_LAUNCH(R_, K_) \
  if (t.RL == R_ && t.KB == K_) return launch_leg_t<R_, K_>(t, s);
  WM_PLAN_SHAPES(WM_LAUNCH)
#undef WM_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace wm
