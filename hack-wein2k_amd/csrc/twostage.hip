// Two-stage reduction of the standard-form matrix C to tridiagonal form, for
// both builds (CX: complex Hermitian, planar; else real symmetric):
//   1. C = Q1 B Q1^H, B of bandwidth BND: per BND columns a Householder QR of the
//      panel below the band (k_sb_qr) and one rank-2 BND update of the trailing
//      matrix, so that the matrix is read by products instead of by one
//      matrix-vector product per column;
//   2. B = Q2 T Q2^H by bulge chasing (k_sb_chase), T real tridiagonal;
//   3. the vectors of T are multiplied by Q2 here (sb_apply_q2) and by Q1 in
//      the drivers' back-transform.
// The reference reduces column by column (dsytrd2.f, zheevx2.f:305-367); both
// give an orthogonally similar T, so eigenvalues agree to rounding and
// eigenvectors up to the phase that they are determined to.
//
// Column by column the matrix is read once per column (HBM bound at large
// orders, 4.5 TB/s) through two dependent launches per column (12-24 us at
// small ones).  Here a panel of BND columns takes six launches, the flops are
// matrix products, and the serial part is 32 short exchanges per panel and
// two steps per sweep.  Whole reduction, before -> now (Q2's application in
// brackets): real N = 221 3.1 -> 1.3 ms, N = 731 10.7 -> 5.3, N = 5951 135 ->
// 60 (+ 6); complex N = 251 5.4 -> 2.5, N = 1950 47 -> 25 (+ 2), N = 10880
// 1018 -> 326 (+ 86).
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include <hip/hip_ext.h>

#include "mfma.h"
#include "seclr4_shared.h"
#include "twostage.h"

namespace w2k {

// ------------------------------------------------------------------ device-wide words
// Data exchanged between work-groups of a running kernel goes through relaxed
// agent-scope accesses, which pass the XCDs' private L2 caches; a wave orders
// its stores before a later flag with vm_drain().
__device__ __forceinline__ double agent_ld(const double *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int agent_ld(const int *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_st(double *p, double v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_st(int *p, int v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every vector memory access of this wave done (vmcnt = 0)
__device__ __forceinline__ void vm_drain()
{
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// sum over the 32 lanes of a half wave, in every lane
__device__ __forceinline__ double sum32(double v)
{
  v = swap_sum<16>(v, v);
  v += bfly_partner<8>(v);
  v += bfly_partner<4>(v);
  v += bfly_partner<2>(v);
  return v + bfly_partner<1>(v);
}

// the lower and the upper half wave's value, in every lane
__device__ __forceinline__ void swap_halves(double v, double &lower, double &upper)
{
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)((unsigned long long)b >> 32);
  const auto x = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  lower = __longlong_as_double((long long)((unsigned long long)y[0] << 32 | x[0]));
  upper = __longlong_as_double((long long)((unsigned long long)y[1] << 32 | x[1]));
}
// t[0..N-1] per lane, summed over the 32 lanes of each half: lane l returns
// entry (l & 31) / (32 / N), N = 4 or 8
template <int N>
__device__ __forceinline__ double half_sums(double *t, int lane)
{
  static_assert(N == 4 || N == 8, "entries");
#pragma unroll
  for (int j = 0; j < N / 2; j++) t[j] = swap_sum<16>(t[j], t[j + N / 2]);
  bfly_step_h<8, N / 4>(t, lane);
  if constexpr (N == 8) bfly_step_h<4, N / 8>(t, lane);
  else t[0] += bfly_partner<4>(t[0]);
  t[0] += bfly_partner<2>(t[0]);
  return t[0] + bfly_partner<1>(t[0]);
}

// xLARFG of (alpha, x) with |x|^2 = ss: H = I - tau v v^H, H^H (alpha; x) =
// (beta; 0), v = (1; scale x), beta real
struct Reflector {
  double beta, tr, ti, sr, si;
};
template <bool CX>
__device__ __forceinline__ Reflector larfg(double ar, double ai, double ss)
{
#pragma clang fp contract(off)  // the same bits wherever it is inlined
  Reflector h;
  if (ss == 0.0 && (!CX || ai == 0.0)) {
    h.beta = ar;
    h.tr = h.ti = h.sr = h.si = 0.0;
    return h;
  }
  // norm and 1 / norm by Goldschmidt's iteration from the hardware's estimate
  // (two rounds and a correction: rounding error only), the library's
  // functions outside its range
  const double x = CX ? fma(ar, ar, fma(ai, ai, ss)) : fma(ar, ar, ss);
  double nrm, inv;
  if (x > 1.0e-280 && x < 1.0e280) {
    const double y = __builtin_amdgcn_rsq(x);
    double q = x * y, hh = 0.5 * y;
    double e = fma(-q, hh, 0.5);
    q = fma(q, e, q);
    hh = fma(hh, e, hh);
    e = fma(-q, hh, 0.5);
    q = fma(q, e, q);
    hh = fma(hh, e, hh);
    nrm = fma(fma(-q, q, x), hh, q);
    inv = 2.0 * fma(hh, fma(-nrm, 2.0 * hh, 1.0), hh);
  } else {
    nrm = sqrt(x);
    inv = 1.0 / nrm;
  }
  const double a = fabs(ar), d = a + nrm;  // alpha - beta = +-d + i alpha_i
  const double den = CX ? fma(d, d, ai * ai) : d;
  double rd;
  if (den > 1.0e-280 && den < 1.0e280) {
    rd = __builtin_amdgcn_rcp(den);
    rd = fma(rd, fma(-den, rd, 1.0), rd);
    rd = fma(rd, fma(-den, rd, 1.0), rd);
  } else {
    rd = 1.0 / den;
  }
  const bool neg = ar < 0.0;
  h.beta = neg ? nrm : -nrm;
  h.tr = fma(a, inv, 1.0);
  if (CX) {
    h.ti = (neg ? -ai : ai) * inv;
    h.sr = (neg ? -d : d) * rd;
    h.si = -ai * rd;
  } else {
    h.ti = h.si = 0.0;
    h.sr = neg ? -rd : rd;
  }
  return h;
}

// ------------------------------------------------------------------ 1a. panel QR
// "not yet written" in the exchange buffer: a NaN pattern that arithmetic does
// not produce (a value with these bits is published as another NaN)
constexpr long long SB_EMPTY = 0x7FF8DEADBEEF5A5All;
constexpr int QR_ROWS = 256;          // rows of a block (one per thread)
constexpr int SB_CLOSED = 1 << 30;    // registration word: no more work-groups
constexpr long long QR_WAIT = 3000;   // registration wait, ticks of the 100 MHz counter (30 us)

__global__ void k_sb_reset(double *exch, size_t cnt, int *sync)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cnt) exch[i] = __longlong_as_double(SB_EMPTY);
  if (i < 4) sync[i] = 0;
}

// values k of blocks b0, b0 + step, .. < nb summed in that order, each taken
// once it has been written; eight loads in flight
__device__ __forceinline__ double gather_sum(const double *ex, int b0, int step, int nb, size_t stride)
{
  double s = 0.0;
  for (int b = b0; b < nb; b += 8 * step) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int bb = b + q * step;
      v[q] = bb < nb ? agent_ld(ex + (size_t)bb * stride) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int bb = b + q * step;
      while (__double_as_longlong(v[q]) == SB_EMPTY) v[q] = agent_ld(ex + (size_t)bb * stride);
      if (bb < nb) s += v[q];
    }
  }
  return s;
}

// Householder QR of the panel A(r0:n, j0:j0+BND), r0 = j0 + BND: R and the
// reflectors in place, V (unit lower trapezoidal, explicit) to P columns
// 0..BND-1 and 2 BND..3 BND-1, tau, and G = V^H V above its diagonal.  One row
// per thread with its BND columns in registers; per column one reduction over
// all rows gives the norm, the products with the remaining columns and those
// with the earlier reflectors (G), exchanged between the work-groups through
// `exch`.  The columns sit rotated: entry k of a row is column j + k
// (mod BND), earlier reflectors take the place of finished columns.
//
// Progress does not depend on all work-groups being resident: a work-group
// registers when it starts, the first one closes the registration once all
// have come or QR_WAIT has passed, later ones leave, and the registered ones
// share the blocks (RES: each has one, held in registers; else all go through
// memory), with the same sums in the same order either way.
template <bool CX>
struct QrShared {
  static constexpr int NV = CX ? 2 * BND : BND, NG = QR_ROWS / NV;
  double red[4][NV], piv[NV], cf[NV], part[NG][NV];
  int share[2];
};

template <bool CX, bool RES>
__device__ __forceinline__ void qr_panel(const SbArgs &g, int j0, int nblk, int idx, int np, QrShared<CX> &sh)
{
#pragma clang fp contract(off)  // both forms round alike
  constexpr int NV = QrShared<CX>::NV, NG = QrShared<CX>::NG;
  const int n = g.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = j0 + BND, m = n - r0, nref = min(BND, m - 1);
  double xr[BND], xi[CX ? BND : 1];
  double *const pv = g.Pr, *const pvi = g.Pi;
  // the row's columns in their rotated places at step j
  auto load = [&](int b, int j) {
    const int pr = b * QR_ROWS + tid;
    const bool live = pr < m;
    const size_t row = r0 + min(pr, m - 1);
#pragma unroll
    for (int k = 0; k < BND; k++) {
      const bool old = k >= BND - j;
      const size_t o = old ? row + (size_t)n * (j + k - BND) : row + (size_t)g.lda * (j0 + j + k);
      const double vr = old ? pv[o] : g.ar[o];
      xr[k] = live ? vr : 0.0;
      if (CX) {
        const double vi = old ? pvi[o] : g.ai[o];
        xi[k] = live ? vi : 0.0;
      }
    }
  };
  if (RES) load(idx, 0);
  for (int j = 0; j < nref; j++) {
    double *const ex = g.exch + (size_t)j * (nblk + 1) * NV;
    for (int b = idx; b < nblk; b += np) {
      if (!RES) load(b, j);
      const int pr = b * QR_ROWS + tid;
      double t[BND];
      const double ar = pr > j ? xr[0] : 0.0, ai = CX ? (pr > j ? xi[0] : 0.0) : 0.0;
#pragma unroll
      for (int k = 0; k < BND; k++) t[k] = CX ? fma(ar, xr[k], ai * xi[k]) : ar * xr[k];
      const double s0 = wave_transpose_sum32x(t, lane);
      if (!(lane & 1)) sh.red[wave][lane >> 1] = s0;
      if (CX) {
#pragma unroll
        for (int k = 0; k < BND; k++) t[k] = fma(ar, xi[k], -(ai * xr[k]));
        const double s1 = wave_transpose_sum32x(t, lane);
        if (!(lane & 1)) sh.red[wave][BND + (lane >> 1)] = s1;
      }
      if (pr == j) {
#pragma unroll
        for (int k = 0; k < BND; k++) {
          sh.piv[k] = xr[k];
          if (CX) sh.piv[BND + k] = xi[k];
        }
      }
      __syncthreads();
      if (nblk > 1) {
        if (tid < NV) {
          double s = ((sh.red[0][tid] + sh.red[1][tid]) + sh.red[2][tid]) + sh.red[3][tid];
          if (__double_as_longlong(s) == SB_EMPTY) s = __longlong_as_double(0x7FF8000000000000ll);
          agent_st(ex + (size_t)b * NV + tid, s);
          if (b == 0) {
            double p = sh.piv[tid];
            if (__double_as_longlong(p) == SB_EMPTY) p = __longlong_as_double(0x7FF8000000000000ll);
            agent_st(ex + (size_t)nblk * NV + tid, p);
          }
        }
        if (!RES) __syncthreads();  // red and piv are written again
      }
      if (RES) break;
    }
    // sum over the rows of conj(x_0) x_k
    auto total = [&](int k) {
      if (nblk == 1) return ((sh.red[0][k] + sh.red[1][k]) + sh.red[2][k]) + sh.red[3][k];
      double s = sh.part[0][k];
#pragma unroll
      for (int q = 1; q < NG; q++) s += sh.part[q][k];
      return s;
    };
    if (nblk > 1) {
      const int k = tid % NV, grp = tid / NV;
      sh.part[grp][k] = gather_sum(ex + k, grp, NG, nblk, NV);
      if (grp == NG - 1) sh.piv[k] = gather_sum(ex + (size_t)nblk * NV + k, 0, 1, 1, NV);
      __syncthreads();
    }
    const Reflector h = larfg<CX>(sh.piv[0], CX ? sh.piv[BND] : 0.0, total(0));
    if (tid < BND) {
      // v^H x_k = p_k + conj(scale) S_k
      const double a = total(tid);
      double wr, wi = 0.0;
      if (CX) {
        const double b = total(BND + tid);
        wr = fma(h.sr, a, fma(h.si, b, sh.piv[tid]));
        wi = fma(h.sr, b, fma(-h.si, a, sh.piv[BND + tid]));
      } else {
        wr = fma(h.sr, a, sh.piv[tid]);
      }
      const bool old = tid >= BND - j;  // an earlier reflector: G(i, j) = conj(v_j^H v_i)
      if (old && idx == 0) {
        g.G[j + tid - BND + BND * j] = wr;
        if (CX) g.G[BND * BND + j + tid - BND + BND * j] = -wi;
      }
      sh.cf[tid] = old ? 0.0 : (CX ? fma(h.tr, wr, h.ti * wi) : h.tr * wr);  // conj(tau) w
      if (CX) sh.cf[BND + tid] = old ? 0.0 : fma(h.tr, wi, -(h.ti * wr));
      if (tid == 0 && idx == 0) {
        g.taur[j0 + j] = h.tr;
        if (CX) g.taui[j0 + j] = h.ti;
      }
    }
    __syncthreads();
    for (int b = idx; b < nblk; b += np) {
      if (!RES) load(b, j);
      const int pr = b * QR_ROWS + tid;
      const double x0r = xr[0], x0i = CX ? xi[0] : 0.0;
      double vr = pr > j ? (CX ? fma(h.sr, x0r, -(h.si * x0i)) : h.sr * x0r) : (pr == j ? 1.0 : 0.0);
      double vi = CX && pr > j ? fma(h.sr, x0i, h.si * x0r) : 0.0;
      if (pr >= m) vr = vi = 0.0;
#pragma unroll
      for (int k = 1; k < BND; k++) {
        const double cr = sh.cf[k];
        if (CX) {
          const double ci = sh.cf[BND + k];
          xr[k - 1] = fma(vi, ci, fma(-vr, cr, xr[k]));
          xi[k - 1] = fma(-vi, cr, fma(-vr, ci, xi[k]));
        } else {
          xr[k - 1] = fma(-vr, cr, xr[k]);
        }
      }
      xr[BND - 1] = vr;
      if (CX) xi[BND - 1] = vi;
      if (pr < m) {
        const size_t row = r0 + pr;
        const size_t oa = row + (size_t)g.lda * (j0 + j), op = row + (size_t)n * j;
        g.ar[oa] = pr > j ? vr : (pr == j ? h.beta : x0r);
        pv[op] = vr;
        pv[op + (size_t)2 * BND * n] = vr;
        if (CX) {
          g.ai[oa] = pr > j ? vi : (pr == j ? 0.0 : x0i);
          pvi[op] = vi;
          pvi[op + (size_t)2 * BND * n] = vi;
        }
        if (!RES) {
#pragma unroll
          for (int k = 1; k < BND; k++) {
            if (k >= BND - j) continue;
            g.ar[row + (size_t)g.lda * (j0 + j + k)] = xr[k - 1];
            if (CX) g.ai[row + (size_t)g.lda * (j0 + j + k)] = xi[k - 1];
          }
        }
      }
      if (RES) break;
    }
  }
  // columns past the last reflector (short panels, one block): R as it is, V = 0
  if (RES && nref < BND) {
    if (tid < m) {
#pragma unroll
      for (int k = 0; k < BND; k++) {
        const int j = nref + k;
        if (j >= BND) continue;
        const size_t row = r0 + tid, oa = row + (size_t)g.lda * (j0 + j), op = row + (size_t)n * j;
        g.ar[oa] = xr[k];
        pv[op] = 0.0;
        pv[op + (size_t)2 * BND * n] = 0.0;
        if (CX) {
          g.ai[oa] = xi[k];
          pvi[op] = 0.0;
          pvi[op + (size_t)2 * BND * n] = 0.0;
        }
      }
    }
    if (tid >= nref && tid < BND && j0 + tid < n) {
      g.taur[j0 + tid] = 0.0;
      if (CX) g.taui[j0 + tid] = 0.0;
    }
  }
}

template <bool CX>
__global__ __launch_bounds__(QR_ROWS) void k_sb_qr(SbArgs g, int j0)
{
  __shared__ QrShared<CX> sh;
  const int tid = threadIdx.x, m = g.n - (j0 + BND);
  const int nblk = (m + QR_ROWS - 1) / QR_ROWS;
  int idx = 0, np = 1;
  if (nblk > 1) {
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(g.sync, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int me = old, cnt = 0;
      if (old & SB_CLOSED || old >= g.qr_cap) {
        me = -1;
      } else if (old == 0) {
        const long long t0 = wall_clock64();
        while (agent_ld(g.sync) < nblk && wall_clock64() - t0 < QR_WAIT) __builtin_amdgcn_s_sleep(1);
        cnt = min(__hip_atomic_fetch_or(g.sync, SB_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), g.qr_cap);
        agent_st(g.sync + 1, cnt);
      } else {
        while ((cnt = agent_ld(g.sync + 1)) == 0) __builtin_amdgcn_s_sleep(1);
      }
      sh.share[0] = me;
      sh.share[1] = cnt;
    }
    __syncthreads();
    idx = __builtin_amdgcn_readfirstlane(sh.share[0]);
    np = __builtin_amdgcn_readfirstlane(sh.share[1]);
    if (idx < 0) return;
  }
  if (np >= nblk) qr_panel<CX, true>(g, j0, nblk, idx, np, sh);
  else qr_panel<CX, false>(g, j0, nblk, idx, np, sh);
}

// T of I - V T V^H from G = V^H V and tau: T(0:i, i) = -tau_i T(0:i, 0:i)
// G(0:i, i), T(i, i) = tau_i; one wave, lanes r and r + 32 taking the even and
// odd terms of row r
template <bool CX>
__device__ __forceinline__ void panel_t(const SbArgs &g, int j0, double (*tm)[BND][BND + 1], double (*gm)[BND][BND + 1])
{
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int nref = min(BND, g.n - (j0 + BND) - 1);
  for (int e = tid; e < BND * BND; e += blockDim.x) {
    const int a = e % BND, b = e / BND;
    const bool in = a < b && b < nref;
    tm[0][a][b] = 0.0;
    gm[0][a][b] = in ? g.G[e] : 0.0;
    if (CX) {
      tm[1][a][b] = 0.0;
      gm[1][a][b] = in ? g.G[BND * BND + e] : 0.0;
    }
  }
  __syncthreads();
  if (tid < 64) {
    for (int i = 0; i < nref; i++) {
      const double tr = g.taur[j0 + i], ti = CX ? g.taui[j0 + i] : 0.0;
      double ar = 0.0, ai = 0.0;
#pragma unroll 4
      for (int q = h; q < i; q += 2) {
        const double a = tm[0][r][q], b = gm[0][q][i];
        if (CX) {
          const double a2 = tm[1][r][q], b2 = gm[1][q][i];
          ar += a * b - a2 * b2;
          ai += a * b2 + a2 * b;
        } else {
          ar += a * b;
        }
      }
      ar += xor32(ar, lane);
      if (CX) ai += xor32(ai, lane);
      if (h == 0 && r <= i) {
        tm[0][r][i] = r < i ? -(CX ? tr * ar - ti * ai : tr * ar) : tr;
        if (CX) tm[1][r][i] = r < i ? -(tr * ai + ti * ar) : ti;
      }
      wave_sync();
    }
  }
  __syncthreads();
  for (int e = tid; e < BND * BND; e += blockDim.x) {
    g.T[e] = tm[0][e % BND][e / BND];
    if (CX) g.T[BND * BND + e] = tm[1][e % BND][e / BND];
  }
}

// ------------------------------------------------------------------ 1b. Y = A V
// Partial products of A(r0:n, r0:n) (lower triangle stored) with the panel V:
// a work-group forms 64 rows of Y over one slice of K, four waves of 16 rows
// each, operands swapped (D = V^T A^T) so that the 16 rows of a result lie
// across lanes.  A goes from memory to registers (no wave shares it), one
// 64-column slab ahead; V through LDS.  Lane group q takes k = 4q + s of a
// 16-wide chunk at step s, which makes the transposed reads (k beyond the
// row) 32 contiguous bytes per lane.
constexpr int AV_K = 64, AV_LD = 36;

// The block past the last row forms the panel's T meanwhile.
template <bool CX>
__global__ __launch_bounds__(256, 2) void k_sb_av(SbArgs g, int r0, int slab, int mp)
{
  constexpr int CP = CX ? 2 : 1;
  __shared__ double lds[CP * AV_K * AV_LD];
  static_assert(AV_K * AV_LD >= 2 * BND * (BND + 1), "T and G fit");
  if ((int)blockIdx.x * 64 >= g.n - r0) {
    if (blockIdx.y == 0)
      panel_t<CX>(g, r0 - BND, reinterpret_cast<double(*)[BND][BND + 1]>(lds),
                  reinterpret_cast<double(*)[BND][BND + 1]>(lds + CP * BND * (BND + 1)));
    return;
  }
  double(*vs)[AV_K][AV_LD] = reinterpret_cast<double(*)[AV_K][AV_LD]>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, q4 = lane >> 4;
  const int m = g.n - r0, n = g.n;
  const int i0 = blockIdx.x * 64 + 16 * wave;  // first row of the wave
  const int kb = blockIdx.y * slab * AV_K, ke = min(m, kb + slab * AV_K);
  const double *ar = g.ar + (size_t)r0 + (size_t)g.lda * r0;
  const double *ai = CX ? g.ai + (size_t)r0 + (size_t)g.lda * r0 : nullptr;
  const int i = min(i0 + l16, m - 1);
  double pr[16], pi[CX ? 16 : 1];
  // chunk c, step s of slab k0: element (i, k), k = k0 + 16 c + 4 q4 + s, from
  // the stored triangle (its conjugate where k > i)
  auto loadA = [&](int k0) {
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = min(k0 + 16 * c + 4 * q4 + s, m - 1);
        const bool up = k > i;
        const size_t o = up ? (size_t)k + (size_t)g.lda * i : (size_t)i + (size_t)g.lda * k;
        pr[4 * c + s] = ar[o];
        if (CX) {
          const double v = ai[o];
          pi[4 * c + s] = up ? -v : (k == i ? 0.0 : v);
        }
      }
  };
  d4 yr[2], yi[CX ? 2 : 1];
  for (int t = 0; t < 2; t++) {
    yr[t] = d4{0.0, 0.0, 0.0, 0.0};
    if (CX) yi[t] = d4{0.0, 0.0, 0.0, 0.0};
  }
  loadA(kb);
  for (int k0 = kb; k0 < ke; k0 += AV_K) {
    double br[16], bi[CX ? 16 : 1];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      br[q] = pr[q];
      if (CX) bi[q] = pi[q];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const int k = tid & 63, col = (tid >> 6) + 4 * c;
      const bool ok = k0 + k < ke;
      const size_t o = (size_t)(r0 + min(k0 + k, m - 1)) + (size_t)n * col;
      const double v = g.Pr[o];
      vs[0][k][col] = ok ? v : 0.0;
      if (CX) {
        const double w = g.Pi[o];
        vs[1][k][col] = ok ? w : 0.0;
      }
    }
    if (k0 + AV_K < ke) loadA(k0 + AV_K);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = 16 * c + 4 * q4 + s, e = 4 * c + s;
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const double vr = vs[0][k][16 * t + l16];
          yr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vr, br[e], yr[t], 0, 0, 0);
          if (CX) {
            const double vi = vs[1][k][16 * t + l16];
            yr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-vi, bi[e], yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vi, br[e], yi[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vr, bi[e], yi[t], 0, 0, 0);
          }
        }
      }
  }
  mfma_settle();
  // D(c, i): lane i + 16 (c % 4), item c / 4
  if (i0 + l16 < m) {
    const size_t plane = (size_t)mp * BND;
    double *out = g.part + (size_t)blockIdx.y * plane * (CX ? 2 : 1);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const size_t o = (size_t)(i0 + l16) + (size_t)mp * (16 * t + q4 + 4 * r);
        out[o] = yr[t][r];
        if (CX) out[plane + o] = yi[t][r];
      }
  }
}

// Z = (sum of the slices) T for 32 rows per work-group (fixed order), and the
// work-group's part of V^H Z
template <bool CX>
__global__ __launch_bounds__(256) void k_sb_y(SbArgs g, int r0, int nz, int mp)
{
  constexpr int CP = CX ? 2 : 1;
  __shared__ double ys[CP][32][BND + 1], vs[CP][32][BND + 1], ts[CP][BND][BND + 1], zs[CP][32][BND + 1];
  const int tid = threadIdx.x, n = g.n, m = n - r0, t0 = blockIdx.x * 32;
  const size_t plane = (size_t)mp * BND;
  const int r = tid & 31, c0 = tid >> 5;
  const bool ok = t0 + r < m;
  const int rr = min(t0 + r, m - 1);
  double ar[4] = {0.0, 0.0, 0.0, 0.0}, ai[4] = {0.0, 0.0, 0.0, 0.0};
  const double *p = g.part + rr + (size_t)mp * c0;
#pragma unroll 4
  for (int z = 0; z < nz; z++) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      ar[q] += p[(size_t)mp * 8 * q];
      if (CX) ai[q] += p[plane + (size_t)mp * 8 * q];
    }
    p += plane * CP;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = c0 + 8 * q;
    const size_t ov = (size_t)(r0 + rr) + (size_t)n * c;
    const double vr = g.Pr[ov];
    ys[0][r][c] = ok ? ar[q] : 0.0;
    vs[0][r][c] = ok ? vr : 0.0;
    ts[0][r][c] = g.T[r + BND * c];
    if (CX) {
      const double vi = g.Pi[ov];
      ys[1][r][c] = ok ? ai[q] : 0.0;
      vs[1][r][c] = ok ? vi : 0.0;
      ts[1][r][c] = g.T[BND * BND + r + BND * c];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; q++) ar[q] = ai[q] = 0.0;
#pragma unroll 4
  for (int a = 0; a < BND; a++) {
    const double yr = ys[0][r][a], yi = CX ? ys[CP - 1][r][a] : 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double tr = ts[0][a][c0 + 8 * q];
      ar[q] += yr * tr;
      if (CX) {
        const double ti = ts[CP - 1][a][c0 + 8 * q];
        ar[q] -= yi * ti;
        ai[q] += yr * ti + yi * tr;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = c0 + 8 * q;
    const size_t ov = (size_t)(r0 + rr) + (size_t)n * c;
    zs[0][r][c] = ar[q];
    if (ok) g.Yr[ov] = ar[q];
    if (CX) {
      zs[CP - 1][r][c] = ai[q];
      if (ok) g.Yi[ov] = ai[q];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; q++) ar[q] = ai[q] = 0.0;
#pragma unroll 4
  for (int x = 0; x < 32; x++) {
    const double vr = vs[0][x][r], vi = CX ? vs[CP - 1][x][r] : 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double zr = zs[0][x][c0 + 8 * q];
      ar[q] += vr * zr;
      if (CX) {
        const double zi = zs[CP - 1][x][c0 + 8 * q];
        ar[q] += vi * zi;
        ai[q] += vr * zi - vi * zr;
      }
    }
  }
  double *out = g.spart + (size_t)blockIdx.x * BND * BND * CP;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int e = r + BND * (c0 + 8 * q);
    out[e] = ar[q];
    if (CX) out[BND * BND + e] = ai[q];
  }
}

// S = V^H Z from its parts, 32 entries per work-group (fixed order)
__global__ __launch_bounds__(256) void k_sb_s(SbArgs g, int nwg, int stride)
{
  __shared__ double red[8][33];
  const int tid = threadIdx.x, e = tid & 31, grp = tid >> 5;
  const double *p = g.spart + (size_t)blockIdx.x * 32 + e;
  double s = 0.0;
#pragma unroll 8
  for (int w = grp; w < nwg; w += 8) s += p[(size_t)w * stride];
  red[grp][e] = s;
  __syncthreads();
  if (tid < 32) {
    s = red[0][tid];
#pragma unroll
    for (int q = 1; q < 8; q++) s += red[q][tid];
    g.S[blockIdx.x * 32 + tid] = s;
  }
}

// W = Z - 1/2 V (T^H S) (P columns BND..2 BND-1), which makes the update
// Q^H A Q = A - V W^H - W V^H; also clears the exchange buffer of the next
// panel's QR
template <bool CX>
__global__ __launch_bounds__(256) void k_sb_w(SbArgs g, int r0, size_t nexch)
{
  constexpr int CP = CX ? 2 : 1;
  __shared__ double vs[CP][32][BND + 1], ts[CP][BND][BND + 1], ss[CP][BND][BND + 1], mm[CP][BND][BND + 1];
  const int tid = threadIdx.x, n = g.n, m = n - r0, t0 = blockIdx.x * 32;
  const int r = tid & 31, c0 = tid >> 5;
  for (size_t i = (size_t)blockIdx.x * 256 + tid; i < nexch; i += (size_t)gridDim.x * 256)
    g.exch[i] = __longlong_as_double(SB_EMPTY);
  if (blockIdx.x == 0 && tid < 4) g.sync[tid] = 0;
  const size_t row = r0 + min(t0 + r, m - 1);
  double zr[4], zi[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = c0 + 8 * q;
    const size_t o = row + (size_t)n * c;
    zr[q] = g.Yr[o];
    vs[0][r][c] = g.Pr[o];
    ts[0][r][c] = g.T[r + BND * c];
    ss[0][r][c] = g.S[r + BND * c];
    if (CX) {
      zi[q] = g.Yi[o];
      vs[CP - 1][r][c] = g.Pi[o];
      ts[CP - 1][r][c] = g.T[BND * BND + r + BND * c];
      ss[CP - 1][r][c] = g.S[BND * BND + r + BND * c];
    }
  }
  __syncthreads();
  double ar[4] = {0.0, 0.0, 0.0, 0.0}, ai[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int a = 0; a < BND; a++) {  // T^H S
    const double tr = ts[0][a][r], ti = CX ? ts[CP - 1][a][r] : 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double sr = ss[0][a][c0 + 8 * q];
      ar[q] += tr * sr;
      if (CX) {
        const double si = ss[CP - 1][a][c0 + 8 * q];
        ar[q] += ti * si;
        ai[q] += tr * si - ti * sr;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    mm[0][r][c0 + 8 * q] = -0.5 * ar[q];
    if (CX) mm[CP - 1][r][c0 + 8 * q] = -0.5 * ai[q];
  }
  __syncthreads();
#pragma unroll 4
  for (int a = 0; a < BND; a++) {
    const double vr = vs[0][r][a], vi = CX ? vs[CP - 1][r][a] : 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double mr = mm[0][a][c0 + 8 * q];
      zr[q] += vr * mr;
      if (CX) {
        const double mi = mm[CP - 1][a][c0 + 8 * q];
        zr[q] -= vi * mi;
        zi[q] += vr * mi + vi * mr;
      }
    }
  }
  if (t0 + r < m) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const size_t o = row + (size_t)n * (BND + c0 + 8 * q);
      g.Pr[o] = zr[q];
      if (CX) g.Pi[o] = zi[q];
    }
  }
}

// ------------------------------------------------------------------ 2. bulge chasing
// band storage: column j at ab + BLD j, entry (i, j) at offset i - j (0..BLD-1)
constexpr int BLD = 2 * BND;
constexpr int BPAD = 4 * BND;  // columns of zeros after the band's last one
constexpr int CHASE_DONE = 1 << 30;
constexpr int CHASE_KD = 3, CHASE_KZ = 2;  // sweeps per work-group (real, complex)

template <bool CX>
__global__ void k_sb_band(SbArgs g)
{
  const int o = threadIdx.x & (BLD - 1), j = blockIdx.x * (blockDim.x / BLD) + threadIdx.x / BLD;
  if (j >= g.n + BPAD) return;
  const bool in = o <= BND && j + o < g.n;
  const size_t a = in ? (size_t)(j + o) + (size_t)g.lda * j : 0, d = (size_t)BLD * j + o;
  g.ab[d] = in ? g.ar[a] : 0.0;
  if (CX) g.ab[(size_t)BLD * (g.n + BPAD) + d] = in && o > 0 ? g.ai[a] : 0.0;
  if (o == 0 && j <= g.n) g.prog[j] = 0;  // the last one: the sweeps' ticket
}

template <class T>
__device__ __forceinline__ T *byte_at(T *p, unsigned bytes)
{
  return (T *)((std::conditional_t<std::is_const_v<T>, const char, char> *)p + bytes);
}

constexpr int CNC = 4;  // columns per lane of a sweep's four waves

// Sweep s reduces column s of the band and chases the bulge that this makes
// down the matrix.  Rows R_t = s + 1 + BND t .. (BND of them); step t applies
// the reflector of R_t to the diagonal block D = A(R_t, R_t) from both sides
// and to C = A(R_t+1, R_t) from the right, and forms the reflector of R_t+1
// from C's first column and applies it to C from the left: it reads and
// writes the band's columns R_t.  Step t of sweep s needs the steps up to
// t + 1 of sweep s - 1 (C's last entry is what that step leaves of its first
// column), so sweeps follow each other two steps apart; step -1 forms the
// reflector of R_0 from column s.
//
// What a sweep costs is that distance: two steps, and the way of the columns
// through memory (drain, flag, poll, load: about 3 us).  So a work-group runs
// K consecutive sweeps, four waves each, in step: at tick k sweep w of the
// group does its step k - 2 w, and hands its columns to the next sweep through
// LDS (two steps' columns, the older ones read at the start of the tick in
// which they are overwritten).  Only the first sweep reads the band from
// memory, a tick ahead, and only the last writes it, publishing its progress a
// tick late, so that neither waits for memory within a tick.
//
// A step itself is bound by the chain of its operations and, with K waves on
// each SIMD, by their issue.  Two barriers a step: between the waves' shares
// of D v and C v and their sums, and before the next sweep reads; what follows
// the sums is done by every wave for itself.  The band has columns of zeros
// after the last one, and sweeps and steps past the matrix' end run on those:
// no step has an edge.  Measured on the reduction as a whole (whose products took
// up to 4 ms more then than now), one sweep per work-group and three barriers a
// step -> as here: real N = 731 7.4 -> 5.3 ms, N = 5951 79 -> 64; complex N =
// 251 2.9 -> 2.6, N = 1950 28.2 -> 25.8.  K = 2, 3, 4 took 5.5, 5.3, 5.5 (N =
// 731) and 69, 64, 63 ms (N = 5951), complex K = 1, 2, 3 3.2, 2.6, 2.5 (N =
// 251) and 30.8, 25.8, 26.4 ms (N = 1950).
//
// A work-group takes groups of sweeps in order from a ticket: the oldest
// unfinished group always has a running work-group and waits for nothing, so
// no residency is assumed.  Lane (r, h) of wave w of a sweep holds row r,
// columns (2 w + h) CNC .. of D (mirrored) and C.
template <bool CX, int K>
__global__ __launch_bounds__(256 * K) void k_sb_chase(SbArgs g)
{
  constexpr int CP = CX ? 2 : 1;
  // columns of a sweep's last two steps for the next sweep; column 64 repeats
  // column 0, so that 32 columns from an odd place on lie in one piece
  constexpr int RING = (2 * BND + 1) * BLD;
  __shared__ double ring[K > 1 ? K - 1 : 1][CP][K > 1 ? RING : 1];
  __shared__ double yz[K][CP][4][2 * BND], xc[K][CP][BND];  // y and z of a wave, side by side
  // the same values from each of a sweep's waves
  __shared__ __align__(16) double vb[K][CP][BND], ub[K][CP][BND], gb[K][CP][BND];
  __shared__ int tick;
  const int n = g.n, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 8), wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  const int r = lane & 31, h = lane >> 5, j0 = (2 * wave + h) * CNC;
  const int ngroup = (n + K - 1) / K;
  const bool first = wave == 0 && h == 0;  // lanes that hold column 0
  const bool lead = (tid & 255) == 0;
  const size_t plane = (size_t)BLD * (n + BPAD);
  // places in the band (bytes from the step's first column): entry (r, j0 + q)
  // of D below the diagonal at ob + QS q, of C CS further; D mirrored at od[q]
  constexpr unsigned QS = 8 * (BLD - 1), CS = 8 * BND;
  const unsigned ob = 8 * (r + (BLD - 1) * j0);
  unsigned od[CNC];
#pragma unroll
  for (int q = 0; q < CNC; q++) {
    const int j = j0 + q;
    od[q] = 8 * (r >= j ? r + (BLD - 1) * j : j + (BLD - 1) * r);
  }
  // what no sweep writes there (entry (31, j < 31) of the next sweep's C) is zero
  if constexpr (K > 1)
    for (int i = tid; i < (K - 1) * CP * RING; i += 256 * K) (&ring[0][0][0])[i] = 0.0;
  // one work-item takes the ticket; a barrier stands on both sides of it, so
  // that no lane runs ahead with the old one
  auto ticket = [&]() {
    return __hip_atomic_fetch_add(g.prog + n, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (tid == 0) tick = ticket();
  __syncthreads();
  int grp = __builtin_amdgcn_readfirstlane(tick);
  while (grp < ngroup) {
    const int s = grp * K + w;
    // steps of the group's first sweep, and one of zeros
    const int nst = (n - 1 - grp * K + BND - 1) / BND + 1, ntick = nst + 2 * (K - 1);
    auto flag = [&]() { return grp > 0 ? agent_ld(g.prog + grp - 1) : CHASE_DONE; };
    auto wait = [&](int need) {
      while (__builtin_amdgcn_readfirstlane(flag()) < need) __builtin_amdgcn_s_sleep(1);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
    };
    double dr[CNC], di[CX ? CNC : 1], cr[CNC], ci[CX ? CNC : 1];    // D and C of the step
    double pd[CNC], pdi[CX ? CNC : 1], pc[CNC], pci[CX ? CNC : 1];  // of the next one (first sweep)
    double vj[CNC], vji[CX ? CNC : 1];                              // v at this lane's columns
    double vr = 0.0, vi = 0.0, tr = 0.0, ti = 0.0;                  // v(r) and tau of the step's reflector
    int done = 0;                                                   // steps to publish (last sweep)
    int seen = 0;                                                   // progress of the group before (first sweep)
    // raw D and C of the step whose rows start at c0, from the band
    auto fetch = [&](int c0) {
      const double *b = g.ab + (size_t)BLD * c0;
#pragma unroll
      for (int q = 0; q < CNC; q++) {
        pd[q] = agent_ld(byte_at(b, od[q]));
        pc[q] = agent_ld(byte_at(b, ob) + (CS + QS * q) / 8);
        if (CX) {
          pdi[q] = agent_ld(byte_at(b + plane, od[q]));
          pci[q] = agent_ld(byte_at(b + plane, ob) + (CS + QS * q) / 8);
        }
      }
    };
    // the reflector of x (rows c1 + r), its sum of squares below the first
    // known: v and tau; v to this lane's columns, v and tau to memory
    auto reflect = [&](int c1, int t1, double x, double x2, double ss) {
      const Reflector f = larfg<CX>(lane_value(x, 0), CX ? lane_value(x2, 0) : 0.0, ss);
      vr = r == 0 ? 1.0 : (CX ? fma(f.sr, x, -(f.si * x2)) : f.sr * x);
      if (CX) vi = r == 0 ? 0.0 : fma(f.sr, x2, f.si * x);
      tr = f.tr;
      ti = f.ti;
      if (h == 0) {
        vb[w][0][r] = vr;
        if (CX) vb[w][CP - 1][r] = vi;
      }
      if (first && s < n - 1 && c1 + r < n) {
        const size_t o = (size_t)c1 + (size_t)n * s;
        (g.V2r + o)[r] = vr;
        if (CX) (g.V2i + o)[r] = vi;
        if (r == 0) {
          const size_t o2 = (size_t)t1 * n + s;
          g.tau2[o2] = tr;
          if (CX) g.tau2[g.ntau2 + o2] = ti;
        }
      }
      return f.beta;
    };
    for (int k = -1; k < ntick; k++) {
      const int t = k - 2 * w, c0 = s + 1 + BND * t;
      const bool act = t >= 0 && t < nst;
      if (act) {
        if (w > 0) {
          // the columns that the sweep before left, one further on
          const double *b = ring[w > 0 ? w - 1 : 0][0] + ((t & 1) * BND + 1) * BLD;
          const double *b2 = ring[w > 0 ? w - 1 : 0][CP - 1] + ((t & 1) * BND + 1) * BLD;
#pragma unroll
          for (int q = 0; q < CNC; q++) {
            dr[q] = *byte_at(b, od[q]);
            cr[q] = byte_at(b, ob)[(CS + QS * q) / 8];
            if (CX) {
              di[q] = *byte_at(b2, od[q]);
              ci[q] = byte_at(b2, ob)[(CS + QS * q) / 8];
            }
          }
        } else {
          // C's last row holds one entry, in its last column; what memory has
          // for the others is older than the bulge
#pragma unroll
          for (int q = 0; q < CNC; q++) {
            const bool okc = r < BND - 1 || j0 + q == BND - 1;
            dr[q] = pd[q];
            cr[q] = okc ? pc[q] : 0.0;
            if (CX) {
              di[q] = pdi[q];
              ci[q] = okc ? pci[q] : 0.0;
            }
          }
        }
        if (CX)
#pragma unroll
          for (int q = 0; q < CNC; q++) di[q] = r < j0 + q ? -di[q] : di[q];
        if (first) {
          xc[w][0][r] = cr[0];
          if (CX) xc[w][CP - 1][r] = ci[0];
        }
        // y = D v, z = C v: this wave's eight columns
        double yr = 0.0, yi = 0.0, zr = 0.0, zi = 0.0;
#pragma unroll
        for (int q = 0; q < CNC; q++) {
          vj[q] = vb[w][0][j0 + q];
          if (CX) vji[q] = vb[w][CP - 1][j0 + q];
          yr = fma(dr[q], vj[q], yr);
          zr = fma(cr[q], vj[q], zr);
          if (CX) {
            yr = fma(-di[q], vji[q], yr);
            yi = fma(di[q], vj[q], fma(dr[q], vji[q], yi));
            zr = fma(-ci[q], vji[q], zr);
            zi = fma(ci[q], vj[q], fma(cr[q], vji[q], zi));
          }
        }
        // lanes of the lower half take y, of the upper half z
        yz[w][0][wave][lane] = swap_sum<32>(yr, zr);
        if (CX) yz[w][CP - 1][wave][lane] = swap_sum<32>(yi, zi);
      }
      if (done) vm_drain();
      __syncthreads();
      if (done && lead) agent_st(g.prog + grp, done);
      done = 0;
      if (w == 0 && t + 1 < nst) {
        if (__builtin_amdgcn_readfirstlane(seen) < t + 3) wait(t + 3);
        fetch(c0 + BND);
        seen = flag();
      }
      if (act) {
        double a = 0.0, a2 = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          a += yz[w][0][q][lane];
          if (CX) a2 += yz[w][CP - 1][q][lane];
        }
        double yr, zr, yi = 0.0, zi = 0.0;
        swap_halves(a, yr, zr);
        if (CX) swap_halves(a2, yi, zi);
        // C's first column after C <- C - tau z v^H (v(0) = 1)
        const double tzr = CX ? fma(tr, zr, -(ti * zi)) : tr * zr, tzi = CX ? fma(tr, zi, ti * zr) : 0.0;
        const double x = xc[w][0][r] - tzr, x2 = CX ? xc[w][CP - 1][r] - tzi : 0.0;
        // v^H y in the lower half, the new column's sum of squares in the upper
        const double py = CX ? fma(vr, yr, vi * yi) : vr * yr;
        const double px = r > 0 ? (CX ? fma(x, x, x2 * x2) : x * x) : 0.0;
        const double sums = sum32(h ? px : py);
        const double p = lane_value(sums, 0), ss = lane_value(sums, 32);
        // u = tau y - 1/2 |tau|^2 (v^H y) v;  D <- D - u v^H - v u^H
        const double hp = 0.5 * p * (CX ? fma(tr, tr, ti * ti) : tr * tr);
        const double ur = fma(-hp, vr, CX ? fma(tr, yr, -(ti * yi)) : tr * yr);
        const double ui = CX ? fma(-hp, vi, fma(tr, yi, ti * yr)) : 0.0;
        if (h == 0) {
          ub[w][0][r] = ur;
          if (CX) ub[w][CP - 1][r] = ui;
        }
#pragma unroll
        for (int q = 0; q < CNC; q++) {
          if (CX) {
            cr[q] = fma(-tzi, vji[q], fma(-tzr, vj[q], cr[q]));
            ci[q] = fma(tzr, vji[q], fma(-tzi, vj[q], ci[q]));
            dr[q] = fma(-ui, vji[q], fma(-ur, vj[q], dr[q]));
            di[q] = fma(ur, vji[q], fma(-ui, vj[q], di[q]));
          } else {
            cr[q] = fma(-tzr, vj[q], cr[q]);
            dr[q] = fma(-ur, vj[q], dr[q]);
          }
        }
        const double v0r = vr, v0i = vi;
        // reflector of the next rows, applied to C from the left
        const double beta = reflect(c0 + BND, t + 1, x, x2, ss);
        double tq[CP * CNC];
#pragma unroll
        for (int q = 0; q < CNC; q++) {
          tq[q] = CX ? fma(vr, cr[q], vi * ci[q]) : vr * cr[q];
          if (CX) tq[CP * CNC - CNC + q] = fma(vr, ci[q], -(vi * cr[q]));
        }
        const double gs = half_sums<CP * CNC>(tq, lane);
        constexpr int SH = CX ? 2 : 3;
        if (!(r & ((1 << SH) - 1))) gb[w][r >> 4 & (CP - 1)][j0 + ((r >> SH) & (CNC - 1))] = gs;
        wave_sync();
#pragma unroll
        for (int q = 0; q < CNC; q++) {
          const double uj = ub[w][0][j0 + q];
          if (CX) {
            const double uji = ub[w][CP - 1][j0 + q];
            dr[q] = fma(-v0i, uji, fma(-v0r, uj, dr[q]));
            di[q] = fma(v0r, uji, fma(-v0i, uj, di[q]));
            if (r == j0 + q) di[q] = 0.0;
          } else {
            dr[q] = fma(-v0r, uj, dr[q]);
          }
        }
        // conj(tau) v
        const double wr = CX ? fma(tr, vr, ti * vi) : tr * vr, wi = CX ? fma(tr, vi, -(ti * vr)) : 0.0;
#pragma unroll
        for (int q = 0; q < CNC; q++) {
          const double gr = gb[w][0][j0 + q];
          if (CX) {
            const double gi = gb[w][CP - 1][j0 + q];
            cr[q] = fma(wi, gi, fma(-wr, gr, cr[q]));
            ci[q] = fma(-wi, gr, fma(-wr, gi, ci[q]));
          } else {
            cr[q] = fma(-wr, gr, cr[q]);
          }
        }
        if (first) {  // column 0 is (beta, 0, ..)
          cr[0] = r == 0 ? beta : 0.0;
          if (CX) ci[0] = 0.0;
        }
        // leave the columns
        if (w == K - 1) {
          double *const b = byte_at(g.ab + (ptrdiff_t)BLD * c0, ob), *const b2 = byte_at(g.ab + plane + (ptrdiff_t)BLD * c0, ob);
#pragma unroll
          for (int q = 0; q < CNC; q++) {
            if (r >= j0 + q) {
              agent_st(b + QS / 8 * q, dr[q]);
              if (CX) agent_st(b2 + QS / 8 * q, di[q]);
            }
            agent_st(b + (CS + QS * q) / 8, cr[q]);
            if (CX) agent_st(b2 + (CS + QS * q) / 8, ci[q]);
          }
          done = t + 1;
        } else {
          double *const b = byte_at(ring[w < K - 1 ? w : 0][0] + (t & 1) * BND * BLD, ob);
          double *const b2 = byte_at(ring[w < K - 1 ? w : 0][CP - 1] + (t & 1) * BND * BLD, ob);
#pragma unroll
          for (int q = 0; q < CNC; q++) {
            if (r >= j0 + q) {
              b[QS / 8 * q] = dr[q];
              if (CX) b2[QS / 8 * q] = di[q];
            }
            b[(CS + QS * q) / 8] = cr[q];
            if (CX) b2[(CS + QS * q) / 8] = ci[q];
          }
          if (first && !(t & 1)) {
            b[2 * BND * BLD] = dr[0];
            b[2 * BND * BLD + BND] = cr[0];
            if (CX) {
              b2[2 * BND * BLD] = di[0];
              b2[2 * BND * BLD + BND] = ci[0];
            }
          }
        }
      } else if (t == -1) {
        // column s: d, e and the reflector of R_0
        const int o = 1 + r;
        double x, x2 = 0.0, dg;
        if (w == 0) {
          const double *b = g.ab + (size_t)BLD * s;
          x = agent_ld(b + o);
          if (CX) x2 = agent_ld(b + plane + o);
          dg = agent_ld(b);
          vm_drain();  // here, so that no later step waits for registers of these loads
        } else {
          x = ring[w > 0 ? w - 1 : 0][0][o];
          if (CX) x2 = ring[w > 0 ? w - 1 : 0][CP - 1][o];
          dg = ring[w > 0 ? w - 1 : 0][0][0];
        }
        const double beta = reflect(s + 1, 0, x, x2, sum32(r > 0 ? (CX ? fma(x, x, x2 * x2) : x * x) : 0.0));
        if (lead && s < n) {
          g.d[s] = dg;
          if (s < n - 1) g.e[s] = beta;
        }
      }
      __syncthreads();
    }
    vm_drain();
    __syncthreads();
    if (tid == 0) {
      agent_st(g.prog + grp, CHASE_DONE);
      tick = ticket();
    }
    __syncthreads();
    grp = __builtin_amdgcn_readfirstlane(tick);
  }
}

// ------------------------------------------------------------------ 3. Q2 times vectors
// The reflectors of BND consecutive sweeps at one step are a block I - V T V^H
// on 2 BND - 1 rows (V a parallelogram): k_sb_frag forms V and -V T of every
// block in the order in which k_sb_q2's lanes read them as MFMA operands.  The
// groups are counted from the last one, which is applied first: group gi has
// gi + 1 blocks, and those of the groups from ga on are held at a time.
__host__ __device__ constexpr size_t frag_block(int ga, int gi, int t)
{
  return ((size_t)gi * (gi + 1) - (size_t)ga * (ga + 1)) / 2 + t;
}
constexpr int FRAG = 4096;  // doubles of a block per plane: 32 + 32 operand fragments of 64

template <bool CX>
__global__ __launch_bounds__(256) void k_sb_frag(SbArgs g, int ntg, int ga, int nsync)
{
  __shared__ double v[CX ? 2 : 1][64][BND + 1], gm[CX ? 2 : 1][BND][BND + 1], tm[CX ? 2 : 1][BND][BND + 1];
  const int gi = ga + blockIdx.y, gr = ntg - 1 - gi, t = blockIdx.x, tid = threadIdx.x, n = g.n;
  // the ticket and progress words of k_sb_q2
  for (size_t i = ((size_t)blockIdx.y * gridDim.x + t) * 256 + tid; i < (size_t)nsync;
       i += (size_t)gridDim.y * gridDim.x * 256)
    g.q2sync[i] = 0;
  if (t > gi) return;
  const int s0 = gr * BND, w0 = s0 + 1 + BND * t;
  for (int e = tid; e < 64 * BND; e += 256) {
    const int x = e & 63, i = e >> 6;
    const bool in = x >= i && x < i + BND && w0 + x < n && s0 + i <= n - 2;
    const size_t o = in ? (size_t)(w0 + x) + (size_t)n * (s0 + i) : 0;
    v[0][x][i] = in ? g.V2r[o] : 0.0;
    if (CX) v[1][x][i] = in ? g.V2i[o] : 0.0;
  }
  for (int e = tid; e < BND * BND; e += 256) {
    tm[0][e & 31][e >> 5] = 0.0;
    if (CX) tm[1][e & 31][e >> 5] = 0.0;
  }
  __syncthreads();
  {
    const int a = tid & 31;
    double sr[4] = {0.0, 0.0, 0.0, 0.0}, si[4] = {0.0, 0.0, 0.0, 0.0};
    for (int x = 0; x < 64; x++) {
      const double ar = v[0][x][a], ai = CX ? v[1][x][a] : 0.0;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int b = (tid >> 5) + 8 * q;
        const double br = v[0][x][b];
        if (CX) {
          const double bi = v[1][x][b];
          sr[q] += ar * br + ai * bi;
          si[q] += ar * bi - ai * br;
        } else {
          sr[q] += ar * br;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      gm[0][a][(tid >> 5) + 8 * q] = sr[q];
      if (CX) gm[1][a][(tid >> 5) + 8 * q] = si[q];
    }
  }
  __syncthreads();
  if (tid < 64) {
    const int lane = tid & 31;
    for (int i = 0; i < BND; i++) {
      const bool in = s0 + i <= n - 2 && w0 + i < n;
      const size_t o = in ? (size_t)t * n + s0 + i : 0;
      const double tr = in ? g.tau2[o] : 0.0, ti = CX && in ? g.tau2[g.ntau2 + o] : 0.0;
      double ar = 0.0, ai = 0.0;
      for (int q = 0; q < i; q++) {
        const double a = tm[0][lane][q], b = gm[0][q][i];
        if (CX) {
          const double a2 = tm[1][lane][q], b2 = gm[1][q][i];
          ar += a * b - a2 * b2;
          ai += a * b2 + a2 * b;
        } else {
          ar += a * b;
        }
      }
      if (tid < 32 && lane <= i) {
        tm[0][lane][i] = lane < i ? -(CX ? tr * ar - ti * ai : tr * ar) : tr;
        if (CX) tm[1][lane][i] = lane < i ? -(tr * ai + ti * ar) : ti;
      }
      wave_sync();
    }
  }
  __syncthreads();
  double *out = g.frag + frag_block(ga, gi, t) * FRAG * (CX ? 2 : 1);
  // V: fragment (w, mt, k): lane (l, q) holds row 16 w + 4 q + k, column 16 mt + l
  for (int e = tid; e < 2048; e += 256) {
    const int lane = e & 63, f = e >> 6, k = f & 3, mt = (f >> 2) & 1, w = f >> 3;
    const int x = 16 * w + 4 * (lane >> 4) + k, c = 16 * mt + (lane & 15);
    out[e] = v[0][x][c];
    if (CX) out[FRAG + e] = v[1][x][c];
  }
  // -V T: fragment (w, s): lane (l, q) holds row 16 w + 4 (l % 4) + l / 4, column 4 s + q
  for (int e = tid; e < 2048; e += 256) {
    const int lane = e & 63, f = e >> 6, s = f & 7, w = f >> 3, l = lane & 15;
    const int x = 16 * w + 4 * (l & 3) + (l >> 2), c = 4 * s + (lane >> 4);
    double ar = 0.0, ai = 0.0;
    for (int q = 0; q <= c; q++) {
      ar += v[0][x][q] * tm[0][q][c];
      if (CX) {
        ar -= v[1][x][q] * tm[1][q][c];
        ai += v[0][x][q] * tm[1][q][c] + v[1][x][q] * tm[0][q][c];
      }
    }
    out[2048 + e] = -ar;
    if (CX) out[FRAG + 2048 + e] = -ai;
  }
}

// rows of the blocked copy of Z (the last window reaches past the matrix)
__host__ __device__ constexpr size_t q2_rows(int n) { return (size_t)n + 2 * BND; }

// Z <- Q2 Z for the groups ga .. gb - 1.  A task is one group of sweeps on a slab of 16 columns of Z: its
// blocks slide down the rows.  A wave holds 16 of the window's 64 rows as MFMA
// accumulators (lane (l, q): column l, rows 4 q + k in item k), which are at
// once the operand of V^H Z; the four partial V^H Z meet in LDS.  Between the
// groups Z lives in a copy with 16 columns side by side, row after row, so that
// such an item is four full lines; the first group that touches a row takes it
// from Z, the last one puts it back.  The window
// moves by 32 rows, so two waves keep their rows and the other two store
// theirs and take the next 32.  Rows and operands are loaded a step ahead and
// rows stored a step late, so that no step waits for memory it has just asked.
//
// The groups of a slab follow each other (the last group first) a few steps
// apart, which keeps the chip busy where there are few slabs: work-groups take
// tasks in order from a ticket, so the group that a task waits for has started
// before it, and every Q2_FLAG steps a task publishes how many it has done.
constexpr int Q2_FLAG = 4;
// From this many columns on a step's rate counts and not its length: two
// work-groups a CU instead of one (complex N = 10886, m = 2177 205 -> 169 ms for
// the whole back-transform; N = 1951, m = 195 6.2 -> 6.6 ms), and real tasks take
// two sets of columns, which halves what the operands' loads move (N = 5940,
// m = 1188 14.4 -> 13.4; N = 731, m = 88 0.87 -> 0.96 ms).
constexpr int Q2_WIDE = 512;

template <bool CX, int NC>
__global__ __launch_bounds__(256, 2) void k_sb_q2(SbArgs g, int ntg, int ga, int gb, int mcol,
                                                  double *__restrict__ Zr, double *__restrict__ Zi, int ldz)
{
  constexpr int CP = CX ? 2 : 1;
  __shared__ double yp[2][CP][NC][4][8][64];
  __shared__ int tick;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l = lane & 15, q4 = lane >> 4;
  const int n = g.n, nslab = (mcol + 16 * NC - 1) / (16 * NC), ntask = nslab * (gb - ga);
  int *const done = g.q2sync + 1;  // steps done of (group from ga, slab)
  const size_t zrows = q2_rows(n), zplane = zrows * (size_t)nslab * NC * 16;
  const int zo = 64 * q4 + l;  // this lane's place in four rows, 4 q4 rows on
  auto ticket = [&]() { return __hip_atomic_fetch_add(g.q2sync, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  if (tid == 0) tick = ticket();
  __syncthreads();
  int task = __builtin_amdgcn_readfirstlane(tick);
  while (task < ntask) {
    const int q = task / nslab, slab = task - q * nslab, gi = ga + q, gr = ntg - 1 - gi, nt = gi + 1;
    double *const zb = g.zb + (size_t)slab * NC * 16 * zrows;
    int seen = q == 0 ? CHASE_DONE : 0;
    // rows of window t are final once the group after this one has done step
    // t; its progress is read a step ahead
    int peek = 0;
    auto progress = [&]() { return q > 0 ? agent_ld(done + (size_t)(q - 1) * nslab + slab) : CHASE_DONE; };
    auto ready = [&](int t) {
      while (seen < t + 1) {
        seen = __builtin_amdgcn_readfirstlane(progress());
        if (seen < t + 1) __builtin_amdgcn_s_sleep(1);
      }
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
    };
    // four rows of each set of columns
    struct Rows {
      d4 r[NC], i[CX ? NC : 1];
    };
    // rows that no group has touched yet, from Z
    auto zfirst = [&](int row0, Rows &z) {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const int col = (slab * NC + c) * 16 + l;
        const size_t zc = (size_t)ldz * min(col, mcol - 1);
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int row = row0 + 4 * q4 + k;
          const size_t o = zc + min(row, n - 1);
          const bool ok = col < mcol && row < n;
          const double x = Zr[o], y = CX ? Zi[o] : 0.0;
          z.r[c][k] = ok ? x : 0.0;
          if (CX) z.i[c][k] = ok ? y : 0.0;
        }
      }
    };
    auto zload = [&](int row0, Rows &z) {
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const double *p = zb + (size_t)c * 16 * zrows + 16 * (size_t)(row0 + k);
          z.r[c][k] = agent_ld(p + zo);
          if (CX) z.i[c][k] = agent_ld(p + zplane + zo);
        }
    };
    auto zstore = [&](int row0, const Rows &z) {
      if (gr > 0) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            double *p = zb + (size_t)c * 16 * zrows + 16 * (size_t)(row0 + k);
            agent_st(p + zo, z.r[c][k]);
            if (CX) agent_st(p + zplane + zo, z.i[c][k]);
          }
        return;
      }
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int col = (slab * NC + c) * 16 + l, row = row0 + 4 * q4 + k;
          if (col < mcol && row < n) {
            Zr[(size_t)ldz * col + row] = z.r[c][k];
            if (CX) Zi[(size_t)ldz * col + row] = z.i[c][k];
          }
        }
    };
    struct Ops {
      double a[8], t[8], ai[CX ? 8 : 1], ti[CX ? 8 : 1];
    };
    auto fetch = [&](Ops &o, int t, int role) {
      const double *f = g.frag + frag_block(ga, gi, t) * FRAG * CP + (size_t)role * 512 + lane;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        o.a[k] = f[k * 64];
        o.t[k] = f[2048 + k * 64];
        if (CX) {
          o.ai[k] = f[FRAG + k * 64];
          o.ti[k] = f[FRAG + 2048 + k * 64];
        }
      }
    };
    int role = wave, w0 = gr * BND + 1, pend = -1;  // pend: first row of the tile to be stored
    Rows z, st;
    ready(0);
    if (gi == 0 || role < 2) zfirst(w0 + 16 * role, z);
    else zload(w0 + 16 * role, z);
    Ops oa, ob;
    fetch(oa, 0, role);
    auto step = [&](const Ops &o, Ops &next, int t) {
      // what the last step asked for has come; then, in this order so that no
      // wait below includes a younger access: rows, operands, stores
      vm_drain();
      seen = max(seen, __builtin_amdgcn_readfirstlane(peek));
      const bool more = t + 1 < nt, leave = role < 2 && more;
      Rows nx;
      if (leave) {
        ready(t + 1);
        zload(w0 + 64 + 16 * role, nx);
      }
      peek = progress();
      fetch(next, more ? t + 1 : t, (role + 2) & 3);
      if (pend >= 0) zstore(pend, st);
      // partial V^H Z over this wave's rows
      d4 yr[NC][2], yi[NC][2];
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
          yr[c][mt] = d4{0.0, 0.0, 0.0, 0.0};
          yi[c][mt] = d4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
      for (int k = 0; k < 4; k++) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int mt = 0; mt < 2; mt++) {
            yr[c][mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[4 * mt + k], z.r[c][k], yr[c][mt], 0, 0, 0);
            if (CX) yi[c][mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[4 * mt + k], z.i[c][k], yi[c][mt], 0, 0, 0);
          }
        if (CX)
#pragma unroll
          for (int c = 0; c < NC; c++)
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
              yr[c][mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.ai[4 * mt + k], z.i[c][k], yr[c][mt], 0, 0, 0);
              yi[c][mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(-o.ai[4 * mt + k], z.r[c][k], yi[c][mt], 0, 0, 0);
            }
      }
      mfma_settle();
      const int par = t & 1;
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            yp[par][0][c][role][4 * mt + k][lane] = yr[c][mt][k];
            if (CX) yp[par][CP - 1][c][role][4 * mt + k][lane] = yi[c][mt][k];
          }
      const bool flag = t % Q2_FLAG == Q2_FLAG - 1;
      if (flag) vm_drain();  // the tiles of the steps before this one are stored
      __syncthreads();
      if (flag && tid == 0) agent_st(done + (size_t)q * nslab + slab, t);
      // Z -= (V T) (V^H Z), for one real set of columns in two accumulator chains
      constexpr bool TWO = !CX && NC == 1;
      d4 z2 = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 8; s++) {
        double a[NC], b[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
          a[c] = yp[par][0][c][0][s][lane];
          if (CX) b[c] = yp[par][CP - 1][c][0][s][lane];
#pragma unroll
          for (int w = 1; w < 4; w++) {
            a[c] += yp[par][0][c][w][s][lane];
            if (CX) b[c] += yp[par][CP - 1][c][w][s][lane];
          }
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
          if (TWO && (s & 1)) z2 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.t[s], a[c], z2, 0, 0, 0);
          else z.r[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.t[s], a[c], z.r[c], 0, 0, 0);
          if (CX) z.i[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.t[s], b[c], z.i[c], 0, 0, 0);
        }
        if (CX)
#pragma unroll
          for (int c = 0; c < NC; c++) {
            z.r[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(-o.ti[s], b[c], z.r[c], 0, 0, 0);
            z.i[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.ti[s], a[c], z.i[c], 0, 0, 0);
          }
      }
      mfma_settle();
      if (TWO) z.r[0] += z2;
      pend = -1;
      if (more) {
        if (leave) {
          pend = w0 + 16 * role;
          st = z;
          z = nx;
        }
        role = (role + 2) & 3;
        w0 += BND;
      }
    };
    for (int t = 0; t < nt; t += 2) {
      step(oa, ob, t);
      if (t + 1 < nt) step(ob, oa, t + 1);
    }
    zstore(w0 + 16 * role, z);
    vm_drain();
    __syncthreads();
    if (tid == 0) {
      agent_st(done + (size_t)q * nslab + slab, CHASE_DONE);
      tick = ticket();
    }
    __syncthreads();
    task = __builtin_amdgcn_readfirstlane(tick);
  }
}

// ------------------------------------------------------------------ host side
static size_t up32(size_t x) { return (x + 31) & ~(size_t)31; }

static int av_slices(int m, int &slab)
{
  const int tiles = (m + 63) / 64;
  int z = std::max(1, std::min(1024 / tiles, tiles));
  slab = (tiles + z - 1) / z;
  return (tiles + slab - 1) / slab;
}

size_t sb_doubles(int n, int cplx, size_t *ints)
{
  const size_t cp = cplx ? 2 : 1, tiles = (n + 63) / 64, nblk = (n + QR_ROWS - 1) / QR_ROWS;
  const size_t ntg = (n - 1 + BND - 1) / BND;
  if (ints) *ints = (size_t)n + 1 + 8;
  return up32(std::max(tiles, std::min((size_t)1024, tiles * tiles)) * 64 * BND * cp) + up32((size_t)n * BND * cp) +
         up32((size_t)(n + 31) / 32 * BND * BND * cp) + 3 * up32(BND * BND * cp) + up32((nblk + 1) * BND * BND * cp) + up32((size_t)BLD * (n + BPAD) * cp) +
         up32((size_t)n * (ntg + 1) * cp);
}

// Application of Q2: its workspace holds the vectors in their blocked order, the
// ticket and progress words, and the operands of as many groups as find room.
// All operands together take 2 n^2 elements, as much as two matrices; so where
// they are more than Q2_OPS, a range of groups at a time is formed and applied
// (every range waits for the one before).  The workspace is the inverse
// iteration's (5 n m doubles), whose factors are dead by then.  1 GiB: all at
// once, 1, 1/2 and 1/4 GiB take 84, 86, 89, 91 ms at complex N = 10880, m =
// 2176 (3.8 GB of operands), 20.0, 20.8, 21.3, 21.8 ms at N = 6559, m = 1311
// and 5.7, 5.7, 6.0, 6.1 ms at real N = 5951, m = 1190.
constexpr size_t Q2_OPS = (size_t)1 << 27;  // doubles

struct Q2Space {
  size_t zb, words, group, all;  // vectors, words (in doubles), operands of the longest group and of all
};
static Q2Space q2_space(int n, size_t m, int cplx)
{
  const size_t ntg = (n - 1 + BND - 1) / BND, cp = cplx ? 2 : 1;
  return {q2_rows(n) * ((m + 31) / 32 * 32) * cp, up32((m + 15) / 16 * ntg / 2 + 1), ntg * FRAG * cp,
          ntg * (ntg + 1) / 2 * FRAG * cp};
}
// doubles that the operands may take; W2K_TEST_Q2_OPERANDS (tests only) sets fewer
static size_t q2_ops(const Q2Space &q, size_t room)
{
  const char *e = std::getenv("W2K_TEST_Q2_OPERANDS");
  if (e) room = std::min(room, (size_t)std::atoll(e));
  return std::min(q.all, std::max(q.group, room));
}

size_t sb_q2_doubles(int n, size_t m, int cplx)
{
  const Q2Space q = q2_space(n, m, cplx);
  return q.zb + q.words + q2_ops(q, Q2_OPS);
}

int sb_buffers(Ctx &c, SbArgs &g, int n, int cplx)
{
  size_t ni = 0;
  int rc;
  const size_t nd = sb_doubles(n, cplx, &ni);
  if ((rc = c.w_sb.alloc(nd)) || (rc = c.w_sbi.alloc(ni))) return rc;
  const size_t cp = cplx ? 2 : 1, tiles = (n + 63) / 64, nblk = (n + QR_ROWS - 1) / QR_ROWS;
  const size_t ntg = (n - 1 + BND - 1) / BND;
  double *p = c.w_sb.p;
  auto take = [&](size_t k) {
    double *q = p;
    p += up32(k);
    return q;
  };
  g.n = n;
  g.part = take(std::max(tiles, std::min((size_t)1024, tiles * tiles)) * 64 * BND * cp);
  g.Yr = take((size_t)n * BND * cp);
  g.Yi = g.Yr + (size_t)n * BND;
  g.spart = take((size_t)(n + 31) / 32 * BND * BND * cp);
  g.T = take(BND * BND * cp);
  g.G = take(BND * BND * cp);
  g.S = take(BND * BND * cp);
  g.exch = take((nblk + 1) * BND * BND * cp);
  g.ab = take((size_t)BLD * (n + BPAD) * cp);
  g.tau2 = take((size_t)n * (ntg + 1) * cp);
  g.ntau2 = (size_t)n * (ntg + 1);
  g.prog = c.w_sbi.p;
  g.sync = c.w_sbi.p + n + 1;
  return 0;
}

// events around every k_sb_av launch while kernel timing is on (carried by the
// dispatch itself, so that a duration is the kernel's own)
int sb_take_times(Ctx &c, hipStream_t s, int n)
{
  if (!c.ktime) return 0;
  W2K_HIP(hipStreamSynchronize(s));
  double tot = 0.0;
  int cnt = 0;
  for (int j0 = 0; n - j0 - BND >= 2; j0 += BND) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, c.kev[2 * cnt], c.kev[2 * cnt + 1]) != hipSuccess) {
      (void)hipGetLastError();
      break;
    }
    tot += ms;
    cnt++;
  }
  c.last_ms[10] = tot;
  c.last_ms[11] = cnt;
  return 0;
}

template <bool CX>
static int reduce(Ctx &c, hipStream_t s, SbArgs &g)
{
  const int n = g.n, cp = CX ? 2 : 1;
  int rc;
  const bool kt = c.ktime != 0;
  while (kt && c.kev.size() < (size_t)2 * (n / BND + 1)) {
    hipEvent_t e;
    W2K_HIP(hipEventCreate(&e));
    c.kev.push_back(e);
  }
  int panel = 0;
  auto nexch = [&](int m) { return (size_t)((m + QR_ROWS - 1) / QR_ROWS + 1) * BND * BND * cp; };
  if (n - BND >= 2) {
    const size_t k = nexch(n - BND);
    hipLaunchKernelGGL(k_sb_reset, dim3((unsigned)((k + 255) / 256)), dim3(256), 0, s, g.exch, k, g.sync);
    W2K_STAGE(s, "k_sb_reset");
  }
  for (int j0 = 0; n - j0 - BND >= 2; j0 += BND) {
    const int r0 = j0 + BND, m = n - r0;
    hipLaunchKernelGGL((k_sb_qr<CX>), dim3((m + QR_ROWS - 1) / QR_ROWS), dim3(QR_ROWS), 0, s, g, j0);
    W2K_STAGE(s, "k_sb_qr");
    int slab = 1;
    const int nz = av_slices(m, slab), tiles = (m + 63) / 64;
    const int nwg = (m + 31) / 32;
    if (kt)
      hipExtLaunchKernelGGL((k_sb_av<CX>), dim3(tiles + 1, nz), dim3(256), 0, s, c.kev[2 * panel], c.kev[2 * panel + 1],
                            0, g, r0, slab, tiles * 64);
    else hipLaunchKernelGGL((k_sb_av<CX>), dim3(tiles + 1, nz), dim3(256), 0, s, g, r0, slab, tiles * 64);
    panel++;
    W2K_STAGE(s, "k_sb_av");
    hipLaunchKernelGGL((k_sb_y<CX>), dim3(nwg), dim3(256), 0, s, g, r0, nz, tiles * 64);
    W2K_STAGE(s, "k_sb_y");
    hipLaunchKernelGGL(k_sb_s, dim3(BND * cp), dim3(256), 0, s, g, nwg, BND * BND * cp);
    W2K_STAGE(s, "k_sb_s");
    hipLaunchKernelGGL((k_sb_w<CX>), dim3(nwg), dim3(256), 0, s, g, r0, nexch(m));
    W2K_STAGE(s, "k_sb_w");
    // A(r0:n, r0:n) -= [V W] [W V]^H, lower triangle
    const size_t o = (size_t)r0 + (size_t)g.lda * r0, ow = (size_t)n * BND + r0;
    if (CX)
      rc = zgemm_fused(s, 'N', 'C', m, m, 2 * BND, -1.0, g.Pr + r0, g.Pi + r0, n, g.Pr + ow, g.Pi + ow, n, 1.0, g.ar + o,
                       g.ai + o, g.lda, 1);
    else rc = dgemm(s, 'N', 'T', m, m, 2 * BND, -1.0, g.Pr + r0, n, g.Pr + ow, n, 1.0, g.ar + o, g.lda, 1);
    if (rc) return rc;
  }
  hipLaunchKernelGGL((k_sb_band<CX>), dim3((n + BPAD + 3) / 4), dim3(4 * BLD), 0, s, g);
  W2K_STAGE(s, "k_sb_band");
  // groups in flight: one per 2 K + 2 steps
  constexpr int K = CX ? CHASE_KZ : CHASE_KD;
  const int nwg = std::min(256, n / (BND * (2 * K + 2)) + 2);
  hipLaunchKernelGGL((k_sb_chase<CX, K>), dim3(nwg), dim3(256 * K), 0, s, g);
  W2K_STAGE(s, "k_sb_chase");
  return 0;
}

int sb_reduce(Ctx &c, hipStream_t s, SbArgs &g, int cplx)
{
  // W2K_TEST_QR_GROUPS (tests only): that many work-groups share a panel, as if
  // the others had come late
  const char *cap = std::getenv("W2K_TEST_QR_GROUPS");
  if (cap) g.qr_cap = std::max(1, std::atoi(cap));
  return cplx ? reduce<true>(c, s, g) : reduce<false>(c, s, g);
}

template <bool CX>
static int apply_q2(hipStream_t s, SbArgs &g, const Q2Space &q, size_t ops, int m, double *Zr, double *Zi, int ldz)
{
  const int ntg = (g.n - 1 + BND - 1) / BND, nc = !CX && m >= Q2_WIDE ? 2 : 1, nslab = (m + 16 * nc - 1) / (16 * nc);
  for (int ga = 0, gb; ga < ntg; ga = gb) {
    gb = ga + 1;
    while (gb < ntg && frag_block(ga, gb + 1, 0) * FRAG * (CX ? 2 : 1) <= ops) gb++;
    const int ntask = nslab * (gb - ga), nwg = std::min(ntask, m >= Q2_WIDE ? 512 : 256);
    hipLaunchKernelGGL((k_sb_frag<CX>), dim3(gb, gb - ga), dim3(256), 0, s, g, ntg, ga, ntask + 1);
    W2K_STAGE(s, "k_sb_frag");
    if (nc == 2)
      hipLaunchKernelGGL((k_sb_q2<false, 2>), dim3(nwg), dim3(256), 0, s, g, ntg, ga, gb, m, Zr, Zi, ldz);
    else hipLaunchKernelGGL((k_sb_q2<CX, 1>), dim3(nwg), dim3(256), 0, s, g, ntg, ga, gb, m, Zr, Zi, ldz);
    W2K_STAGE(s, "k_sb_q2");
  }
  return 0;
}

int sb_apply_q2(Ctx &c, hipStream_t s, SbArgs &g, int cplx, int m, double *Zr, double *Zi, int ldz)
{
  if (g.n < 2 || m == 0) return 0;
  const Q2Space q = q2_space(g.n, m, cplx);
  if (c.w_fac.n < sb_q2_doubles(g.n, m, cplx)) return W2K_ESTATE;
  g.zb = c.w_fac.p;
  g.q2sync = reinterpret_cast<int *>(g.zb + q.zb);
  g.frag = g.zb + q.zb + q.words;
  const size_t ops = q2_ops(q, c.w_fac.n - q.zb - q.words);
  return cplx ? apply_q2<true>(s, g, q, ops, m, Zr, Zi, ldz) : apply_q2<false>(s, g, q, ops, m, Zr, Zi, ldz);
}

}  // namespace w2k
