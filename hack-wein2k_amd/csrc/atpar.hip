// ATPAR's radial part on the device (atpar.f:212-330, 470-561): the radial
// functions u_l(E_l), their energy derivatives and the local-orbital functions
// of every atom type by outward integration of the scalar-relativistic radial
// equation (OUTWIN, outwin.f:1-113), their boundary values and norms, and the
// non-spherical radial integrals VNS1..3 / VNS1LO..3LO (RINT13, rint13.f:1-64).
// The functions stay on the device for the adjoint with respect to V_LM(r).
//
// Arithmetic follows the reference step by step: OUTWIN's predictor-corrector
// over the logarithmic mesh r_k = RO exp(DH (k-1)), the normalisation by
// 1/sqrt(RINT13(u, u)), the energy derivative by the difference of the
// functions at E -+ DELE (DELE = 2e-3 Hartree, scaled by 0.25/DELE), its
// orthogonalisation to u, and RINT13's Simpson sum (as a weighted sum over the
// mesh).
#include <algorithm>
#include <cmath>
#include <tuple>
#include <vector>

#include "w2k_internal.h"

namespace w2k {

struct AtparArgs {
  int nat, nt, nslmax, lomax, jrid, lmaxd;
  int rel;
  const int *jrj;
  const double *ro, *dh, *zz, *vr;    // vr: [a][jrid], r V in Hartree
  const double *e;                     // [a][lmaxd] energies (Ry)
  const double *elo;                   // [a][LOMAXP]: energy of the LO radial function (Ry)
  const int *loor;                     // [a][LOMAXP]
  double *fn;                          // [a][l < nslmax][4][jrid]: A1, B1, AE1, BE1
  double *fnlo;                        // [a][l <= lomax][2][jrid]: A1LO, B1LO
  double *work;                        // [a][l][AT_ROWS][jrid]: A, B of OUTWIN per energy; weights
  double *out;                         // [a][l][6]: P, DP, PE, DPE, PEI, E used
  double *outlo;                       // [a][l][4]: PLO, DPLO, PI12LO, PE12LO
};

// OUTWIN (outwin.f:20-112) is a recurrence along the mesh.  All that its step
// needs besides the functions themselves is formed beforehand, for AT_CH mesh
// points and AT_NE energies at once: U and Y of outwin.f:73-80 (X = -DH) and
// 1 / DET, whose rounding error goes along: with one rounding more per point
// the difference of the functions at E -+ DELE would lose a digit's fraction.
constexpr int AT_NE = 4;    // energies E - DELE, E + DELE, E and the local orbital's
constexpr int AT_CH = 64;   // mesh points formed at a time
constexpr int AT_PF = 4;    // mesh points whose operands are read at a time
constexpr int AT_NC = 4;    // 1 / DET in two parts, U, Y
constexpr int AT_NT = 64 * (1 + AT_NE);
constexpr int AT_ROWS = 2 * AT_NE + 1;  // rows of an (atom, l): A and B of each energy, RINT13's weights

struct AtparShared {
  double __attribute__((aligned(16))) c[2][AT_CH + 2 * AT_PF][AT_NE][AT_NC];  // of this piece of the mesh and the next
  double f[2][2][AT_CH][AT_NE];  // A, B of this piece and the one before
  double red[2][AT_NT / 64][3];
  double end[2][AT_NE], norm[AT_NE];  // value and slope at the boundary; 1 / sqrt of the norm
};

// OUTWIN's coefficients at mesh point k; of the first three points A, B and
// their derivatives instead (outwin.f:49-60)
__device__ __forceinline__ void outwin_coef(bool rel, double v, double rnot, double dh, double eh, double fl, double z,
                                            int k, double *o)
{
  const double e = eh * 2.0, zz = z + z, c = rel ? 2.0 * 137.0359895 : 1.0e10;
  const double fllp1 = fl * (fl + 1.0);
  const double r = rnot * exp(dh * (double)k), drdi = dh * r;
  if (k < 3) {
    const bool bare = z < 0.9;
    const double aa = zz / c, s0 = sqrt(fllp1 + 1.0 - aa * aa);
#pragma unroll 1
    for (int q = 0; q < 2; q++) {
      const double s = !bare ? s0 : q == 0 ? fl + 1.0 : fl;
      const double f0 = q == 0 ? 1.0 : bare ? fl / c : (s0 - 1.0) / aa;
      o[q] = pow(r, s) * f0;
      o[2 + q] = drdi * o[q] * s / r;
    }
    return;
  }
  const double phi = (e - 2.0 * v / r) * drdi / c;
  const double u = drdi * c + phi, x = -dh;
  const double y = -fllp1 * x * x / u + phi;
  const double det = 64.0 / 9.0 - x * x + u * y, inv = 1.0 / det;
  o[0] = inv;
  o[1] = inv * fma(-det, inv, 1.0);
  o[2] = u;
  o[3] = y;
}

// RINT13 (rint13.f:28-62) as a weighted sum: weight of mesh point k (0-based)
__device__ __forceinline__ double rint13_w(double rnot, double dx, int jri, int k)
{
  const double r = rnot * exp(dx * (double)k);
  const int k0 = 2 - jri % 2;  // first point of weight 4
  double w = k == jri - 1 ? r * dx / 3.0 : k >= k0 ? ((k - k0) & 1 ? 2.0 : 4.0) * r * dx / 3.0 : 0.0;
  if (k == k0 - 1) w = r * dx / 3.0 + (k0 > 1 ? 0.5 * dx * r : 0.0);
  if (k == 0) w += rnot / 3.0 + (k0 > 1 ? 0.5 * dx * rnot : 0.0);
  return w;
}
// RINT13 leaves no sum at zero (rint13.f:37)
__device__ __forceinline__ double rint13_nonzero(double s, double dx) { return s == 0.0 ? dx * (4.0 * 2.0e-55) / 3.0 : s; }

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll 1
  for (int m = 32; m; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// sums over the block of N values each; `slot` alternates between calls
template <int N>
__device__ __forceinline__ void block_sums(AtparShared &sh, int &slot, double (&s)[N])
{
  for (int q = 0; q < N; q++) {
    s[q] = wave_sum(s[q]);
    if ((threadIdx.x & 63) == 0) sh.red[slot][threadIdx.x >> 6][q] = s[q];
  }
  __syncthreads();
  for (int q = 0; q < N; q++) {
    s[q] = 0.0;
#pragma unroll 1
    for (int w = 0; w < AT_NT / 64; w++) s[q] += sh.red[slot][w][q];
  }
  slot ^= 1;
}

// one block per (atom type, l): atpar.f:212-289 and, for l <= LOMAX with a
// local-orbital function, atpar.f:297-330.  The functions of l < NSLMAX are
// kept (fn, fnlo).
//
// Bound by the recurrences' chain (six dependent FP64 operations a mesh point,
// three or four functions an l) and by the fetch of code that runs once, far
// from any throughput: so the functions of an l run in lanes of one wave, side
// by side, their operands read from LDS ahead, while the other four
// waves form what the next 64 points need (one energy each, a point per lane:
// an exponential and four divisions a point) and write back the last 64; and
// the integrals are weighted sums in three loops.  One work-item per l did all
// of it in turn.  64 atom types, 781 points, 11 l: 3.75 ->
// 0.18 ms.
__global__ __launch_bounds__(AT_NT, 4) void k_atpar_l(AtparArgs g)
{
  __shared__ AtparShared sh;
  const int l = blockIdx.x, a = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool rel = g.rel != 0;
  const double c1 = 1.0, c2 = rel ? 1.0 / (137.0359895 * 137.0359895) : 1.0e-22;
  const double dele = 2.0e-3, delei = 0.25 / dele;
  const double cl = rel ? 2.0 * 137.0359895 : 1.0e10;
  const int jri = g.jrj[a];
  const double rnot = g.ro[a], dx = g.dh[a], z = g.zz[a];
  const double *v = g.vr + (size_t)a * g.jrid;
  const size_t ld = g.jrid;
  double *const work = g.work + (size_t)(a * g.nt + l) * AT_ROWS * ld, *const wt = work + 2 * AT_NE * ld;
  const double fl = (double)l;
  const bool lo = l <= g.lomax && g.loor[a * (g.lomax + 1) + l];
  const double elo = lo ? g.elo[a * (g.lomax + 1) + l] / 2.0 : 0.0;
  double ei = g.e[(size_t)a * g.lmaxd + l] / 2.0;
  int slot = 0;
  double *const A1 = l < g.nslmax ? g.fn + ((size_t)(a * g.nslmax + l) * 4) * ld : nullptr;
  double *const ALO = lo ? g.fnlo + ((size_t)(a * (g.lomax + 1) + l) * 2) * ld : nullptr;
  for (int pass = 0; pass < 2; pass++) {
    const int ne = lo ? AT_NE : AT_NE - 1;
    const int nch = (jri + AT_CH - 1) / AT_CH;
    // the chain's state, one energy per lane of wave 0
    double a0 = 0, b0 = 0, dg1 = 0, dg2 = 0, dg3 = 0, df1 = 0, df2 = 0, df3 = 0;
#pragma unroll 1
    for (int ch = -1; ch <= nch; ch++) {
      if (wave > 0) {
        const int en = wave - 1, k = (ch + 1) * AT_CH + lane, kp = (ch - 1) * AT_CH + lane;
        if (en < ne && k < jri) {
          const double eh = en == 0 ? ei - dele : en == 1 ? ei + dele : en == 2 ? ei : elo;
          outwin_coef(rel, v[k], rnot, dx, eh, fl, z, k, sh.c[(ch + 1) & 1][lane][en]);
        }
        if (en < ne && ch > 0 && kp < jri) {
          work[2 * en * ld + kp] = sh.f[(ch - 1) & 1][0][lane][en];
          work[(2 * en + 1) * ld + kp] = sh.f[(ch - 1) & 1][1][lane][en] * cl / 2.0;
          if (en == 0) wt[kp] = rint13_w(rnot, dx, jri, kp);
        }
      } else if (ch >= 0 && ch < nch && lane < ne) {
        const double h83 = 8.0 / 3.0, r1 = 1.0 / 9.0, r2 = -5.0 * r1, r3 = 19.0 * r1, x = -dx;
        const double(&c)[AT_CH + 2 * AT_PF][AT_NE][AT_NC] = sh.c[ch & 1];
        double(&f)[2][AT_CH][AT_NE] = sh.f[ch & 1];
        const int k1 = min(AT_CH, jri - ch * AT_CH);
        int k = 0;
        if (ch == 0) {
#pragma unroll 1
          for (; k < 3; k++) {
            a0 = c[k][lane][0];
            b0 = c[k][lane][1];
            dg1 = dg2; dg2 = dg3; dg3 = c[k][lane][2];
            df1 = df2; df2 = df3; df3 = c[k][lane][3];
            f[0][k][lane] = a0;
            f[1][k][lane] = b0;
          }
        }
        // AT_PF points a turn, their operands read a turn ahead (past the
        // piece's end from rows that hold nothing yet, and not used)
        double o[AT_PF][AT_NC], p[AT_PF][AT_NC];
        auto read = [&](double(&o)[AT_PF][AT_NC], int k) {
#pragma unroll
          for (int m = 0; m < AT_PF; m++)
#pragma unroll
            for (int q = 0; q < AT_NC; q++) o[m][q] = c[k + m][lane][q];
        };
        auto points = [&](const double(&o)[AT_PF][AT_NC]) {
#pragma unroll
          for (int m = 0; m < AT_PF; m++, k++) {
            if (k == k1) break;
            const double b11 = a0 * h83 + (r1 * dg1 + r2 * dg2) + r3 * dg3;
            const double b22 = b0 * h83 + (r1 * df1 + r2 * df2) + r3 * df3;
            const double u = o[m][2], y = o[m][3];
            a0 = b11 * (h83 - x) + b22 * u;
            b0 = b22 * (h83 + x) - b11 * y;
            a0 = fma(a0, o[m][0], a0 * o[m][1]);
            b0 = fma(b0, o[m][0], b0 * o[m][1]);
            dg1 = dg2; dg2 = dg3; dg3 = u * b0 - x * a0;
            df1 = df2; df2 = df3; df3 = x * b0 - y * a0;
            f[0][k][lane] = a0;
            f[1][k][lane] = b0;
          }
        };
        read(o, k);
#pragma unroll 1
        while (k < k1) {
          read(p, k + AT_PF);
          points(o);
          if (k == k1) break;
          read(o, k + AT_PF);
          points(p);
        }
        if (ch == nch - 1) {
          const double rj = rnot * exp(dx * (double)(jri - 1)), val = a0 / rj;
          sh.end[0][lane] = val;
          sh.end[1][lane] = (dg3 / (dx * rj) - val) / rj;
        }
      }
      __syncthreads();
    }
    // norms (atpar.f:222-262), a wave for each energy
    if (wave < ne) {
      const double *A = work + 2 * wave * ld, *B = A + ld;
      double s = 0.0;
#pragma unroll 4
      for (int k = lane; k < jri; k += 64) s += wt[k] * (c1 * A[k] * A[k] + c2 * B[k] * B[k]);
      s = wave_sum(s);
      if (lane == 0) sh.norm[wave] = 1.0 / sqrt(rint13_nonzero(s, dx));
    }
    __syncthreads();
    const double tr1 = sh.norm[0], tr2 = sh.norm[1], tr3 = sh.norm[2], trx = lo ? sh.norm[3] : 0.0;
    const double P = tr3 * sh.end[0][2], DP = tr3 * sh.end[1][2];
    // the normalised function and its energy derivative, made orthogonal to it
    double s1[1] = {0.0};
#pragma unroll 1
    for (int k = tid; k < jri; k += AT_NT) {
      const double A = tr3 * work[4 * ld + k], B = tr3 * work[5 * ld + k];
      const double AE = delei * (tr2 * work[2 * ld + k] - tr1 * work[k]);
      const double BE = delei * (tr2 * work[3 * ld + k] - tr1 * work[ld + k]);
      s1[0] += wt[k] * (c1 * A * AE + c2 * B * BE);
    }
    block_sums(sh, slot, s1);
    const double tr = -rint13_nonzero(s1[0], dx);
    const double PE = delei * (tr2 * sh.end[0][1] - tr1 * sh.end[0][0]) + tr * P;
    const double DPE = delei * (tr2 * sh.end[1][1] - tr1 * sh.end[1][0]) + tr * DP;
    // a function almost zero at the boundary: the energy is lowered by
    // 0.05 Ry and the l is done again, once (atpar.f:281-290)
    if (pass == 0 && fabs(P) < 1.0e-3) {
      ei = (g.e[(size_t)a * g.lmaxd + l] - 0.05) / 2.0;
      continue;
    }
    double s3[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
    for (int k = tid; k < jri; k += AT_NT) {
      const double A = tr3 * work[4 * ld + k], B = tr3 * work[5 * ld + k];
      const double AE = delei * (tr2 * work[2 * ld + k] - tr1 * work[k]) + tr * A;
      const double BE = delei * (tr2 * work[3 * ld + k] - tr1 * work[ld + k]) + tr * B;
      s3[0] += wt[k] * (c1 * AE * AE + c2 * BE * BE);
      if (A1) {
        A1[k] = A;
        A1[ld + k] = B;
        A1[2 * ld + k] = AE;
        A1[3 * ld + k] = BE;
      }
      if (lo) {
        const double AL = trx * work[6 * ld + k], BL = trx * work[7 * ld + k];
        ALO[k] = AL;
        ALO[ld + k] = BL;
        s3[1] += wt[k] * (c1 * A * AL + c2 * B * BL);
        s3[2] += wt[k] * (c1 * AE * AL + c2 * BE * BL);
      }
    }
    block_sums(sh, slot, s3);
    if (tid == 0) {
      double *o = g.out + (size_t)(a * g.nt + l) * 6;
      o[0] = P; o[1] = DP; o[2] = PE; o[3] = DPE; o[4] = rint13_nonzero(s3[0], dx); o[5] = 2.0 * ei;
      if (lo) {
        double *q = g.outlo + (size_t)(a * (g.lomax + 1) + l) * 4;
        q[0] = trx * sh.end[0][3];
        q[1] = trx * sh.end[1][3];
        q[2] = rint13_nonzero(s3[1], dx);
        q[3] = rint13_nonzero(s3[2], dx);
      }
    }
    break;
  }
}

// one wave per (atom type, l0, lm, lp) triple that the coupling list reads:
// VNS1..3 and, for l0 <= LOMAX, the local-orbital integrals (atpar.f:489-552),
// all of them in one pass over the mesh.  64 atom types, 781 points: 563 us
// with one work-item per triple -> 20 us.
struct VnsTriple {
  int a, l0, lm, lp;
};

__global__ __launch_bounds__(256) void k_atpar_vns(int ntrip, const VnsTriple *__restrict__ trip, AtparArgs g,
                                                   const double *__restrict__ vlm, int lmmxd, double *__restrict__ res)
{
  const int t = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64, lane = threadIdx.x & 63;
  if (t >= ntrip) return;
  const VnsTriple q = trip[t];
  const bool rel = g.rel != 0;
  const double c1 = 1.0, c2 = rel ? 1.0 / (137.0359895 * 137.0359895) : 1.0e-22;
  const int jri = g.jrj[q.a];
  const double dx = g.dh[q.a];
  const size_t ld = g.jrid;
  const double *wt = g.work + ((size_t)q.a * g.nt * AT_ROWS + 2 * AT_NE) * ld;  // l = 0's row
  const double *V = vlm + ((size_t)q.a * lmmxd + q.lm) * ld;
  const double *f0 = g.fn + ((size_t)(q.a * g.nslmax + q.l0) * 4) * ld;
  const double *fp = g.fn + ((size_t)(q.a * g.nslmax + q.lp) * 4) * ld;
  const bool lo0 = q.l0 <= g.lomax && g.loor[q.a * (g.lomax + 1) + q.l0];
  const bool lop = lo0 && q.lp <= g.lomax && g.loor[q.a * (g.lomax + 1) + q.lp];
  // without a local orbital the integrals that are not wanted read u instead
  const double *L0 = lo0 ? g.fnlo + ((size_t)(q.a * (g.lomax + 1) + q.l0) * 2) * ld : f0;
  const double *Lp = lop ? g.fnlo + ((size_t)(q.a * (g.lomax + 1) + q.lp) * 2) * ld : fp;
  // VNS1 = <u_l0 V u_lp>, VNS2 = <ue V ue>, VNS3 = <u_l0 V ue_lp>, and with the
  // local orbitals <lo V u>, <lo V ue>, <lo V lo>
  auto f = [&](int k, double(&y)[6]) {
    const double A = f0[k] * V[k], B = f0[ld + k] * V[k], AE = f0[2 * ld + k] * V[k], BE = f0[3 * ld + k] * V[k];
    const double Ap = fp[k], Bp = fp[ld + k], AEp = fp[2 * ld + k], BEp = fp[3 * ld + k];
    const double L = L0[k] * V[k], Lb = L0[ld + k] * V[k];
    y[0] = c1 * A * Ap + c2 * B * Bp;
    y[1] = c1 * AE * AEp + c2 * BE * BEp;
    y[2] = c1 * A * AEp + c2 * B * BEp;
    y[3] = c1 * L * Ap + c2 * Lb * Bp;
    y[4] = c1 * L * AEp + c2 * Lb * BEp;
    y[5] = c1 * L * Lp[k] + c2 * Lb * Lp[ld + k];
  };
  double z[6] = {};
  for (int k = lane; k < jri; k += 64) {
    double y[6];
    f(k, y);
    for (int m = 0; m < 6; m++) z[m] += wt[k] * y[m];
  }
  for (int m = 0; m < 6; m++) {
    const double s = rint13_nonzero(wave_sum(z[m]), dx);
    if (lane == 0) res[(size_t)t * 6 + m] = m < 3 || (m < 5 ? lo0 : lop) ? s : 0.0;
  }
}

// RINT13's weight of mesh point k (0-based): the integral is sum_k W_k f_k
// with W as RINT13 forms it (Simpson sums over alternate points, end
// corrections); the mesh points are multiplied out as in rint13.f
__device__ double rint13_weight(double rnot, double dx, int jri, int k)
{
  const double d = exp(dx);
  const int j0 = 3 - (jri % 2);  // first Z4 point (1-based)
  const int kk = k + 1;          // 1-based
  double w = 0.0;
  if (kk >= j0 && kk <= jri - 1) {
    double r = rnot * pow(d, (double)(j0 - 1));
    for (int j = j0; j < kk; j++) r = r * d;
    w = (((kk - j0) % 2 == 0) ? 4.0 : 2.0) * r * dx / 3.0;
  }
  if (kk == jri) {
    double r = rnot * pow(d, (double)(j0 - 1));
    for (int j = j0; j < jri; j++) r = r * d;
    w += r * dx / 3.0;
  }
  const int j1 = j0 - 1;
  const double r1 = rnot * pow(d, (double)(j0 - 1)) / d;
  if (kk == 1) w += rnot / 3.0 + (j1 > 1 ? 0.5 * dx * rnot : 0.0);
  if (kk == j1) w += dx * r1 / 3.0 + (j1 > 1 ? 0.5 * dx * r1 : 0.0);
  return w;
}

// dE/dV_LM(r_k) for every (atom type, lm, k): sum over the integrals of that
// (atom, lm) of dE/dVNS times the weight times the product of the two radial
// functions at r_k
struct VlmTerm {
  int a, lm, l0, lp, kind;  // kind 0..5: VNS1, VNS2, VNS3, VNS1LO, VNS2LO, VNS3LO
  double gv;                // dE/dVNS of that integral
};

__global__ void k_adjoint_vlm(int nterm, const VlmTerm *__restrict__ terms, const int *__restrict__ tstart, int ngroup,
                              AtparArgs g, double *__restrict__ gvlm, int lmmxd)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int grp = blockIdx.y;
  if (grp >= ngroup) return;
  const int t0 = tstart[grp], t1 = tstart[grp + 1];
  if (t0 >= t1) return;
  const int a = terms[t0].a, lm = terms[t0].lm;
  const int jri = g.jrj[a];
  if (k >= jri) return;
  const bool rel = g.rel != 0;
  const double c1 = 1.0, c2 = rel ? 1.0 / (137.0359895 * 137.0359895) : 1.0e-22;
  double acc = 0.0;
  for (int t = t0; t < t1; t++) {
    const VlmTerm q = terms[t];
    const double *f0 = g.fn + ((size_t)(a * g.nslmax + q.l0) * 4) * g.jrid;
    const double *fp = g.fn + ((size_t)(a * g.nslmax + q.lp) * 4) * g.jrid;
    double x0a, x0b, xpa, xpb;
    if (q.kind >= 3) {
      const double *L0 = g.fnlo + ((size_t)(a * (g.lomax + 1) + q.l0) * 2) * g.jrid;
      x0a = L0[k];
      x0b = L0[g.jrid + k];
    } else if (q.kind == 1) {
      x0a = f0[2 * (size_t)g.jrid + k];
      x0b = f0[3 * (size_t)g.jrid + k];
    } else {
      x0a = f0[k];
      x0b = f0[g.jrid + k];
    }
    if (q.kind == 0 || q.kind == 3) {
      xpa = fp[k];
      xpb = fp[g.jrid + k];
    } else if (q.kind == 5) {
      const double *Lp = g.fnlo + ((size_t)(a * (g.lomax + 1) + q.lp) * 2) * g.jrid;
      xpa = Lp[k];
      xpb = Lp[g.jrid + k];
    } else {
      xpa = fp[2 * (size_t)g.jrid + k];
      xpb = fp[3 * (size_t)g.jrid + k];
    }
    acc += q.gv * (c1 * x0a * xpa + c2 * x0b * xpb);
  }
  gvlm[((size_t)a * lmmxd + lm) * g.jrid + k] = acc * rint13_weight(g.ro[a], g.dh[a], jri, k);
}

// ------------------------------------------------------------------ host
template <class T>
static int put(DBuf<T> &b, const T *src, size_t count, hipStream_t s)
{
  int rc = b.alloc(count > 0 ? count : 1);
  if (rc) return rc;
  if (count) W2K_HIP(hipMemcpyAsync(b.p, src, sizeof(T) * count, hipMemcpyHostToDevice, s));
  return 0;
}

static AtparArgs atpar_args(RunDev &R)
{
  AtparArgs g;
  g.nat = R.nat;
  g.nt = R.at_nt;
  g.nslmax = W2K_NSLMAX;
  g.lomax = W2K_LOMAX;
  g.jrid = R.at_jrid;
  g.lmaxd = W2K_LMAX;
  g.rel = R.at_rel;
  g.jrj = R.d_at_jrj.p;
  g.ro = R.d_at_ro.p;
  g.dh = R.d_at_dh.p;
  g.zz = R.d_at_zz.p;
  g.vr = nullptr;
  g.e = g.elo = nullptr;
  g.loor = nullptr;
  g.fn = R.d_at_fn.p;
  g.fnlo = R.d_at_fnlo.p;
  g.work = g.out = g.outlo = nullptr;
  return g;
}

// the unique (atom, l0, lm, lp) triples of the run's HNS coupling terms
static std::vector<VnsTriple> vns_triples(const RunDev &R)
{
  std::vector<VnsTriple> t;
  for (const RunDev::HnsTerm &h : R.hns_terms) t.push_back({h.a, h.x, h.lmx, h.y});
  std::sort(t.begin(), t.end(), [](const VnsTriple &p, const VnsTriple &q) {
    return std::make_tuple(p.a, p.l0, p.lm, p.lp) < std::make_tuple(q.a, q.l0, q.lm, q.lp);
  });
  t.erase(std::unique(t.begin(), t.end(),
                      [](const VnsTriple &p, const VnsTriple &q) {
                        return p.a == q.a && p.l0 == q.l0 && p.lm == q.lm && p.lp == q.lp;
                      }),
          t.end());
  return t;
}

int atpar(Ctx &c, const w2k_radial_desc *rd, double *const out[16])
{
  RunDev &R = c.run();
  hipStream_t s = c.stream;
  const int nat = R.nat, nt = R.ltop;
  if (!rd || !rd->jrj || !rd->ro || !rd->dh || !rd->zz || !rd->vr || rd->jrid < 5) return W2K_EINVAL;
  for (int a = 0; a < nat; a++)
    if (rd->jrj[a] < 5 || rd->jrj[a] > rd->jrid || !(rd->dh[a] > 0.0) || !(rd->ro[a] > 0.0)) return W2K_EINVAL;
  if (rd->vlm) {
    for (const RunDev::HnsTerm &h : R.hns_terms)
      if (h.lmx < 0 || h.lmx >= rd->lmmxd) return W2K_EINVAL;
  }
  const int jrid = rd->jrid;
  int rc;
  R.at_ready = 0;
  R.at_rel = rd->rel ? 1 : 0;
  R.at_jrid = jrid;
  R.at_nt = nt;
  // LO energies ELO(l, ILO(l)) of the l that carry a local-orbital function
  std::vector<double> elo((size_t)nat * W2K_LOMAXP, 0.0);
  std::vector<int> loor((size_t)nat * W2K_LOMAXP, 0);
  for (int a = 0; a < nat; a++)
    for (int l = 0; l <= W2K_LOMAX; l++) {
      const int il = R.ilo[l + W2K_LOMAXP * a];
      loor[a * W2K_LOMAXP + l] = R.loor[l + W2K_LOMAXP * a] ? 1 : 0;
      if (il > 0) elo[a * W2K_LOMAXP + l] = R.elo[l + W2K_LOMAXP * ((il - 1) + W2K_NLOAT * (size_t)a)];
    }
  DBuf<double> &d_vr = c.at_d[0], &d_e = c.at_d[1], &d_elo = c.at_d[2], &d_work = c.at_d[3], &d_out = c.at_d[4];
  DBuf<double> &d_outlo = c.at_d[5];
  DBuf<int> &d_loor = c.at_i[0];
  if ((rc = put(R.d_at_jrj, rd->jrj, nat, s)) || (rc = put(R.d_at_ro, rd->ro, nat, s)) ||
      (rc = put(R.d_at_dh, rd->dh, nat, s)) || (rc = put(R.d_at_zz, rd->zz, nat, s)) ||
      (rc = put(d_vr, rd->vr, (size_t)jrid * nat, s)) || (rc = put(d_e, R.e.data(), R.e.size(), s)) ||
      (rc = put(d_elo, elo.data(), elo.size(), s)) || (rc = put(d_loor, loor.data(), loor.size(), s)))
    return rc;
  if ((rc = R.d_at_fn.alloc((size_t)nat * W2K_NSLMAX * 4 * jrid)) ||
      (rc = R.d_at_fnlo.alloc((size_t)nat * W2K_LOMAXP * 2 * jrid)) ||
      (rc = d_work.alloc((size_t)nat * nt * AT_ROWS * jrid)) ||
      (rc = d_out.alloc((size_t)nat * nt * 6)) || (rc = d_outlo.alloc((size_t)nat * W2K_LOMAXP * 4)))
    return rc;
  W2K_HIP(hipMemsetAsync(R.d_at_fnlo.p, 0, sizeof(double) * nat * W2K_LOMAXP * 2 * jrid, s));
  W2K_HIP(hipMemsetAsync(d_outlo.p, 0, sizeof(double) * nat * W2K_LOMAXP * 4, s));
  AtparArgs g = atpar_args(R);
  g.vr = d_vr.p;
  g.e = d_e.p;
  g.elo = d_elo.p;
  g.loor = d_loor.p;
  g.work = d_work.p;
  g.out = d_out.p;
  g.outlo = d_outlo.p;
  const int nth = nat * nt;
  hipLaunchKernelGGL(k_atpar_l, dim3(nt, nat), dim3(AT_NT), 0, s, g);
  W2K_STAGE(s, "k_atpar_l");
  std::vector<double> o((size_t)nth * 6), olo((size_t)nat * W2K_LOMAXP * 4);
  W2K_HIP(hipMemcpyAsync(o.data(), d_out.p, sizeof(double) * o.size(), hipMemcpyDeviceToHost, s));
  W2K_HIP(hipMemcpyAsync(olo.data(), d_outlo.p, sizeof(double) * olo.size(), hipMemcpyDeviceToHost, s));
  // non-spherical integrals of the coupling list
  std::vector<VnsTriple> trip;
  std::vector<double> vres;
  if (rd->vlm && !R.hns_terms.empty()) {
    trip = vns_triples(R);
    DBuf<int> &d_trip = c.at_i[1];
    DBuf<double> &d_vlm = c.at_d[6], &d_res = c.at_d[7];
    if ((rc = put(d_trip, reinterpret_cast<const int *>(trip.data()), trip.size() * 4, s)) ||
        (rc = put(d_vlm, rd->vlm, (size_t)jrid * rd->lmmxd * nat, s)) || (rc = d_res.alloc(trip.size() * 6)))
      return rc;
    const int ntr = (int)trip.size();
    hipLaunchKernelGGL(k_atpar_vns, dim3((ntr + 3) / 4), dim3(256), 0, s, ntr,
                       reinterpret_cast<const VnsTriple *>(d_trip.p), g, d_vlm.p, rd->lmmxd, d_res.p);
    W2K_STAGE(s, "k_atpar_vns");
    vres.resize(trip.size() * 6);
    W2K_HIP(hipMemcpyAsync(vres.data(), d_res.p, sizeof(double) * vres.size(), hipMemcpyDeviceToHost, s));
  }
  W2K_HIP(hipStreamSynchronize(s));
  for (int a = 0; a < nat; a++)
    for (int l = 0; l < nt; l++)
      for (int q = 0; q < 6; q++)
        if (out[q]) out[q][l + W2K_LMAX * (size_t)a] = o[((size_t)a * nt + l) * 6 + q];
  for (int a = 0; a < nat; a++)
    for (int l = 0; l <= W2K_LOMAX; l++)
      if (loor[a * W2K_LOMAXP + l])
        for (int q = 0; q < 4; q++)
          if (out[6 + q]) out[6 + q][l + W2K_LOMAXP * (size_t)a] = olo[((size_t)a * W2K_LOMAXP + l) * 4 + q];
  const size_t LOP2 = W2K_LOMAX + 2;
  for (size_t t = 0; t < trip.size(); t++) {
    const VnsTriple &q = trip[t];
    const double *v = &vres[t * 6];
    const size_t o3 = q.l0 + W2K_NSLMAX * (q.lm + (size_t)R.lmmxd * (q.lp + W2K_NSLMAX * (size_t)q.a));
    for (int k = 0; k < 3; k++)
      if (out[10 + k]) out[10 + k][o3] = v[k];
    if (q.l0 <= W2K_LOMAX) {
      const size_t ol = q.l0 + LOP2 * (q.lm + (size_t)R.lmmxd * (q.lp + W2K_NSLMAX * (size_t)q.a));
      // atpar.f:509-552: VNS1LO, VNS2LO zero unless LOOR(l0); VNS3LO only
      // written for LOOR(l0) and lp <= LOMAX (zero unless LOOR(lp) too)
      if (out[13]) out[13][ol] = v[3];
      if (out[14]) out[14][ol] = v[4];
      if (loor[q.a * W2K_LOMAXP + q.l0] && q.lp <= W2K_LOMAX && out[15]) out[15][ol] = v[5];
    }
  }
  R.at_ready = 1;
  return 0;
}

int adjoint_vlm(Ctx &c, const double *f_host, int lmmxd, double *g_vlm)
{
  RunDev &R = c.run();
  if (!R.at_ready) return W2K_ESTATE;
  hipStream_t s = c.stream;
  const int nat = R.nat;
  const size_t nlo3 = (size_t)(W2K_LOMAX + 2) * R.lmmxd * W2K_NSLMAX * nat;
  const size_t n3 = (size_t)W2K_NSLMAX * R.lmmxd * W2K_NSLMAX * nat;
  std::vector<double> gv[6];
  double *g6[6];
  for (int k = 0; k < 6; k++) {
    gv[k].assign(k < 3 ? n3 : nlo3, 0.0);
    g6[k] = gv[k].data();
  }
  int rc = adjoint_vns(c, f_host, g6);
  if (rc) return rc;
  // one term per distinct VNS entry the coupling list reads
  std::vector<VlmTerm> terms;
  for (const RunDev::HnsTerm &h : R.hns_terms) {
    const size_t ld = h.arr < 3 ? W2K_NSLMAX : W2K_LOMAX + 2;
    const size_t o = h.x + ld * (h.lmx + (size_t)R.lmmxd * (h.y + W2K_NSLMAX * (size_t)h.a));
    terms.push_back({h.a, h.lmx, h.x, h.y, h.arr, gv[h.arr][o]});
  }
  std::sort(terms.begin(), terms.end(), [](const VlmTerm &p, const VlmTerm &q) {
    return std::make_tuple(p.a, p.lm, p.kind, p.l0, p.lp) < std::make_tuple(q.a, q.lm, q.kind, q.l0, q.lp);
  });
  terms.erase(std::unique(terms.begin(), terms.end(),
                          [](const VlmTerm &p, const VlmTerm &q) {
                            return p.a == q.a && p.lm == q.lm && p.kind == q.kind && p.l0 == q.l0 && p.lp == q.lp;
                          }),
              terms.end());
  for (const VlmTerm &t : terms)
    if (t.lm >= lmmxd) return W2K_EINVAL;
  std::vector<int> start;
  for (size_t t = 0; t < terms.size(); t++)
    if (t == 0 || terms[t].a != terms[t - 1].a || terms[t].lm != terms[t - 1].lm) start.push_back((int)t);
  const int ngroup = (int)start.size();
  start.push_back((int)terms.size());
  const size_t ng = (size_t)R.at_jrid * lmmxd * nat;
  std::fill(g_vlm, g_vlm + ng, 0.0);
  if (ngroup == 0) return 0;
  DBuf<int> d_terms, d_start;
  DBuf<double> d_g;
  static_assert(sizeof(VlmTerm) % sizeof(int) == 0, "VlmTerm as ints");
  if ((rc = put(d_terms, reinterpret_cast<const int *>(terms.data()), terms.size() * sizeof(VlmTerm) / sizeof(int), s)) ||
      (rc = put(d_start, start.data(), start.size(), s)) || (rc = d_g.alloc(ng)))
    return rc;
  W2K_HIP(hipMemsetAsync(d_g.p, 0, sizeof(double) * ng, s));
  AtparArgs g = atpar_args(R);
  hipLaunchKernelGGL(k_adjoint_vlm, dim3((R.at_jrid + 255) / 256, ngroup), dim3(256), 0, s, (int)terms.size(),
                     reinterpret_cast<const VlmTerm *>(d_terms.p), d_start.p, ngroup, g, d_g.p, lmmxd);
  W2K_STAGE(s, "k_adjoint_vlm");
  W2K_HIP(hipMemcpyAsync(g_vlm, d_g.p, sizeof(double) * ng, hipMemcpyDeviceToHost, s));
  W2K_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // namespace w2k
