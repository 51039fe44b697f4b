// SECLR4 of the complex build (lapw1c) on the GPU: seclr4.F:155-358 with the
// Z-routines ZPOTRF, ZHCGST (zhcgst.f:116-163), ZHETRD2/ZHEEVX2
// (zheevx2.f:305-367), DSTEBZ2 and the back-transforms.
//
// Conventions of the reference kept exactly (and restated by the oracle):
//   - HS is conjugated on entry (seclr4.F:159-166): the lower triangle then
//     holds H, the strict upper triangle conj(S) and HSDIAG diag(S);
//   - S = U^H U (ZPOTRF 'U') on that upper triangle;
//   - ZHCGST reduces with V = conj(U): C = V^-H H V^-1;
//   - the Hermitian tridiagonalisation uses ZLARFG reflectors (beta real,
//     tau complex), so the tridiagonal matrix is real and the bisection and
//     inverse iteration are those of the real build;
//   - Z = V^-1 Q Zt.
// Complex matrices are planar on the device (real parts, then imaginary parts
// one matrix further), and every complex product is four real MFMA GEMMs.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <functional>
#include <vector>

#include "chol_leaf.h"
#include "seclr4_shared.h"
#include "twostage.h"

namespace w2k {

// C = alpha op(A) op(B) + beta C, planar complex; op: 'N', 'T' (transpose),
// 'C' (conjugate transpose), 'R' (conjugate, not transposed); alpha, beta real
static int zgemm(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha, const double *Ar,
                 const double *Ai, int lda, const double *Br, const double *Bi, int ldb, double beta, double *Cr,
                 double *Ci, int ldc, int tri = 0, int atri = 0, int btri = 0, double *ws = nullptr, size_t wsn = 0)
{
  // products with dense operands and no split K: one fused complex kernel
  // (C read and written once); short K (rank updates) is where it pays
  if (atri == 0 && btri == 0 && ws == nullptr && k <= 256)
    return zgemm_fused(s, ta, tb, m, n, k, alpha, Ar, Ai, lda, Br, Bi, ldb, beta, Cr, Ci, ldc, tri);
  // dense products with a long K onto few output tiles (the back-transform's
  // V^H Z and Gram matrices): the fused kernel with split K reads each
  // operand plane once and feeds 16 MFMAs from 8 LDS reads per step, against
  // 4 from 4 in the real 64 x 64 kernel
  const long ztiles = (long)((m + 63) / 64) * ((n + 63) / 64);
  if (atri == 0 && btri == 0 && tri == 0 && ws != nullptr && ztiles < 256 && k >= W2K_ZSPLIT_KMIN &&
      wsn >= (size_t)4 * m * n)
    return zgemm_fused(s, ta, tb, m, n, k, alpha, Ar, Ai, lda, Br, Bi, ldb, beta, Cr, Ci, ldc, tri, ws, wsn);
  const double sa = (ta == 'C' || ta == 'R') ? -1.0 : 1.0, sb = (tb == 'C' || tb == 'R') ? -1.0 : 1.0;
  const char ra = (ta == 'T' || ta == 'C') ? 'T' : 'N', rb = (tb == 'T' || tb == 'C') ? 'T' : 'N';
  int rc;
  // Cr = alpha (Ar Br - sa sb Ai Bi) + beta Cr ; Ci = alpha (sb Ar Bi + sa Ai Br) + beta Ci
  if ((rc = dgemm(s, ra, rb, m, n, k, alpha, Ar, lda, Br, ldb, beta, Cr, ldc, tri, atri, btri, ws, wsn))) return rc;
  if ((rc = dgemm(s, ra, rb, m, n, k, -alpha * sa * sb, Ai, lda, Bi, ldb, 1.0, Cr, ldc, tri, atri, btri, ws, wsn)))
    return rc;
  if ((rc = dgemm(s, ra, rb, m, n, k, alpha * sb, Ar, lda, Bi, ldb, beta, Ci, ldc, tri, atri, btri, ws, wsn)))
    return rc;
  if ((rc = dgemm(s, ra, rb, m, n, k, alpha * sa, Ai, lda, Br, ldb, 1.0, Ci, ldc, tri, atri, btri, ws, wsn)))
    return rc;
  return 0;
}

// D (rows x cols, ld rows) = X + s Y (ld ldx)
__global__ void k_zsum(int rows, int cols, const double *__restrict__ X, const double *__restrict__ Y, int ldx,
                       double s, double *__restrict__ D)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= rows || j >= cols) return;
  const size_t o = (size_t)i + (size_t)ldx * j;
  D[(size_t)i + (size_t)rows * j] = X[o] + s * Y[o];
}

// three-product combination on the output (triangle tri): mode 0 after T =
// A_r B_r: Cr = a T + b Cr, Ci -= a T; mode 1 after T = Im(op A) Im(op B):
// Cr -= a T, Ci -= a T
__global__ void k_z3m_comb(int m, int n, const double *__restrict__ T, double a, double b, double *__restrict__ Cr,
                           double *__restrict__ Ci, int ldc, int tri, int mode)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= m || j >= n) return;
  if ((tri == 1 && i < j) || (tri == 2 && i > j)) return;
  const double t = a * T[(size_t)i + (size_t)m * j];
  const size_t o = (size_t)i + (size_t)ldc * j;
  if (mode == 0) {
    Cr[o] = (b != 0.0 ? b * Cr[o] : 0.0) + t;
    Ci[o] -= t;
  } else {
    Cr[o] -= t;
    Ci[o] -= t;
  }
}

// K up to which a complex product below the three-product size runs on the
// fused kernel (triangular operands read as dense): 1024 measured 2 ms
// faster than 512 on the 100-atom Cholesky, 4096 no faster than 1024
constexpr int ZFUSED_KMAX = 1024;

// zgemm for the large products: three real products instead of four
// (Ci = (Ar + Im op A)(Br + Im op B) - Ar Br - Im op A Im op B), which takes a
// quarter of the arithmetic off at the cost of three elementwise passes and
// an error of the imaginary part bounded by |A| |B| rather than by the
// products of the parts.  Smaller products, and calls inside the
// allocation-free entry point, go to the fused kernel (K <= ZFUSED_KMAX) or zgemm.
static int zgemm3(Ctx &c, hipStream_t s, char ta, char tb, int m, int n, int k, double alpha, const double *Ar,
                  const double *Ai, int lda, const double *Br, const double *Bi, int ldb, double beta, double *Cr,
                  double *Ci, int ldc, int tri = 0, int atri = 0, int btri = 0, double *ws = nullptr, size_t wsn = 0)
{
  const bool big = (double)m * n * k >= 1073741824.0 && k > 256;
  if (!big || g_arena || m <= 0 || n <= 0 || k <= 0) {
    // the triangular operands of these products (U, U^-1, V^-1) hold zeros in
    // their other triangle, so the fused kernel may read them as dense: one
    // launch instead of four for the many small products of the recursions
    if (k <= ZFUSED_KMAX)
      return zgemm_fused(s, ta, tb, m, n, k, alpha, Ar, Ai, lda, Br, Bi, ldb, beta, Cr, Ci, ldc, tri);
    return zgemm(s, ta, tb, m, n, k, alpha, Ar, Ai, lda, Br, Bi, ldb, beta, Cr, Ci, ldc, tri, atri, btri, ws, wsn);
  }
  const double sa = (ta == 'C' || ta == 'R') ? -1.0 : 1.0, sb = (tb == 'C' || tb == 'R') ? -1.0 : 1.0;
  const char ra = (ta == 'T' || ta == 'C') ? 'T' : 'N', rb = (tb == 'T' || tb == 'C') ? 'T' : 'N';
  // stored extents of A and B
  const int arows = ra == 'T' ? k : m, acols = ra == 'T' ? m : k;
  const int brows = rb == 'T' ? n : k, bcols = rb == 'T' ? k : n;
  const size_t na = (size_t)arows * acols, nbb = (size_t)brows * bcols, nt = (size_t)m * n;
  int rc;
  if ((rc = c.w_3m.alloc(na + nbb + nt))) return rc;
  double *SA = c.w_3m.p, *SB = SA + na, *T = SB + nbb;
  hipLaunchKernelGGL(k_zsum, dim3((arows + 255) / 256, acols), dim3(256), 0, s, arows, acols, Ar, Ai, lda, sa, SA);
  W2K_STAGE(s, "k_zsum");
  hipLaunchKernelGGL(k_zsum, dim3((brows + 255) / 256, bcols), dim3(256), 0, s, brows, bcols, Br, Bi, ldb, sb, SB);
  W2K_STAGE(s, "k_zsum");
  const dim3 gc((m + 255) / 256, n);
  if ((rc = dgemm(s, ra, rb, m, n, k, alpha, SA, arows, SB, brows, beta, Ci, ldc, tri, atri, btri, ws, wsn))) return rc;
  if ((rc = dgemm(s, ra, rb, m, n, k, 1.0, Ar, lda, Br, ldb, 0.0, T, m, tri, atri, btri, ws, wsn))) return rc;
  hipLaunchKernelGGL(k_z3m_comb, gc, dim3(256), 0, s, m, n, T, alpha, beta, Cr, Ci, ldc, tri, 0);
  W2K_STAGE(s, "k_z3m_comb");
  if ((rc = dgemm(s, ra, rb, m, n, k, sa * sb, Ai, lda, Bi, ldb, 0.0, T, m, tri, atri, btri, ws, wsn))) return rc;
  hipLaunchKernelGGL(k_z3m_comb, gc, dim3(256), 0, s, m, n, T, alpha, beta, Cr, Ci, ldc, tri, 1);
  W2K_STAGE(s, "k_z3m_comb");
  return 0;
}

// ------------------------------------------------------------------ set-up
// U (upper, diagonal from HSDIAG) = conj of the stored upper triangle;
// H full Hermitian from the stored lower triangle (conjugated back)
__global__ void k_zprep(int n, const double *__restrict__ hs, const double *__restrict__ hsdiag, double *Ur, double *Ui,
                        double *Hr, double *Hi)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= n) return;
  const size_t o = (size_t)i + (size_t)n * j;
  if (i < j) {
    Ur[o] = hs[2 * o];
    Ui[o] = -hs[2 * o + 1];
    const size_t t = (size_t)j + (size_t)n * i;
    Hr[o] = hs[2 * t];
    Hi[o] = hs[2 * t + 1];
  } else if (i == j) {
    Ur[o] = hsdiag[2 * i];
    Ui[o] = -hsdiag[2 * i + 1];
    Hr[o] = hs[2 * o];
    Hi[o] = 0.0;
  } else {
    Ur[o] = 0.0;
    Ui[o] = 0.0;
    Hr[o] = hs[2 * o];
    Hi[o] = -hs[2 * o + 1];
  }
}

// Cholesky S = U^H U of the kb x kb diagonal block at k0 (over S) and U^-1 into
// the same block of W (zero below the diagonal); INFO as k_chol_diag.  91 + 32
// us as two kernels -> 37 us.
__global__ __launch_bounds__(256) void k_zchol_diag(int n, int k0, int kb, double *__restrict__ Ur,
                                                    double *__restrict__ Ui, double *__restrict__ Wr,
                                                    double *__restrict__ Wi, int *__restrict__ info)
{
  __shared__ Leaf<true> s;
  const int r = threadIdx.x & 63, g = threadIdx.x >> 6;
  {
    double lr[16], li[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const size_t o = (size_t)(k0 + min(r, kb - 1)) + (size_t)n * (k0 + min(g + 4 * q, kb - 1));
      lr[q] = Ur[o];
      li[q] = Ui[o];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int c = g + 4 * q;
      s.m[0][r][c] = r <= c && c < kb ? lr[q] : (r == c ? 1.0 : 0.0);
      s.m[1][r][c] = r <= c && c < kb ? li[q] : 0.0;
    }
  }
  __syncthreads();
  const int first = chol_leaf<true>(s, [](double p) { return p > 0.0; });
  if (r < kb)
    for (int c = g; c < kb; c += 4) {
      const size_t o = (size_t)(k0 + r) + (size_t)n * (k0 + c);
      if (r <= c) {
        Ur[o] = s.m[0][r][c];
        Ui[o] = s.m[1][r][c];
      }
      Wr[o] = s.x[0][r][c];
      Wi[o] = s.x[1][r][c];
    }
  if (threadIdx.x == 0 && first != 0 && *info == 0) *info = k0 + first;
}

// R = S^-1 for a 64 x 64 upper triangular complex S in LDS (zero below the
// diagonal; R zero on entry), by all 256 threads of the block: the 16 x 16
// diagonal blocks by column back-substitution (threads 0..63, at most 16
// steps each), then two doubling steps X12 = -X11 (S12 X22) over the block's
// threads, through the product buffer P.  The longest dependent chain is
// about 140 complex multiply-adds instead of 2080 for back-substitution
// over all 64 rows.
__device__ void ztri_inv64(double (*sr)[NB + 1], double (*si)[NB + 1], double (*rr)[NB + 1], double (*ri)[NB + 1],
                           double (*pr)[NB / 2 + 1], double (*pi)[NB / 2 + 1], int t)
{
  static_assert(NB == 64, "64 x 64 blocks");
  if (t < NB) {
    const int b0 = (t / 16) * 16, c = t;
    for (int r = c; r >= b0; r--) {
      double xr = (r == c) ? 1.0 : 0.0, xi = 0.0;
      for (int q = r + 1; q <= c; q++) {
        xr -= sr[r][q] * rr[q][c] - si[r][q] * ri[q][c];
        xi -= sr[r][q] * ri[q][c] + si[r][q] * rr[q][c];
      }
      const double dr = sr[r][r], di = si[r][r], den = dr * dr + di * di;
      rr[r][c] = (xr * dr + xi * di) / den;
      ri[r][c] = (xi * dr - xr * di) / den;
    }
  }
  __syncthreads();
  for (int h = 16; h < NB; h *= 2) {
    const int nout = (NB / (2 * h)) * h * h;  // outputs of all pairs of this step
    for (int o = t; o < nout; o += blockDim.x) {
      const int pp = o / (h * h), rc = o % (h * h), r = rc % h, c = rc / h, b = 2 * h * pp;
      double ar = 0.0, ai = 0.0;  // P(r, c) = sum_{q <= c} S(b + r, b + h + q) X22(q, c)
      for (int q = 0; q <= c; q++) {
        const double s_r = sr[b + r][b + h + q], s_i = si[b + r][b + h + q];
        const double x_r = rr[b + h + q][b + h + c], x_i = ri[b + h + q][b + h + c];
        ar += s_r * x_r - s_i * x_i;
        ai += s_r * x_i + s_i * x_r;
      }
      pr[h * pp + r][c] = ar;
      pi[h * pp + r][c] = ai;
    }
    __syncthreads();
    for (int o = t; o < nout; o += blockDim.x) {
      const int pp = o / (h * h), rc = o % (h * h), r = rc % h, c = rc / h, b = 2 * h * pp;
      double ar = 0.0, ai = 0.0;  // X12(r, c) = -sum_{q >= r} X11(r, q) P(q, c)
      for (int q = r; q < h; q++) {
        const double x_r = rr[b + r][b + q], x_i = ri[b + r][b + q];
        const double p_r = pr[h * pp + q][c], p_i = pi[h * pp + q][c];
        ar += x_r * p_r - x_i * p_i;
        ai += x_r * p_i + x_i * p_r;
      }
      rr[b + r][b + h + c] = -ar;
      ri[b + r][b + h + c] = -ai;
    }
    __syncthreads();
  }
}

__global__ void k_zfill(size_t cnt, double *p, double v)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cnt) p[i] = v;
}

__global__ void k_negate(size_t cnt, double *p)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cnt) p[i] = -p[i];
}

// Hermitian completion: C(j,i) = conj C(i,j) for i > j, real diagonal
__global__ void k_zmirror_lower(int n, double *Cr, double *Ci)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= n || i < j) return;
  if (i == j) {
    Ci[(size_t)i + (size_t)n * i] = 0.0;
    return;
  }
  const size_t lo = (size_t)i + (size_t)n * j, up = (size_t)j + (size_t)n * i;
  Cr[up] = Cr[lo];
  Ci[up] = -Ci[lo];
}

// ------------------------------------------------------------------ back-transforms
__global__ void k_zvpanel(int n, int p0, int nb, const double *__restrict__ ar, const double *__restrict__ ai,
                          double *__restrict__ vr, double *__restrict__ vi)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  if (r >= n || k >= nb) return;
  const int i = p0 + k;
  double xr = 0.0, xi = 0.0;
  if (r == i + BND) xr = 1.0;
  else if (r > i + BND) { xr = ar[(size_t)r + (size_t)n * i]; xi = ai[(size_t)r + (size_t)n * i]; }
  vr[(size_t)r + (size_t)n * k] = xr;
  vi[(size_t)r + (size_t)n * k] = xi;
}

// T of I - V T V^H from G = V^H V (ZLARFT 'F','C'), whose recurrence
// T(0:i,i) = -tau_i T(0:i,0:i) G(0:i,i) says T = M^-1 with M upper
// triangular, M(i,i) = 1/tau_i and M(q,i) = G(q,i) above the diagonal.  A
// reflector with tau_i = 0 is the identity: its row and column of M are
// cleared (M(i,i) = 1) and T(i,i) is set to 0 afterwards.  nb <= 64.
__global__ __launch_bounds__(256) void k_zlarft(int nb, const double *__restrict__ gr, const double *__restrict__ gi,
                                                const double *__restrict__ taur, const double *__restrict__ taui,
                                                double *__restrict__ tmr, double *__restrict__ tmi)
{
  __shared__ double sr[NB][NB + 1], si[NB][NB + 1], rr[NB][NB + 1], ri[NB][NB + 1];
  __shared__ double pr[NB / 2][NB / 2 + 1], pi[NB / 2][NB / 2 + 1];
  __shared__ int zero[NB];
  const int t = threadIdx.x;
  if (t < NB) zero[t] = !(t < nb && (taur[t] != 0.0 || taui[t] != 0.0));
  __syncthreads();
  for (int idx = t; idx < NB * NB; idx += blockDim.x) {
    const int r = idx % NB, c = idx / NB;
    double vr = 0.0, vi = 0.0;
    if (r == c) {
      if (zero[r]) {
        vr = 1.0;
      } else {
        const double a = taur[r], b = taui[r], den = a * a + b * b;
        vr = a / den;
        vi = -b / den;
      }
    } else if (r < c && !zero[r] && !zero[c]) {
      vr = gr[r + nb * c];
      vi = gi[r + nb * c];
    }
    sr[r][c] = vr;
    si[r][c] = vi;
    rr[r][c] = 0.0;
    ri[r][c] = 0.0;
  }
  __syncthreads();
  ztri_inv64(sr, si, rr, ri, pr, pi, t);
  for (int idx = t; idx < nb * nb; idx += blockDim.x) {
    const int r = idx % nb, c = idx / nb;
    const bool keep = r <= c && !(r == c && zero[r]);
    tmr[r + nb * c] = keep ? rr[r][c] : 0.0;
    tmi[r + nb * c] = keep ? ri[r][c] : 0.0;
  }
}

__global__ void k_zgather_cols(int n, int m, const int *__restrict__ perm, const double *__restrict__ sr,
                               const double *__restrict__ si, double *__restrict__ dr, double *__restrict__ di)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (r >= n || c >= m) return;
  dr[(size_t)r + (size_t)n * c] = sr[(size_t)r + (size_t)n * perm[c]];
  di[(size_t)r + (size_t)n * c] = si[(size_t)r + (size_t)n * perm[c]];
}

__global__ void k_interleave(size_t cnt, const double *__restrict__ re, const double *__restrict__ im,
                             double *__restrict__ out)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  out[2 * i] = re[i];
  out[2 * i + 1] = im[i];
}

// ------------------------------------------------------------------ driver
int seclr4_complex(Ctx &c, double el, double eu, int nume, int *ne_out, int *nbelw_out)
{
  const int n = c.n;
  hipStream_t s = c.stream;
  int rc;
  const size_t nn = (size_t)n * n;
  // planar complex workspaces: U, H then C (then reflectors), W = V^-1, X
  if ((rc = c.w_a.alloc(2 * nn)) || (rc = c.w_b.alloc(2 * nn)) || (rc = c.w_c.alloc(2 * nn))) return rc;
  if ((rc = c.w_x.alloc(2 * nn))) return rc;
  if ((rc = c.w_gk.alloc((size_t)1 << 22))) return rc;
  double *Ur = c.w_a.p, *Ui = Ur + nn, *Hr = c.w_b.p, *Hi = Hr + nn, *Wr = c.w_c.p, *Wi = Wr + nn;
  double *Xr = c.w_x.p, *Xi = Xr + nn;
  double *ws = c.w_gk.p;
  const size_t wsn = c.w_gk.n;
  Seclr4Bufs B;
  if ((rc = seclr4_buffers(c, n, 1, B))) return rc;

  W2K_HIP(hipEventRecord(c.ev[6], s));
  // ---- 1. Cholesky S = U^H U
  {
    dim3 g2((n + 255) / 256, n);
    hipLaunchKernelGGL(k_zprep, g2, dim3(256), 0, s, n, c.d_hs.p, c.d_hsdiag.p, Ur, Ui, Hr, Hi);
    W2K_STAGE(s, "k_zprep");
    // W: U^-1 (zero below the diagonal), formed with U and conjugated by the
    // reduction
    hipLaunchKernelGGL(k_zfill, dim3((unsigned)((2 * nn + 255) / 256)), dim3(256), 0, s, 2 * nn, Wr, 0.0);
    W2K_STAGE(s, "k_zfill");
    // S = U^H U and W = U^-1 together, by recursive halving over the
    // NB-blocks: with S = [S11 S12; . S22], U11 and W11 from the first half,
    // U12 = W11^H S12, S22 -= U12^H U12, U22 and W22 from the second half and
    // W12 = -W11 U12 W22.  The block kernels factor and invert one NB-block;
    // the rest is a few large products instead of one thin product per
    // block row.
    std::function<int(int, int)> chol = [&](int lo, int hi) -> int {
      const int nblk = (hi - lo + NB - 1) / NB;
      if (nblk <= 1) {
        const int kb = hi - lo;
        hipLaunchKernelGGL(k_zchol_diag, dim3(1), dim3(256), 0, s, n, lo, kb, Ur, Ui, Wr, Wi, B.info);
        W2K_STAGE(s, "k_zchol_diag");
        return 0;
      }
      const int mid = lo + (nblk / 2) * NB;
      const int s1 = mid - lo, s2 = hi - mid;
      const size_t o11 = (size_t)lo + (size_t)n * lo, o12 = (size_t)lo + (size_t)n * mid;
      const size_t o22 = (size_t)mid + (size_t)n * mid;
      int r;
      if ((r = chol(lo, mid))) return r;
      // U12 = W11^H S12 (W11^H lower triangular), through X
      if ((r = zgemm3(c, s, 'C', 'N', s1, s2, s1, 1.0, Wr + o11, Wi + o11, n, Ur + o12, Ui + o12, n, 0.0, Xr, Xi, n, 0,
                      2, 0, ws, wsn)))
        return r;
      W2K_HIP(hipMemcpy2DAsync(Ur + o12, sizeof(double) * n, Xr, sizeof(double) * n, sizeof(double) * s1, s2,
                               hipMemcpyDeviceToDevice, s));
      W2K_HIP(hipMemcpy2DAsync(Ui + o12, sizeof(double) * n, Xi, sizeof(double) * n, sizeof(double) * s1, s2,
                               hipMemcpyDeviceToDevice, s));
      // S22 -= U12^H U12 (upper triangle)
      if ((r = zgemm3(c, s, 'C', 'N', s2, s2, s1, -1.0, Ur + o12, Ui + o12, n, Ur + o12, Ui + o12, n, 1.0, Ur + o22,
                      Ui + o22, n, 2)))
        return r;
      if ((r = chol(mid, hi))) return r;
      // W12 = -(W11 U12) W22 (W11, W22 upper triangular)
      if ((r = zgemm3(c, s, 'N', 'N', s1, s2, s1, 1.0, Wr + o11, Wi + o11, n, Ur + o12, Ui + o12, n, 0.0, Xr, Xi, n, 0,
                      1, 0, ws, wsn)))
        return r;
      return zgemm3(c, s, 'N', 'N', s1, s2, s2, -1.0, Xr, Xi, n, Wr + o22, Wi + o22, n, 0.0, Wr + o12, Wi + o12, n, 0,
                    0, 1, ws, wsn);
    };
    if ((rc = chol(0, n))) return rc;
  }
  W2K_HIP(hipEventRecord(c.ev[7], s));
  int hinfo[4];
  W2K_HIP(hipMemcpyAsync(hinfo, B.info, sizeof(int) * 4, hipMemcpyDeviceToHost, s));
  W2K_HIP(hipStreamSynchronize(s));
  if (hinfo[0] != 0) return hinfo[0];  // ZPOTRF INFO, seclr4.F:200-205
  // ---- 2. reduction with V = conj(U): W = V^-1, X = H W, C = W^H X
  {
    // V^-1 = conj(U^-1), the Cholesky's W conjugated
    hipLaunchKernelGGL(k_negate, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, s, nn, Wi);
    W2K_STAGE(s, "k_negate");
    if ((rc = zgemm3(c, s, 'N', 'N', n, n, n, 1.0, Hr, Hi, n, Wr, Wi, n, 0.0, Xr, Xi, n, 0, 0, 1))) return rc;
    if ((rc = zgemm3(c, s, 'C', 'N', n, n, n, 1.0, Wr, Wi, n, Xr, Xi, n, 0.0, Hr, Hi, n, 1, 2, 0))) return rc;
    dim3 g2((n + 255) / 256, n);
    hipLaunchKernelGGL(k_zmirror_lower, g2, dim3(256), 0, s, n, Hr, Hi);
    W2K_STAGE(s, "k_zmirror_lower");
  }
  W2K_HIP(hipEventRecord(c.ev[8], s));
  // ---- 3. Hermitian tridiagonalisation of C (in H): band, then bulge chasing
  SbArgs g;
  if ((rc = sb_buffers(c, g, n, 1))) return rc;
  g.lda = n; g.ar = Hr; g.ai = Hi;
  g.Pr = B.P; g.Pi = B.P + (size_t)3 * n * BND;
  g.d = B.d; g.e = B.e;
  g.taur = B.tau; g.taui = B.tau + n;
  g.V2r = Ur; g.V2i = Ui;  // U is not needed after the inversion
  if ((rc = sb_reduce(c, s, g, 1))) return rc;
  W2K_HIP(hipEventRecord(c.ev[9], s));
  if ((rc = sb_take_times(c, s, n))) return rc;
  // ---- 4./5. real tridiagonal eigenpairs (shared with the real build)
  double *Zt = Xr;  // n x m real, then the real part of Q Zt
  double *Zi = Xi;  // imaginary part of Q Zt
  int m = 0, nbelw = 0;
  if ((rc = tridiag_eigen(c, B, el, eu, nume, Zt, &m, &nbelw))) return rc;
  *nbelw_out = nbelw;
  c.nbelw = nbelw;
  if ((rc = c.d_z.alloc((size_t)2 * n * (m > 0 ? m : 1)))) return rc;
  W2K_HIP(hipEventRecord(c.ev[10], s));
  if (m > 0) {
    // ---- 6. Z = Q Zt with complex reflectors, sort, Z = V^-1 Z
    const size_t zc = (size_t)n * m;
    hipLaunchKernelGGL(k_zfill, dim3((unsigned)((zc + 255) / 256)), dim3(256), 0, s, zc, Zi, 0.0);
    W2K_STAGE(s, "k_zfill");
    if ((rc = sb_apply_q2(c, s, g, 1, m, Zt, Zi, n))) return rc;
    // blocks of ZBT reflectors (the launches of a block, not its arithmetic,
    // set the pace at these orders: 64-reflector blocks halve them)
    constexpr int ZBT = 64;
    // The reflector panel V, its Gram matrix and T depend on the reflectors
    // only: they are formed on the second stream up to two blocks ahead, in
    // two buffers, while this stream applies the blocks to Z (Y1 = V^H Z,
    // Y2 = T Y1, Z -= V Y2).  bt_ready[u]: block in buffer u formed;
    // bt_used[u]: its products with Z done.
    // w_bt: V (re, im: n x ZBT each) x 2, T (re, im) x 2, the Gram matrix,
    // Y1 and Y2 (re, im: ZBT x m each), the Gram products' split-K workspace
    constexpr size_t GWS = (size_t)64 * ZBT * ZBT;
    if ((rc = c.w_bt.alloc((size_t)2 * (2 * n + 3 * ZBT + 2 * m) * ZBT + GWS))) return rc;
    double *vr[2], *vi[2], *tr[2], *ti[2];
    double *q = c.w_bt.p;
    for (int u = 0; u < 2; u++) {
      vr[u] = q; vi[u] = q + (size_t)n * ZBT; q += (size_t)2 * n * ZBT;
    }
    for (int u = 0; u < 2; u++) {
      tr[u] = q; ti[u] = q + ZBT * ZBT; q += 2 * ZBT * ZBT;
    }
    double *gmr = q, *gmi = q + ZBT * ZBT;
    q += 2 * ZBT * ZBT;
    double *y1r = q, *y1i = y1r + (size_t)ZBT * m, *y2r = y1i + (size_t)ZBT * m, *y2i = y2r + (size_t)ZBT * m;
    double *gws = y2i + (size_t)ZBT * m;
    const int nref = std::max(0, n - BND - 1);  // reflectors of Q1; v_i starts at row i + BND
    const int nblk = nref > 0 ? (nref + ZBT - 1) / ZBT : 0;
    hipStream_t sa = c.aux;
    auto p0_of = [&](int k) { return (nblk - 1 - k) * ZBT; };
    auto prep = [&](int k) -> int {
      const int u = k & 1, p0 = p0_of(k), nb = std::min(ZBT, nref - p0);
      if (k >= 2) W2K_HIP(hipStreamWaitEvent(sa, c.bt_used[u], 0));
      hipLaunchKernelGGL(k_zvpanel, dim3((n + 255) / 256, nb), dim3(256), 0, sa, n, p0, nb, Hr, Hi, vr[u], vi[u]);
      W2K_STAGE(sa, "k_zvpanel");
      // the block's reflectors are zero above row p0+BND: the products start at
      // that row rounded down to 16 rows, which keeps the operands' 128-byte alignment
      const int o = (p0 + BND) & ~15, nr = n - o;
      int r2;
      if ((r2 = zgemm(sa, 'C', 'N', nb, nb, nr, 1.0, vr[u] + o, vi[u] + o, n, vr[u] + o, vi[u] + o, n, 0.0, gmr, gmi,
                      nb, 0, 0, 0, gws, GWS)))
        return r2;
      hipLaunchKernelGGL(k_zlarft, dim3(1), dim3(256), 0, sa, nb, gmr, gmi, g.taur + p0, g.taui + p0, tr[u],
                         ti[u]);
      W2K_STAGE(sa, "k_zlarft");
      W2K_HIP(hipEventRecord(c.bt_ready[u], sa));
      return 0;
    };
    if (nblk > 0) {
      // the second stream starts once the reflectors and Zt are in place
      W2K_HIP(hipEventRecord(c.bt_start, s));
      W2K_HIP(hipStreamWaitEvent(sa, c.bt_start, 0));
      for (int k = 0; k < std::min(nblk, 2); k++)
        if ((rc = prep(k))) return rc;
    }
    for (int k = 0; k < nblk; k++) {
      const int u = k & 1, p0 = p0_of(k), nb = std::min(ZBT, nref - p0);
      const int o = (p0 + BND) & ~15, nr = n - o;  // the block's reflectors are zero above row p0+BND
      W2K_HIP(hipStreamWaitEvent(s, c.bt_ready[u], 0));
      if ((rc = zgemm(s, 'C', 'N', nb, m, nr, 1.0, vr[u] + o, vi[u] + o, n, Zt + o, Zi + o, n, 0.0, y1r, y1i, nb, 0,
                      0, 0, ws, wsn)))
        return rc;
      if ((rc = zgemm(s, 'N', 'N', nb, m, nb, 1.0, tr[u], ti[u], nb, y1r, y1i, nb, 0.0, y2r, y2i, nb, 0, 1, 0)))
        return rc;
      if ((rc = zgemm(s, 'N', 'N', nr, m, nb, -1.0, vr[u] + o, vi[u] + o, n, y2r, y2i, nb, 1.0, Zt + o, Zi + o, n)))
        return rc;
      if (k + 2 < nblk) {
        W2K_HIP(hipEventRecord(c.bt_used[u], s));
        if ((rc = prep(k + 2))) return rc;
      }
    }
    if ((rc = sort_eigen(c, B, m))) return rc;
    hipLaunchKernelGGL(k_zgather_cols, dim3((n + 255) / 256, m), dim3(256), 0, s, n, m, B.perm, Zt, Zi, Ur, Ui);
    W2K_STAGE(s, "k_zgather_cols");
    // Z = W Zs into the (free) H storage, then interleaved into d_z
    if ((rc = zgemm3(c, s, 'N', 'N', n, m, n, 1.0, Wr, Wi, n, Ur, Ui, n, 0.0, Hr, Hi, n, 0, 1, 0))) return rc;
    hipLaunchKernelGGL(k_interleave, dim3((unsigned)((zc + 255) / 256)), dim3(256), 0, s, zc, Hr, Hi, c.d_z.p);
    W2K_STAGE(s, "k_interleave");
    W2K_HIP(hipMemcpyAsync(c.d_eig.p, B.wv, sizeof(double) * m, hipMemcpyDeviceToDevice, s));
  }
  W2K_HIP(hipEventRecord(c.ev[11], s));
  W2K_HIP(hipStreamSynchronize(s));
  take_ms(c, 3, 6, 7);
  take_ms(c, 4, 7, 8);
  take_ms(c, 5, 8, 9);
  take_ms(c, 6, 9, 10);
  take_ms(c, 7, 10, 11);
  c.ne = m;
  *ne_out = m;
  return 0;
}

}  // namespace w2k
