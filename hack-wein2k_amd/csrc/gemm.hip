// FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4_f64).
//
//   C = alpha * op(A) * op(B) + beta * C        (column-major, Fortran layout)
//
// with optional structure: the output restricted to its lower or upper
// triangle (tiles outside skipped, diagonal tiles masked per element), and
// op(A) / op(B) triangular (k range clipped per tile, elements outside the
// triangle read as zero, so the caller's storage there may hold anything).
//
// Tile 64x64x16, 256 threads = 4 wave64 in a 2x2 arrangement, each wave a
// 32x32 block of four 16x16 MFMA accumulators.  Operands staged through LDS
// k-major so that the MFMA operand reads (lane l -> row l%16, k l/16) are
// bank-conflict free; LDS double-buffered so the next k-slab's global loads
// overlap the current slab's MFMAs.  No MFMA of these kernels accumulates onto
// the one just before it, so that their results need no mfma_settle().
#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>

#include "w2k_internal.h"

namespace w2k {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int BM = 64, BN = 64, BK = 16;
constexpr int PAD = 2;  // LDS row padding (doubles)

struct GemmArgs {
  int m, n, k;
  int kslice;        // split-K: K range of one z-slice (0: no split)
  double *ws;        // split-K: m x n partial products per slice
  double alpha, beta;
  const double *A;
  int lda;
  const double *B;
  int ldb;
  double *C;
  int ldc;
  int ta, tb;        // 1 = transposed
  int tri;           // output: 0 full, 1 lower, 2 upper
  int atri, btri;    // op(A): 1 upper / 2 lower; op(B): 1 upper / 2 lower
};

// One slab of an operand for a tile: ROWS rows (of op(A); columns of op(B)) from
// r0 on by BK steps of k, by 256 work-items; T: k is the contiguous index.
// What varies over the work-items is a 32-bit offset that stays the same from
// slab to slab, so that a load costs no vector arithmetic: the kernels spent
// most of the time that the MFMAs left on 64-bit addresses, clamps and masks.
// Rows past the matrix are read as its last row (they enter only outputs that
// are not written); only a slab that ends past kend or crosses the operand's
// triangle (mode 1: zero for k < row, 2: zero for k > row) goes element by
// element.
template <int T, int ROWS>
struct Slab {
  static constexpr int C = ROWS / 16, STEP = 256 / ROWS;
  unsigned off[C];
  __device__ __forceinline__ static int row(int r) { return T ? (threadIdx.x >> 4) + 16 * r : threadIdx.x & (ROWS - 1); }
  __device__ __forceinline__ static int step(int r) { return T ? threadIdx.x & 15 : threadIdx.x / ROWS + STEP * r; }
  __device__ __forceinline__ void init(int ld, int r0, int nrow)
  {
#pragma unroll
    for (int r = 0; r < C; r++) {
      const unsigned i = min(row(r), nrow - 1 - r0);
      off[r] = 8 * (T ? step(r) + (unsigned)ld * i : i + (unsigned)ld * step(r));
    }
  }
  __device__ __forceinline__ static const double *base(const double *X, int ld, int r0, int k0)
  {
    return T ? X + k0 + (size_t)ld * r0 : X + r0 + (size_t)ld * k0;
  }
  __device__ __forceinline__ static bool whole(int r0, int k0, int kend, int mode)
  {
    return k0 + BK <= kend && (mode != 1 || k0 >= r0 + ROWS - 1) && (mode != 2 || k0 + BK - 1 <= r0);
  }
  __device__ __forceinline__ void load(const double *p, double (&v)[C]) const
  {
#pragma unroll
    for (int r = 0; r < C; r++) v[r] = *(const double *)((const char *)p + off[r]);
  }
  __device__ __forceinline__ static void load_part(const double *X, int ld, int r0, int nrow, int k0, int kend, int mode,
                                                   double (&v)[C])
  {
#pragma unroll
    for (int r = 0; r < C; r++) {
      const int i = r0 + row(r), kk = k0 + step(r);
      const bool ok = kk < kend && (mode != 1 || kk >= i) && (mode != 2 || kk <= i);
      const int ic = min(i, nrow - 1), kc = min(kk, kend - 1);
      const double x = X[T ? (size_t)kc + (size_t)ld * ic : (size_t)ic + (size_t)ld * kc];
      v[r] = ok ? x : 0.0;
    }
  }
  __device__ __forceinline__ static void store(double *s, int pitch, const double (&v)[C])
  {
#pragma unroll
    for (int r = 0; r < C; r++) s[step(r) * pitch + row(r)] = v[r];
  }
};
// Output tiles (mt x nt of them; tri 1: those with I >= J, 2: I <= J) in the order
// that the work-groups take them: strips of eight tile columns, row by row, and
// each XCD (work-groups go to them in turn) a contiguous eighth of that, so that
// what runs on an XCD at a time shares rows and columns in its L2.  Tiles
// outside a triangle have no work-group: launched as a square grid whose other
// half left at once, the lower triangle of 31 x 31 tiles put 66 tiles on one
// XCD's 64 places and took two turns (5.4 instead of 2.7 ms).  With a
// triangular operand the work of a tile depends on its place, and the order is
// plain.
constexpr int STRIP = 8, XCDS = 8;
__host__ __device__ inline int tile_count(int mt, int nt, int tri)
{
  if (tri == 0) return mt * nt;
  const int R = tri == 1 ? mt : nt, C = min(tri == 1 ? nt : mt, R);
  return C * R - C * (C - 1) / 2;
}
__device__ __forceinline__ void tile_at(int id, int mt, int nt, int tri, bool spread, int &I, int &J)
{
  if (spread) {
    const int T = tile_count(mt, nt, tri), x = id % XCDS, q = id / XCDS;
    id = x * (T / XCDS) + min(x, T % XCDS) + q;
  }
  const int R = tri == 2 ? nt : mt, C = tri == 2 ? mt : nt;  // tri 2: of the transposed triangle
  for (int c = 0; c < C; c += STRIP) {
    const int w = min(STRIP, C - c);
    const int top = tri ? min(w, max(R - c, 0)) : 0;       // rows of 1, 2, .. tiles
    const int tt = top * (top + 1) / 2, rows = tri ? max(R - c - top, 0) : R;
    const int cnt = tt + rows * w;
    if (id >= cnt) {
      id -= cnt;
      continue;
    }
    if (id < tt) {
      int t = 0;
      while (id > t) id -= ++t;
      I = c + t;
      J = c + id;
    } else {
      id -= tt;
      I = (tri ? c + top : 0) + id / w;
      J = c + id % w;
    }
    break;
  }
  if (tri == 2) {
    const int t = I;
    I = J;
    J = t;
  }
}

// the triangle of op(B) in terms of its columns
__device__ __forceinline__ int btri_mode(int btri) { return btri == 1 ? 2 : btri == 2 ? 1 : 0; }

template <bool SPLIT, bool DEEP, int TA, int TB>
__global__ __launch_bounds__(256, 2) void k_dgemm(GemmArgs g)
{
  __shared__ double As[2][BK][BM + PAD];
  __shared__ double Bs[2][BK][BN + PAD];
  const int tid = threadIdx.x;
  int i0, j0;
  tile_at(blockIdx.x, (g.m + BM - 1) / BM, (g.n + BN - 1) / BN, g.tri, !g.atri && !g.btri, i0, j0);
  i0 *= BM;
  j0 *= BN;
  // k range from operand structure
  int kbeg = 0, kend = g.k;
  if (g.atri == 1) kbeg = max(kbeg, i0);
  if (g.atri == 2) kend = min(kend, i0 + BM);
  if (g.btri == 1) kend = min(kend, j0 + BN);
  if (g.btri == 2) kbeg = max(kbeg, j0);
  if (SPLIT) {
    kbeg = max(kbeg, (int)blockIdx.z * g.kslice);
    kend = min(kend, ((int)blockIdx.z + 1) * g.kslice);
  }
  kbeg = (kbeg / BK) * BK;

  const int lane = tid & 63, wave = tid >> 6;
  const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
  const int li = lane & 15, lk = lane >> 4;

  d4 acc[2][2];
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};

  // C (beta != 0) is read before the K loop, from clamped addresses, so that
  // its loads overlap the products instead of following them
  double pc[2][2][4];
  if (!SPLIT && g.beta != 0.0) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int i = min(i0 + wi + 16 * a + li, g.m - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int j = min(j0 + wj + 16 * b + lk + 4 * r, g.n - 1);
          pc[a][b][r] = g.C[(size_t)i + (size_t)g.ldc * j];
        }
      }
  }
  const int bmode = btri_mode(g.btri);
  Slab<TA, BM> sa;
  Slab<!TB, BN> sb;
  sa.init(g.lda, i0, g.m);
  sb.init(g.ldb, j0, g.n);
  // A slab's MFMAs are shorter than its way from memory.  Where few work-groups
  // share a CU (DEEP), slabs are asked for two ahead
  struct Regs {
    double a[4], b[4];
  };
  auto whole = [&](int k0) { return sa.whole(i0, k0, kend, g.atri) && sb.whole(j0, k0, kend, bmode); };
  auto load = [&](int k0, Regs &x) {
    sa.load(sa.base(g.A, g.lda, i0, k0), x.a);
    sb.load(sb.base(g.B, g.ldb, j0, k0), x.b);
  };
  auto load_any = [&](int k0, Regs &x) {
    if (whole(k0)) {
      load(k0, x);
    } else {
      sa.load_part(g.A, g.lda, i0, g.m, k0, kend, g.atri, x.a);
      sb.load_part(g.B, g.ldb, j0, g.n, k0, kend, bmode, x.b);
    }
  };
  auto sstore = [&](int buf, const Regs &x) {
    sa.store(&As[buf][0][0], BM + PAD, x.a);
    sb.store(&Bs[buf][0][0], BN + PAD, x.b);
  };
  auto products = [&](int buf) {
#pragma unroll
    for (int kq = 0; kq < BK; kq += 4) {
      double av[2], bv[2];
      for (int a = 0; a < 2; a++) av[a] = As[buf][kq + lk][wi + 16 * a + li];
      for (int b = 0; b < 2; b++) bv[b] = Bs[buf][kq + lk][wj + 16 * b + li];
      for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[b], av[a], acc[a][b], 0, 0, 0);
    }
  };

  if (kbeg < kend) {
    Regs x, y;
    int buf = 0, k = kbeg;  // the slab in LDS
    load_any(k, x);
    sstore(0, x);
    __syncthreads();
    auto advance = [&](const Regs &x) {
      products(buf);
      sstore(buf ^ 1, x);
      __syncthreads();
      buf ^= 1;
      k += BK;
    };
    while (k + BK < kend) {
      if (DEEP && whole(k + BK) && whole(k + 2 * BK)) {
        // nothing conditional between a slab's loads and their use: the wait
        // for a slab is then not one for the slab after it
        load(k + BK, x);
        for (;;) {
          if (!whole(k + 2 * BK)) {
            advance(x);
            break;
          }
          load(k + 2 * BK, y);
          advance(x);
          if (!whole(k + 2 * BK)) {
            advance(y);
            break;
          }
          load(k + 2 * BK, x);
          advance(y);
        }
      } else {
        load_any(k + BK, x);
        advance(x);
      }
    }
    products(buf);
  }
  // epilogue: an MFMA result has rows lane/16 + 4r (r = 0..3), column lane%16
  // of each 16x16 block; with op(B) as the first operand these are columns and
  // row of C, so that sixteen lanes write 128 contiguous bytes
  for (int a = 0; a < 2; a++) {
    for (int b = 0; b < 2; b++) {
      const int i = i0 + wi + 16 * a + li;
      for (int r = 0; r < 4; r++) {
        const int j = j0 + wj + 16 * b + lk + 4 * r;
        if (i >= g.m || j >= g.n) continue;
        if (g.tri == 1 && i < j) continue;
        if (g.tri == 2 && i > j) continue;
        if (SPLIT) {
          g.ws[((size_t)blockIdx.z * g.n + j) * g.m + i] = acc[a][b][r];
          continue;
        }
        double v = g.alpha * acc[a][b][r];
        if (g.beta != 0.0) v += g.beta * pc[a][b][r];
        g.C[(size_t)i + (size_t)g.ldc * j] = v;
      }
    }
  }
}

// Large products: tile 128x128x16, 256 threads = 4 wave64 in a 2x2
// arrangement, each wave a 64x64 block of sixteen 16x16 MFMA accumulators
// (eight operand reads from LDS per sixteen MFMAs); LDS double-buffered as
// above.
constexpr int LM = 128, LN = 128, LK = 16;

template <int TA, int TB>
__global__ __launch_bounds__(256, 2) void k_dgemm_big(GemmArgs g)
{
  __shared__ double As[2][LK][LM + PAD];
  __shared__ double Bs[2][LK][LN + PAD];
  const int tid = threadIdx.x;
  int i0, j0;
  tile_at(blockIdx.x, (g.m + LM - 1) / LM, (g.n + LN - 1) / LN, g.tri, !g.atri && !g.btri, i0, j0);
  i0 *= LM;
  j0 *= LN;
  int kbeg = 0, kend = g.k;
  if (g.atri == 1) kbeg = max(kbeg, i0);
  if (g.atri == 2) kend = min(kend, i0 + LM);
  if (g.btri == 1) kend = min(kend, j0 + LN);
  if (g.btri == 2) kbeg = max(kbeg, j0);
  kbeg = (kbeg / LK) * LK;

  const int lane = tid & 63, wave = tid >> 6;
  const int wi = (wave & 1) * 64, wj = (wave >> 1) * 64;
  const int li = lane & 15, lk = lane >> 4;
  d4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};

  const int bmode = btri_mode(g.btri);
  Slab<TA, LM> sa;
  Slab<!TB, LN> sb;
  sa.init(g.lda, i0, g.m);
  sb.init(g.ldb, j0, g.n);
  double ra[8], rb[8];
  auto gload = [&](int k0) {
    const double *pa = sa.base(g.A, g.lda, i0, k0), *pb = sb.base(g.B, g.ldb, j0, k0);
    if (sa.whole(i0, k0, kend, g.atri) && sb.whole(j0, k0, kend, bmode)) {
      sa.load(pa, ra);
      sb.load(pb, rb);
    } else {
      sa.load_part(g.A, g.lda, i0, g.m, k0, kend, g.atri, ra);
      sb.load_part(g.B, g.ldb, j0, g.n, k0, kend, bmode, rb);
    }
  };
  auto sstore = [&](int buf) {
    sa.store(&As[buf][0][0], LM + PAD, ra);
    sb.store(&Bs[buf][0][0], LN + PAD, rb);
  };

  if (kbeg < kend) {
    gload(kbeg);
    sstore(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = kbeg; k0 < kend; k0 += LK) {
      const bool more = (k0 + LK < kend);
      if (more) gload(k0 + LK);
#pragma unroll
      for (int kq = 0; kq < LK; kq += 4) {
        double av[4], bv[4];
#pragma unroll
        for (int a = 0; a < 4; a++) av[a] = As[buf][kq + lk][wi + 16 * a + li];
#pragma unroll
        for (int b = 0; b < 4; b++) bv[b] = Bs[buf][kq + lk][wj + 16 * b + li];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
          for (int b = 0; b < 4; b++)
            acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[b], av[a], acc[a][b], 0, 0, 0);
      }
      if (more) {
        sstore(buf ^ 1);
        __syncthreads();
        buf ^= 1;
      }
    }
  }
  // epilogue: as in k_dgemm; C
  // (beta != 0) sixteen entries at a time, from clamped addresses
#pragma unroll
  for (int b = 0; b < 4; b++) {
    double pc[4][4];
    if (g.beta != 0.0) {
#pragma unroll
      for (int a = 0; a < 4; a++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          pc[a][r] = g.C[(size_t)min(i0 + wi + 16 * a + li, g.m - 1) +
                         (size_t)g.ldc * min(j0 + wj + 16 * b + lk + 4 * r, g.n - 1)];
    }
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + wi + 16 * a + li, j = j0 + wj + 16 * b + lk + 4 * r;
        if (i >= g.m || j >= g.n) continue;
        if (g.tri == 1 && i < j) continue;
        if (g.tri == 2 && i > j) continue;
        double v = g.alpha * acc[a][b][r];
        if (g.beta != 0.0) v += g.beta * pc[a][r];
        g.C[(size_t)i + (size_t)g.ldc * j] = v;
      }
  }
}

// C = alpha * sum_z ws[z] + beta * C, fixed summation order; with a
// triangular output (tri 1 lower, 2 upper) only that triangle is written
__global__ void k_splitk_reduce(int m, int n, int nz, const double *__restrict__ ws, double alpha, double beta,
                                double *__restrict__ C, int ldc, int tri)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= m || j >= n) return;
  if ((tri == 1 && i < j) || (tri == 2 && i > j)) return;
  double v = 0.0;
  for (int z = 0; z < nz; z++) v += ws[((size_t)z * n + j) * m + i];
  double *cp = C + (size_t)i + (size_t)ldc * j;
  v *= alpha;
  if (beta != 0.0) v += beta * *cp;
  *cp = v;
}

// ------------------------------------------------------------------ complex
// Planar complex product C = alpha op(A) op(B) + beta C (alpha, beta real)
// in one kernel: each work-group forms a 64x64 tile of both Re C and Im C
// from the same staged operands (four real MFMA products per k-step, the
// imaginary parts of op(A) and op(B) signed for conjugation at staging), so
// C is read and written once instead of four times as by four real GEMMs.
// op: transpose TA/TB (template), conjugation sa/sb = -1 (runtime); output
// restricted to a triangle (tri 1 lower, 2 upper) as in k_dgemm.
struct ZGemmArgs {
  int m, n, k;
  double alpha, beta;
  const double *Ar, *Ai;
  int lda;
  const double *Br, *Bi;
  int ldb;
  double *Cr, *Ci;
  int ldc;
  double sa, sb;  // sign of the imaginary parts of op(A), op(B)
  int tri;
};

template <int TA, int TB>
__global__ __launch_bounds__(256, 2) void k_zgemm(ZGemmArgs g)
{
  __shared__ double Ar_s[2][BK][BM + PAD], Ai_s[2][BK][BM + PAD];
  __shared__ double Br_s[2][BK][BN + PAD], Bi_s[2][BK][BN + PAD];
  const int tid = threadIdx.x;
  int i0, j0;
  tile_at(blockIdx.x, (g.m + BM - 1) / BM, (g.n + BN - 1) / BN, g.tri, true, i0, j0);
  i0 *= BM;
  j0 *= BN;
  const int lane = tid & 63, wave = tid >> 6;
  const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  // C (beta != 0) is read before the K loop, from clamped addresses, so that
  // its loads overlap the products instead of following them
  double pcr[2][2][4], pci[2][2][4];
  if (g.beta != 0.0) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int i = min(i0 + wi + 16 * a + li, g.m - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int j = min(j0 + wj + 16 * b + lk + 4 * r, g.n - 1);
          const size_t o = (size_t)i + (size_t)g.ldc * j;
          pcr[a][b][r] = g.Cr[o];
          pci[a][b][r] = g.Ci[o];
        }
      }
  }
  d4 cr[2][2], ci[2][2];
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++) {
      cr[a][b] = d4{0.0, 0.0, 0.0, 0.0};
      ci[a][b] = d4{0.0, 0.0, 0.0, 0.0};
    }
  // both planes of an operand lie alike: one set of offsets
  Slab<TA, BM> sa;
  Slab<!TB, BN> sb;
  sa.init(g.lda, i0, g.m);
  sb.init(g.ldb, j0, g.n);
  double rar[4], rai[4], rbr[4], rbi[4];
  auto gload = [&](int k0) {
    const double *par = sa.base(g.Ar, g.lda, i0, k0), *pai = sa.base(g.Ai, g.lda, i0, k0);
    const double *pbr = sb.base(g.Br, g.ldb, j0, k0), *pbi = sb.base(g.Bi, g.ldb, j0, k0);
    if (k0 + BK <= g.k) {
      sa.load(par, rar);
      sa.load(pai, rai);
      sb.load(pbr, rbr);
      sb.load(pbi, rbi);
    } else {
      sa.load_part(g.Ar, g.lda, i0, g.m, k0, g.k, 0, rar);
      sa.load_part(g.Ai, g.lda, i0, g.m, k0, g.k, 0, rai);
      sb.load_part(g.Br, g.ldb, j0, g.n, k0, g.k, 0, rbr);
      sb.load_part(g.Bi, g.ldb, j0, g.n, k0, g.k, 0, rbi);
    }
  };
  // the imaginary parts signed for conjugation
  auto sstore = [&](int buf) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      rai[r] *= g.sa;
      rbi[r] *= g.sb;
    }
    sa.store(&Ar_s[buf][0][0], BM + PAD, rar);
    sa.store(&Ai_s[buf][0][0], BM + PAD, rai);
    sb.store(&Br_s[buf][0][0], BN + PAD, rbr);
    sb.store(&Bi_s[buf][0][0], BN + PAD, rbi);
  };
  if (g.k > 0) {
    gload(0);
    sstore(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < g.k; k0 += BK) {
      const bool more = (k0 + BK < g.k);
      if (more) gload(k0 + BK);
#pragma unroll
      for (int kq = 0; kq < BK; kq += 4) {
        double ar[2], ai[2], br[2], bi[2], nbi[2];
        for (int a = 0; a < 2; a++) {
          ar[a] = Ar_s[buf][kq + lk][wi + 16 * a + li];
          ai[a] = Ai_s[buf][kq + lk][wi + 16 * a + li];
        }
        for (int b = 0; b < 2; b++) {
          br[b] = Br_s[buf][kq + lk][wj + 16 * b + li];
          bi[b] = Bi_s[buf][kq + lk][wj + 16 * b + li];
          nbi[b] = -bi[b];
        }
        // the two products of an accumulator eight MFMAs apart
        for (int a = 0; a < 2; a++)
          for (int b = 0; b < 2; b++) {
            cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(br[b], ar[a], cr[a][b], 0, 0, 0);
            ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bi[b], ar[a], ci[a][b], 0, 0, 0);
          }
        for (int a = 0; a < 2; a++)
          for (int b = 0; b < 2; b++) {
            cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(nbi[b], ai[a], cr[a][b], 0, 0, 0);
            ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(br[b], ai[a], ci[a][b], 0, 0, 0);
          }
      }
      if (more) {
        sstore(buf ^ 1);
        __syncthreads();
        buf ^= 1;
      }
    }
  }
  for (int a = 0; a < 2; a++) {
    for (int b = 0; b < 2; b++) {
      const int i = i0 + wi + 16 * a + li;
      for (int r = 0; r < 4; r++) {
        const int j = j0 + wj + 16 * b + lk + 4 * r;
        if (i >= g.m || j >= g.n) continue;
        if (g.tri == 1 && i < j) continue;
        if (g.tri == 2 && i > j) continue;
        const size_t o = (size_t)i + (size_t)g.ldc * j;
        double vr = g.alpha * cr[a][b][r], vi = g.alpha * ci[a][b][r];
        if (g.beta != 0.0) {
          vr += g.beta * pcr[a][b][r];
          vi += g.beta * pci[a][b][r];
        }
        g.Cr[o] = vr;
        g.Ci[o] = vi;
      }
    }
  }
}

// The fused kernel over one slice of K per blockIdx.z (slice z: k in
// [z kslice, (z + 1) kslice)), its raw sums into wsr/wsi[(z n + j) m + i];
// k_zsplitk_reduce adds the slices and applies alpha, beta and C.  A kernel
// of its own: folding the K range into k_zgemm changed that kernel's code
// and cost the tridiagonalisation's rank-64 updates 24 ms per 100-atom
// k-point.
template <int TA, int TB>
__global__ __launch_bounds__(256, 2) void k_zgemm_split(ZGemmArgs g, int kslice, double *__restrict__ wsr, double *__restrict__ wsi)
{
  __shared__ double Ar_s[2][BK][BM + PAD], Ai_s[2][BK][BM + PAD];
  __shared__ double Br_s[2][BK][BN + PAD], Bi_s[2][BK][BN + PAD];
  const int tid = threadIdx.x;
  int i0, j0;
  tile_at(blockIdx.x, (g.m + BM - 1) / BM, (g.n + BN - 1) / BN, g.tri, true, i0, j0);
  i0 *= BM;
  j0 *= BN;
  const int lane = tid & 63, wave = tid >> 6;
  const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  const int kbeg = blockIdx.z * kslice, kend = min(g.k, kbeg + kslice);
  d4 cr[2][2], ci[2][2];
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++) {
      cr[a][b] = d4{0.0, 0.0, 0.0, 0.0};
      ci[a][b] = d4{0.0, 0.0, 0.0, 0.0};
    }
  // both planes of an operand lie alike: one set of offsets
  Slab<TA, BM> sa;
  Slab<!TB, BN> sb;
  sa.init(g.lda, i0, g.m);
  sb.init(g.ldb, j0, g.n);
  double rar[4], rai[4], rbr[4], rbi[4];
  auto gload = [&](int k0) {
    const double *par = sa.base(g.Ar, g.lda, i0, k0), *pai = sa.base(g.Ai, g.lda, i0, k0);
    const double *pbr = sb.base(g.Br, g.ldb, j0, k0), *pbi = sb.base(g.Bi, g.ldb, j0, k0);
    if (k0 + BK <= kend) {
      sa.load(par, rar);
      sa.load(pai, rai);
      sb.load(pbr, rbr);
      sb.load(pbi, rbi);
    } else {
      sa.load_part(g.Ar, g.lda, i0, g.m, k0, kend, 0, rar);
      sa.load_part(g.Ai, g.lda, i0, g.m, k0, kend, 0, rai);
      sb.load_part(g.Br, g.ldb, j0, g.n, k0, kend, 0, rbr);
      sb.load_part(g.Bi, g.ldb, j0, g.n, k0, kend, 0, rbi);
    }
  };
  // the imaginary parts signed for conjugation
  auto sstore = [&](int buf) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      rai[r] *= g.sa;
      rbi[r] *= g.sb;
    }
    sa.store(&Ar_s[buf][0][0], BM + PAD, rar);
    sa.store(&Ai_s[buf][0][0], BM + PAD, rai);
    sb.store(&Br_s[buf][0][0], BN + PAD, rbr);
    sb.store(&Bi_s[buf][0][0], BN + PAD, rbi);
  };
  if (kbeg < kend) {
    gload(kbeg);
    sstore(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = kbeg; k0 < kend; k0 += BK) {
      const bool more = (k0 + BK < kend);
      if (more) gload(k0 + BK);
#pragma unroll
      for (int kq = 0; kq < BK; kq += 4) {
        double ar[2], ai[2], br[2], bi[2], nbi[2];
        for (int a = 0; a < 2; a++) {
          ar[a] = Ar_s[buf][kq + lk][wi + 16 * a + li];
          ai[a] = Ai_s[buf][kq + lk][wi + 16 * a + li];
        }
        for (int b = 0; b < 2; b++) {
          br[b] = Br_s[buf][kq + lk][wj + 16 * b + li];
          bi[b] = Bi_s[buf][kq + lk][wj + 16 * b + li];
          nbi[b] = -bi[b];
        }
        // the two products of an accumulator eight MFMAs apart
        for (int a = 0; a < 2; a++)
          for (int b = 0; b < 2; b++) {
            cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(br[b], ar[a], cr[a][b], 0, 0, 0);
            ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bi[b], ar[a], ci[a][b], 0, 0, 0);
          }
        for (int a = 0; a < 2; a++)
          for (int b = 0; b < 2; b++) {
            cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(nbi[b], ai[a], cr[a][b], 0, 0, 0);
            ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(br[b], ai[a], ci[a][b], 0, 0, 0);
          }
      }
      if (more) {
        sstore(buf ^ 1);
        __syncthreads();
        buf ^= 1;
      }
    }
  }
  // raw sums of this K slice (no triangle: the split needs a full output)
  for (int a = 0; a < 2; a++) {
    for (int b = 0; b < 2; b++) {
      const int i = i0 + wi + 16 * a + li;
      for (int r = 0; r < 4; r++) {
        const int j = j0 + wj + 16 * b + lk + 4 * r;
        if (i >= g.m || j >= g.n) continue;
        const size_t o = ((size_t)blockIdx.z * g.n + j) * g.m + i;
        wsr[o] = cr[a][b][r];
        wsi[o] = ci[a][b][r];
      }
    }
  }
}

// C = alpha sum_z ws[z] + beta C for both planes, fixed summation order
__global__ void k_zsplitk_reduce(int m, int n, int nz, const double *__restrict__ wsr, const double *__restrict__ wsi,
                                 double alpha, double beta, double *Cr, double *Ci, int ldc)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= m) return;
  double vr = 0.0, vi = 0.0;
  for (int z = 0; z < nz; z++) {
    const size_t o = ((size_t)z * n + j) * m + i;
    vr += wsr[o];
    vi += wsi[o];
  }
  const size_t o = (size_t)i + (size_t)ldc * j;
  vr *= alpha;
  vi *= alpha;
  if (beta != 0.0) {
    vr += beta * Cr[o];
    vi += beta * Ci[o];
  }
  Cr[o] = vr;
  Ci[o] = vi;
}

int zgemm_fused(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha, const double *Ar, const double *Ai,
                int lda, const double *Br, const double *Bi, int ldb, double beta, double *Cr, double *Ci, int ldc,
                int tri, double *ws, size_t wsn)
{
  if (m <= 0 || n <= 0) return 0;
  ZGemmArgs g;
  g.m = m; g.n = n; g.k = k > 0 ? k : 0; g.alpha = alpha; g.beta = beta;
  g.Ar = Ar; g.Ai = Ai; g.lda = lda; g.Br = Br; g.Bi = Bi; g.ldb = ldb; g.Cr = Cr; g.Ci = Ci; g.ldc = ldc;
  g.sa = (ta == 'C' || ta == 'R') ? -1.0 : 1.0;
  g.sb = (tb == 'C' || tb == 'R') ? -1.0 : 1.0;
  g.tri = tri;
  const bool ttA = (ta == 'T' || ta == 'C'), ttB = (tb == 'T' || tb == 'C');
  dim3 grid((m + BM - 1) / BM, (n + BN - 1) / BN);
  // few output tiles and a long K (the rule of dgemm's first split): K in
  // slices, partial sums in ws (two planes of m x n per slice)
  constexpr int ksl = W2K_ZSPLIT_KMIN / 2;
  const long tiles = (long)grid.x * grid.y;
  grid = dim3(tile_count(grid.x, grid.y, tri));
  if (ws && tri == 0 && tiles < 256 && k >= W2K_ZSPLIT_KMIN) {
    int nz = (int)std::min<long>((k + ksl - 1) / ksl, std::max<long>(1, 1024 / tiles));
    nz = (int)std::min<size_t>((size_t)nz, wsn / ((size_t)2 * m * n));
    if (nz >= 2) {
      const int kslice = ((k + nz - 1) / nz + BK - 1) / BK * BK;
      nz = (k + kslice - 1) / kslice;
      double *wsr = ws, *wsi = ws + (size_t)nz * m * n;
      grid.z = nz;
      if (!ttA && !ttB) hipLaunchKernelGGL((k_zgemm_split<0, 0>), grid, dim3(256), 0, s, g, kslice, wsr, wsi);
      else if (ttA && !ttB) hipLaunchKernelGGL((k_zgemm_split<1, 0>), grid, dim3(256), 0, s, g, kslice, wsr, wsi);
      else if (!ttA && ttB) hipLaunchKernelGGL((k_zgemm_split<0, 1>), grid, dim3(256), 0, s, g, kslice, wsr, wsi);
      else hipLaunchKernelGGL((k_zgemm_split<1, 1>), grid, dim3(256), 0, s, g, kslice, wsr, wsi);
      W2K_STAGE(s, "k_zgemm_split");
      hipLaunchKernelGGL(k_zsplitk_reduce, dim3((m + 255) / 256, n), dim3(256), 0, s, m, n, nz, wsr, wsi, alpha, beta,
                         Cr, Ci, ldc);
      W2K_STAGE(s, "k_zsplitk_reduce");
      return 0;
    }
  }
  if (!ttA && !ttB) hipLaunchKernelGGL((k_zgemm<0, 0>), grid, dim3(256), 0, s, g);
  else if (ttA && !ttB) hipLaunchKernelGGL((k_zgemm<1, 0>), grid, dim3(256), 0, s, g);
  else if (!ttA && ttB) hipLaunchKernelGGL((k_zgemm<0, 1>), grid, dim3(256), 0, s, g);
  else hipLaunchKernelGGL((k_zgemm<1, 1>), grid, dim3(256), 0, s, g);
  W2K_STAGE(s, "k_zgemm");
  return 0;
}

// ------------------------------------------------------------------ tile choice
// Products that both tile kernels can serve (at least 128 x 128 outputs and
// K >= 64) get their kernel from a per-device table keyed by the shape class
// (transposes, structure flags, floor(log2) of m, n and k): the first call of
// a class runs the heuristic's kernel between two events, the next call of
// the class the other kernel, and once both durations are in (read with
// hipEventQuery, never waited for) the faster one is kept.  The two kernels
// accumulate every product in the same order (MFMA steps of four along k,
// zero products only added for elements outside a triangle), so their
// results are bit-identical and the choice never changes a result.
// W2K_GEMM_TUNE=0 keeps the heuristic (128x128 tiles for outputs of at least
// 256 x 256 with K >= 256).
namespace {
struct TuneKey {
  int dev, ta, tb, tri, atri, btri, lm, ln, lk;
  bool operator<(const TuneKey &o) const
  {
    const int a[9] = {dev, ta, tb, tri, atri, btri, lm, ln, lk};
    const int b[9] = {o.dev, o.ta, o.tb, o.tri, o.atri, o.btri, o.lm, o.ln, o.lk};
    return std::lexicographical_compare(a, a + 9, b, b + 9);
  }
};
struct TuneEntry {
  int choice = -1;
  float ms[2] = {-1.f, -1.f};
  int pending[2] = {0, 0};
  hipEvent_t ev[2][2] = {{nullptr, nullptr}, {nullptr, nullptr}};
};
std::mutex tune_mu;
std::map<TuneKey, TuneEntry> tune_table;
int ilog2(int x) { return 31 - __builtin_clz((unsigned)x); }
bool tuning_on()
{
  static const bool on = !(getenv("W2K_GEMM_TUNE") && atoi(getenv("W2K_GEMM_TUNE")) == 0);
  return on;
}
}  // namespace

template <bool SPLIT, bool DEEP>
static void launch_dgemm_as(hipStream_t s, const GemmArgs &g, dim3 grid)
{
  if (!g.ta && !g.tb) hipLaunchKernelGGL((k_dgemm<SPLIT, DEEP, 0, 0>), grid, dim3(256), 0, s, g);
  else if (g.ta && !g.tb) hipLaunchKernelGGL((k_dgemm<SPLIT, DEEP, 1, 0>), grid, dim3(256), 0, s, g);
  else if (!g.ta && g.tb) hipLaunchKernelGGL((k_dgemm<SPLIT, DEEP, 0, 1>), grid, dim3(256), 0, s, g);
  else hipLaunchKernelGGL((k_dgemm<SPLIT, DEEP, 1, 1>), grid, dim3(256), 0, s, g);
}
// Slabs two ahead up to two work-groups a CU and from eight slabs on: 200^3 18.2
// -> 14.8 us; with more work-groups the
// registers cost more than the waits (lower triangle of 5951, K = 64 79 -> 93
// us; one ahead 69), and with few slabs there is nothing to run ahead of (64 x 731 x 64 7.2
// -> 9.0 us)
template <bool SPLIT>
static void launch_dgemm(hipStream_t s, const GemmArgs &g, dim3 grid)
{
  const int slabs = ((SPLIT ? g.kslice : g.k) + BK - 1) / BK;
  if ((long)grid.x * grid.z <= 512 && slabs >= 8) launch_dgemm_as<SPLIT, true>(s, g, grid);
  else launch_dgemm_as<SPLIT, false>(s, g, grid);
}

// variant 0: 64x64 tiles, 1: 128x128 tiles
static int launch_tiles(hipStream_t s, const GemmArgs &g, int variant)
{
  if (variant == 1) {
    const dim3 gb(tile_count((g.m + LM - 1) / LM, (g.n + LN - 1) / LN, g.tri));
    if (!g.ta && !g.tb) hipLaunchKernelGGL((k_dgemm_big<0, 0>), gb, dim3(256), 0, s, g);
    else if (g.ta && !g.tb) hipLaunchKernelGGL((k_dgemm_big<1, 0>), gb, dim3(256), 0, s, g);
    else if (!g.ta && g.tb) hipLaunchKernelGGL((k_dgemm_big<0, 1>), gb, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((k_dgemm_big<1, 1>), gb, dim3(256), 0, s, g);
    W2K_STAGE(s, "k_dgemm_big");
    return 0;
  }
  launch_dgemm<false>(s, g, dim3(tile_count((g.m + BM - 1) / BM, (g.n + BN - 1) / BN, g.tri)));
  W2K_STAGE(s, "k_dgemm");
  return 0;
}

static GemmArgs gemm_args(char ta, char tb, int m, int n, int k, double alpha, const double *A, int lda,
                          const double *B, int ldb, double beta, double *C, int ldc, int tri, int atri, int btri)
{
  GemmArgs g;
  g.m = m; g.n = n; g.k = k > 0 ? k : 0; g.alpha = alpha; g.beta = beta;
  g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc;
  g.ta = (ta == 'T' || ta == 't'); g.tb = (tb == 'T' || tb == 't');
  g.tri = tri; g.atri = atri; g.btri = btri;
  g.kslice = 0; g.ws = nullptr;
  return g;
}

int dgemm_tiles(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha, const double *A, int lda,
                const double *B, int ldb, double beta, double *C, int ldc, int tri, int atri, int btri, int variant)
{
  if (m <= 0 || n <= 0) return 0;
  const GemmArgs g = gemm_args(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, tri, atri, btri);
  return launch_tiles(s, g, (variant == 1 && g.k > 0) ? 1 : 0);
}

int dgemm(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha, const double *A, int lda,
          const double *B, int ldb, double beta, double *C, int ldc, int tri, int atri, int btri, double *ws,
          size_t wsn)
{
  if (m <= 0 || n <= 0) return 0;
  GemmArgs g = gemm_args(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, tri, atri, btri);
  // few output tiles and a long K: split K over z-slices so that the whole
  // chip works, then reduce the slices in a fixed order.  Products with a
  // triangular operand or output and up to 4096 tiles are split into slices
  // of about 1024 as well: their K range grows across the tiles, and
  // unsplit, the tiles with the full K set the duration.  The rule depends
  // on the shape and the workspace only, so a product is always summed the
  // same way.
  dim3 grid((m + BM - 1) / BM, (n + BN - 1) / BN);
  const long tiles = (long)grid.x * grid.y;
  const bool structured = tri || atri || btri;
  int nz = 0;
  if (ws && tri == 0 && tiles < 256 && k >= 2 * 256)
    nz = (int)std::min<long>((k + 255) / 256, std::max<long>(1, 1024 / tiles));
  else if (ws && structured && tiles >= 256 && tiles <= 4096 && k >= 1024)
    nz = std::min((k + 1023) / 1024, 4);
  if (nz >= 2) {
    nz = (int)std::min<size_t>((size_t)nz, wsn / ((size_t)m * n));
    if (nz >= 2) {
      g.kslice = ((k + nz - 1) / nz + BK - 1) / BK * BK;
      nz = (k + g.kslice - 1) / g.kslice;
      g.ws = ws;
      grid = dim3(tile_count(grid.x, grid.y, tri), 1, nz);
      launch_dgemm<true>(s, g, grid);
      W2K_STAGE(s, "k_dgemm<split>");
      hipLaunchKernelGGL(k_splitk_reduce, dim3((m + 255) / 256, n), dim3(256), 0, s, m, n, nz, ws, alpha, beta, C,
                         ldc, tri);
      W2K_STAGE(s, "k_splitk_reduce");
      return 0;
    }
  }
  int variant = (m >= 256 && n >= 256 && k >= 256) ? 1 : 0;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  // (not inside the allocation-free entry point, which creates no events)
  if (m >= 128 && n >= 128 && k >= 64 && tuning_on() && !g_arena && hipStreamIsCapturing(s, &cap) == hipSuccess &&
      cap == hipStreamCaptureStatusNone) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    const TuneKey key{dev, g.ta, g.tb, tri, atri, btri, ilog2(m), ilog2(n), ilog2(k)};
    std::unique_lock<std::mutex> lk(tune_mu);
    TuneEntry &e = tune_table[key];
    for (int v = 0; v < 2; v++) {
      if (e.pending[v] && hipEventQuery(e.ev[v][1]) == hipSuccess) {
        float ms = -1.f;
        if (hipEventElapsedTime(&ms, e.ev[v][0], e.ev[v][1]) == hipSuccess) e.ms[v] = ms;
        e.pending[v] = 0;
      }
    }
    (void)hipGetLastError();  // a query of an unfinished event is not an error here
    if (e.choice < 0 && e.ms[0] >= 0.f && e.ms[1] >= 0.f) e.choice = e.ms[1] < e.ms[0] ? 1 : 0;
    if (e.choice >= 0) {
      variant = e.choice;
    } else {
      int v = -1;
      for (int u : {variant, 1 - variant})
        if (v < 0 && e.ms[u] < 0.f && !e.pending[u]) v = u;
      if (v >= 0) {
        for (int q = 0; q < 2; q++)
          if (!e.ev[v][q]) W2K_HIP(hipEventCreate(&e.ev[v][q]));
        W2K_HIP(hipEventRecord(e.ev[v][0], s));
        int rc;
        if ((rc = launch_tiles(s, g, v))) return rc;
        W2K_HIP(hipEventRecord(e.ev[v][1], s));
        e.pending[v] = 1;
        return 0;
      }
    }
  }
  return launch_tiles(s, g, g.k > 0 ? variant : 0);
}

}  // namespace w2k
