// Two-stage tridiagonal reduction (twostage.hip), shared by the SECLR4 drivers.
#pragma once

#include "w2k_internal.h"

namespace w2k {

constexpr int BND = 32;  // bandwidth of the intermediate matrix

// complex quantities are planar (imaginary parts in the second pointer, or one
// plane further where there is one pointer)
struct SbArgs {
  int n = 0, lda = 0;
  double *ar = nullptr, *ai = nullptr;      // matrix, lower triangle; then reflectors below the band
  double *Pr = nullptr, *Pi = nullptr;      // panel buffer n x 3 BND: V, W, V
  double *Yr = nullptr, *Yi = nullptr;      // A V T, n x BND
  double *part = nullptr, *spart = nullptr; // partial sums of A V and of V^H A V
  double *T = nullptr, *G = nullptr, *S = nullptr;  // BND x BND of a panel
  double *taur = nullptr, *taui = nullptr;  // reflector scalars of Q1, n
  double *exch = nullptr;                   // sums exchanged within a panel's QR
  int *sync = nullptr;
  int qr_cap = 1 << 30;                     // most work-groups that share a panel (tests set fewer)
  double *ab = nullptr;                     // band, 2 BND x (n + 4 BND): columns of zeros past the last
  double *d = nullptr, *e = nullptr;        // tridiagonal matrix
  double *V2r = nullptr, *V2i = nullptr;    // reflectors of Q2: sweep s in column s, n x n
  double *tau2 = nullptr;                   // their scalars, [step][sweep]
  size_t ntau2 = 0;
  int *prog = nullptr;                      // finished steps per group of sweeps; entry n: the next group
  double *frag = nullptr;                   // operands of the Q2 blocks of some groups
  double *zb = nullptr;                     // vectors between the groups of Q2, 16 columns side by side
  int *q2sync = nullptr;                    // ticket and progress of their application
};

// doubles (and ints) of the work buffers that sb_buffers carves; doubles that
// sb_apply_q2 wants in Ctx::w_fac
size_t sb_doubles(int n, int cplx, size_t *ints);
size_t sb_q2_doubles(int n, size_t m, int cplx);
int sb_buffers(Ctx &c, SbArgs &g, int n, int cplx);
// A -> tridiagonal (d, e); A keeps Q1's reflectors: column i holds v_i from
// row i + BND + 1 on (v_i(i + BND) = 1), tau_i in taur/taui, i < n - BND - 1
int sb_reduce(Ctx &c, hipStream_t s, SbArgs &g, int cplx);
// while kernel timing is on: the summed time of the products of the panels
// with the trailing matrix and their number, into the context's timings
int sb_take_times(Ctx &c, hipStream_t s, int n);
// Z <- Q2 Z (n x m); overwrites the inverse iteration's factors
int sb_apply_q2(Ctx &c, hipStream_t s, SbArgs &g, int cplx, int m, double *Zr, double *Zi, int ldz);

}  // namespace w2k
