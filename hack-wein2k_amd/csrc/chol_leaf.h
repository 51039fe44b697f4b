// Cholesky factor and its inverse of one block of order 64, by one work-group
// of four waves: S = U^H U (CX: complex Hermitian, planar), X = U^-1.
//
// What such a block costs is latency, and the fetch of its code: unrolled over
// 64 steps by one wave (real) or with three barriers a step (complex) a factor
// took 38 and 91 us (the complex inverse 32 more).  Here the serial part is 16 steps at a time, by one wave,
// unrolled once and run four times: lane c holds rows r0 .. r0 + 15 of column
// c, so that the same steps factor the diagonal block and solve for the rest
// of its rows, with the row of a step handed round by readlane and no barrier;
// a second wave runs the steps on the diagonal block and the identity, which
// gives the inverse's diagonal block.  What is left are 16 x 16 products on the
// matrix cores: the trailing blocks, and X_ij = -X_ii sum_k U_ik X_kj.
#pragma once

#include "mfma.h"

namespace w2k {

__device__ __forceinline__ double rsqrt_nr(double x)
{
  double y = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * x;
  double e = fma(-h * y, y, 0.5);
  y = fma(y, e, y);
  e = fma(-h * y, y, 0.5);
  return fma(y, e, y);
}

constexpr int LEAF = 64, LEAF_LD = LEAF + 2;

template <bool CX>
struct Leaf {
  static constexpr int CP = CX ? 2 : 1;
  double m[CP][LEAF][LEAF_LD];  // S (upper triangle; identity past its order), then U
  double x[CP][LEAF][LEAF_LD];  // U^-1
  double t[3][CP][16][18];
};

// s.m -> U, s.x = U^-1, both zero below the diagonal.  A pivot that ok() turns
// down is taken as 1; returns the number (from 1) of the first such, 0 if
// none, in the first wave.
template <bool CX, class OK>
__device__ __forceinline__ int chol_leaf(Leaf<CX> &s, OK ok)
{
  constexpr int CP = CX ? 2 : 1;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q4 = lane >> 4;
  int first = 0;
  for (int i = tid; i < CP * LEAF * LEAF_LD; i += 256) (&s.x[0][0][0])[i] = 0.0;
  __syncthreads();
#pragma unroll 1
  for (int kb = 0; kb < 4; kb++) {
    const int r0 = 16 * kb;
    // lanes base .. base + 15 hold the diagonal block's columns
    const int base = w == 0 ? r0 : 0;
    double v[16], vi[CX ? 16 : 1];
    if (w < 2) {
      const int col = w == 0 ? lane : r0 + l16;
      const bool unit = w == 1 && lane >= 16;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const double a = s.m[0][r0 + r][col], b = CX ? s.m[CP - 1][r0 + r][col] : 0.0;
        v[r] = unit ? (r == l16 ? 1.0 : 0.0) : a;
        if (CX) vi[r] = unit ? 0.0 : b;
      }
    }
    // the second wave has its copy of the diagonal block before the first one
    // puts U over it
    __syncthreads();
    if (w < 2) {
#pragma unroll
      for (int j = 0; j < 16; j++) {
        const double ajj = lane_value(v[j], base + j);
        const bool good = ok(ajj);
        first = !good && first == 0 ? r0 + j + 1 : first;
        const double d = good ? ajj : 1.0, rs = rsqrt_nr(d);
        double piv = d * rs;
        piv = fma(fma(-piv, piv, d), 0.5 * rs, piv);
        auto quot = [&](double a) {
          const double q = a * rs;
          return fma(fma(-q, piv, a), rs, q);
        };
        const bool diag = lane == base + j;
        v[j] = diag ? piv : quot(v[j]);
        if (CX) vi[j] = diag ? 0.0 : quot(vi[j]);
#pragma unroll
        for (int r = j + 1; r < 16; r++) {
          const double ur = lane_value(v[j], base + r);
          if (CX) {
            const double ui = lane_value(vi[j], base + r);
            v[r] = fma(-ui, vi[j], fma(-ur, v[j], v[r]));
            vi[r] = fma(ui, v[j], fma(-ur, vi[j], vi[r]));
          } else {
            v[r] = fma(-ur, v[j], v[r]);
          }
        }
      }
      if (w == 0) {
        if (lane >= r0)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            s.m[0][r0 + r][lane] = lane >= r0 + r ? v[r] : 0.0;
            if (CX) s.m[CP - 1][r0 + r][lane] = lane >= r0 + r ? vi[r] : 0.0;
          }
      } else if (lane >= 16 && lane < 32) {
        // column l16 of U^-H
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (r >= l16) {
            s.x[0][r0 + l16][r0 + r] = v[r];
            if (CX) s.x[CP - 1][r0 + l16][r0 + r] = -vi[r];
          }
      }
    }
    __syncthreads();
    // S_ij -= U_ki^H U_kj, k = kb < i <= j
    int turn = 0;
    for (int i = kb + 1; i < 4; i++)
      for (int j = i; j < 4; j++) {
        if ((turn++ & 3) != w) continue;
        d4 ar = d4{0.0, 0.0, 0.0, 0.0}, ai = ar;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const double p = s.m[0][r0 + 4 * k + q4][16 * i + l16], q = s.m[0][r0 + 4 * k + q4][16 * j + l16];
          ar = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, ar, 0, 0, 0);
          if (CX) {
            const double p2 = s.m[CP - 1][r0 + 4 * k + q4][16 * i + l16], q2 = s.m[CP - 1][r0 + 4 * k + q4][16 * j + l16];
            ai = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q2, ai, 0, 0, 0);
            ar = __builtin_amdgcn_mfma_f64_16x16x4f64(p2, q2, ar, 0, 0, 0);
            ai = __builtin_amdgcn_mfma_f64_16x16x4f64(-p2, q, ai, 0, 0, 0);
          }
        }
        mfma_settle();
#pragma unroll
        for (int r = 0; r < 4; r++) {
          s.m[0][16 * i + q4 + 4 * r][16 * j + l16] -= ar[r];
          if (CX) s.m[CP - 1][16 * i + q4 + 4 * r][16 * j + l16] -= ai[r];
        }
      }
    __syncthreads();
  }
  // the inverse's blocks by block diagonals, one wave each
#pragma unroll 1
  for (int d = 1; d < 4; d++) {
    if (w + d < 4) {
      const int i = w, j = w + d;
      d4 ar = d4{0.0, 0.0, 0.0, 0.0}, ai = ar;
#pragma unroll 1
      for (int kb = i + 1; kb <= j; kb++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int kk = 16 * kb + 4 * k + q4;
          const double p = s.m[0][16 * i + l16][kk], q = s.x[0][kk][16 * j + l16];
          ar = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, ar, 0, 0, 0);
          if (CX) {
            const double p2 = s.m[CP - 1][16 * i + l16][kk], q2 = s.x[CP - 1][kk][16 * j + l16];
            ai = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q2, ai, 0, 0, 0);
            ar = __builtin_amdgcn_mfma_f64_16x16x4f64(-p2, q2, ar, 0, 0, 0);
            ai = __builtin_amdgcn_mfma_f64_16x16x4f64(p2, q, ai, 0, 0, 0);
          }
        }
      mfma_settle();
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s.t[i][0][q4 + 4 * r][l16] = ar[r];
        if (CX) s.t[i][CP - 1][q4 + 4 * r][l16] = ai[r];
      }
      wave_sync();
      ar = ai = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const double p = -s.x[0][16 * i + l16][16 * i + 4 * k + q4], q = s.t[i][0][4 * k + q4][l16];
        ar = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, ar, 0, 0, 0);
        if (CX) {
          const double p2 = -s.x[CP - 1][16 * i + l16][16 * i + 4 * k + q4], q2 = s.t[i][CP - 1][4 * k + q4][l16];
          ai = __builtin_amdgcn_mfma_f64_16x16x4f64(p, q2, ai, 0, 0, 0);
          ar = __builtin_amdgcn_mfma_f64_16x16x4f64(-p2, q2, ar, 0, 0, 0);
          ai = __builtin_amdgcn_mfma_f64_16x16x4f64(p2, q, ai, 0, 0, 0);
        }
      }
      mfma_settle();
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s.x[0][16 * i + q4 + 4 * r][16 * j + l16] = ar[r];
        if (CX) s.x[CP - 1][16 * i + q4 + 4 * r][16 * j + l16] = ai[r];
      }
    }
    __syncthreads();
  }
  return first;
}

}  // namespace w2k
