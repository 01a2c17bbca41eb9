// sx_spd.h -- inversion of a small symmetric positive definite matrix in LDS
// by one 256-thread workgroup (device code shared by the element
// condensation and the dissection factorisation).
#pragma once
#include <hip/hip_runtime.h>

namespace sx {

typedef double spd_v4d __attribute__ ((ext_vector_type (4)));

// In-place Gauss-Jordan of one 16x16 block by one wavefront: lane (r, q) =
// (lane % 16, lane / 16) holds columns 4q..4q+3 of row r.  Returns the
// 1-based index of the first pivot that is not positive, or 0.
__device__ __forceinline__ int spd_invert16 (double (&a)[4], int lane)
{
  const int r = lane & 15, q = lane >> 4;
  int bad = 0;
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const int tq = t >> 2, tc = t & 3;
    const double p = __shfl (a[tc], t + 16 * tq, 64), cv = __shfl (a[tc], r + 16 * tq, 64);
    double rv[4];
#pragma unroll
    for (int c = 0; c < 4; c++) rv[c] = __shfl (a[c], t + 16 * q, 64);
    if (!(p > 0.0) && !bad) bad = t + 1;
    const double d = 1.0 / p, f = cv * d;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const bool jc = q == tq && c == tc;
      a[c] = r == t ? (jc ? d : rv[c] * d) : jc ? -f : a[c] - f * rv[c];
    }
  }
  return bad;
}

// P (N x N, row stride LD, N = 16 nb) <- P^-1; W: scratch of 16 LD doubles,
// D: scratch of 16 * 17 doubles.  256 threads, all of them; P is complete on
// entry for every thread (the caller's barrier) and on return.  The 16-row
// pivot blocks are inverted by one wavefront, the rest are FP64 MFMA tiles:
// with pivots b, W = P_bb^-1 P_b, every other block P_ij -= P_ib W_j, where
// P_ib = +-P_bi^T (minus once i is eliminated), so only rows b are read.
// *bad (LDS, cleared by the caller): 1-based index of a bad pivot.
__device__ __forceinline__ void spd_invert (double* P, int LD, int nb, double* W, double* D,
                                            int* bad)
{
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lq = lane >> 4;
  for (int b = 0; b < nb; b++) {
    double* Pb = P + (size_t) 16 * b * LD;
    if (wave == 0) {
      double a[4];
#pragma unroll
      for (int c = 0; c < 4; c++) a[c] = Pb[lr * LD + 16 * b + 4 * lq + c];
      const int e = spd_invert16 (a, lane);
#pragma unroll
      for (int c = 0; c < 4; c++) D[lr * 17 + 4 * lq + c] = a[c];
      if (lane == 0 && e && !*bad) *bad = 16 * b + e;
    }
    __syncthreads ();
    for (int j = wave; j < nb; j += 4) {
      if (j == b) continue;
      spd_v4d acc = {};
#pragma unroll
      for (int s = 0; s < 4; s++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64 (
            D[lr * 17 + 4 * s + lq], Pb[(4 * s + lq) * LD + 16 * j + lr], acc, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; r++) W[(4 * r + lq) * LD + 16 * j + lr] = acc[r];
    }
    __syncthreads ();
    const int m = nb - 1;
    for (int t = wave; t < m * m; t += 4) {
      const int i = t / m + (t / m >= b), j = t % m + (t % m >= b);
      const double sg = i < b ? -1.0 : 1.0;
      spd_v4d acc = {};
#pragma unroll
      for (int s = 0; s < 4; s++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64 (
            sg * Pb[(4 * s + lq) * LD + 16 * i + lr], W[(4 * s + lq) * LD + 16 * j + lr], acc, 0,
            0, 0);
#pragma unroll
      for (int r = 0; r < 4; r++) P[(size_t) (16 * i + 4 * r + lq) * LD + 16 * j + lr] -= acc[r];
    }
    __syncthreads ();
    for (int j = wave; j < nb; j += 4) {
      const double sg = j < b ? 1.0 : -1.0;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 4 * r + lq;
        const double w = j == b ? D[i * 17 + lr] : W[i * LD + 16 * j + lr];
        Pb[i * LD + 16 * j + lr] = w;
        if (j != b) P[(size_t) (16 * j + lr) * LD + 16 * b + i] = sg * w;
      }
    }
    __syncthreads ();
  }
}

}  // namespace sx
