// sx_tree.hip -- dissection solve of the condensed FP64 systems (the matrix
// of src/matrix.cpp:132-267, solved by the reference with a banded
// Cholesky, src/field.cpp:672-709).
//
// The banded factor makes a solve a chain of 64-row block steps; its length
// (132 steps at 4,208 rows, 72 for the twisted split) bounds the solve, not
// its bytes.  Here the elements are split recursively (sx_tree_plan.cpp)
// and the unknowns eliminated front by front, a level of fronts at once:
// 1 to 5 levels instead of tens of block steps.  A front with eliminated
// unknowns K and boundary B has its operators formed at set-up,
//   E = A_KK^-1 A_KB,   A_KK^-1,   S = A_BB - A_KB^T E  (passed up),
// and a solve is two dense products per front,
//   up:    v_K = r_K + (parts' contributions),  c_B = (parts') - E^T v_K
//   down:  x_K = A_KK^-1 v_K - E x_B
// so every level is one launch of independent products on FP64 MFMA tiles.
// Fronts of one class share their operators (a uniform 16x16-element mesh
// has a few classes per level), so up to 16 right-hand-side columns of a
// class are taken by one tile and the operators come from the L2s.
//
// Operators are stored in MFMA fragment order: per 16-row block and pair of
// k steps, [lane][2] doubles, so a wavefront reads 1 KB by 16-byte loads.
#include <algorithm>
#include <cstdlib>
#include <string>
#include <vector>

#include "sx_internal.h"
#include "sx_spd.h"
#include "sx_tree.h"

namespace sx {
namespace {

typedef double v4d __attribute__ ((ext_vector_type (4)));

constexpr int TB = 64;                 // pivot block and tile of the factorisation

// ---------------------------------------------------------------------------
// Set-up
// ---------------------------------------------------------------------------
// Front matrices of a level: each entry the sum of its parts' entries
// (elements: their condensed matrix; fronts: their trailing block).  In a
// singular mode (the last unknown dropped) the pinned unknown is replaced
// by the identity.  Front matrices are kept by their upper 64x64 tiles only
// (diagonal tiles whole): they stay symmetric up to the sign the elimination
// gives (k_tree_update).
__device__ __forceinline__ bool upper_tile (int i, int j) { return (i >> 6) <= (j >> 6); }

__global__ __launch_bounds__(256) void k_tree_assemble (
    const TreeClass* __restrict__ cls, int cls0, const TreeChild* __restrict__ child,
    const int* __restrict__ map, const double* __restrict__ Sel, int next, int nec,
    const double* __restrict__ Fc, size_t fcs, double* F, size_t fs,
    const int* __restrict__ nsolve, int nsfull)
{
  const TreeClass C = cls[cls0 + blockIdx.y];
  const int mode = blockIdx.z, n = C.k + C.b;
  const bool pinned = C.pin >= 0 && nsolve[mode] < nsfull;
  for (size_t e = (size_t) blockIdx.x * 256 + threadIdx.x; e < (size_t) n * n;
       e += (size_t) gridDim.x * 256) {
    const int i = (int) (e / n), j = (int) (e % n);
    if (!upper_tile (i, j)) continue;
    double s = 0.0;
    if (pinned && (i == C.pin || j == C.pin)) {
      s = i == j ? 1.0 : 0.0;
    } else {
      for (int c = 0; c < C.nch; c++) {
        const TreeChild ch = child[C.ch0 + c];
        const int a = map[ch.map0 + i], b = map[ch.map0 + j];
        if (a < 0 || b < 0) continue;
        if (ch.front) {
          const TreeClass D = cls[ch.cls];
          const int nd = D.k + D.b, r = D.k + a, t = D.k + b;
          const bool up = upper_tile (r, t);
          s += Fc[(size_t) mode * fcs + D.foff + (size_t) (up ? r : t) * nd + (up ? t : r)];
        } else {
          s += Sel[(((size_t) mode * nec + ch.cls) * next + a) * next + b];
        }
      }
    }
    F[(size_t) mode * fs + C.foff + e] = s;
  }
}

// One step of the in-place Gauss-Jordan elimination of a front's first k
// unknowns, pivots P = [p0, p0 + pb): this kernel inverts the pivot block
// and forms, for a tile of 64 columns, R = F_P (the rows as they are) and
// W = F_PP^-1 F_P (F_PP^-1 itself in the columns of P) into RW (rows of ldw,
// zero past n).  Every tile's workgroup inverts the block for itself, so a
// step is two launches.  It is bound by that inversion's chain of pivots
// (one wavefront, 16 at a time): 38 us a step with the 64 pivots one after
// another, a barrier each.
__global__ __launch_bounds__(256) void k_tree_panel (
    const TreeClass* __restrict__ cls, int cls0, const double* __restrict__ F, size_t fs,
    double* RW, int ldw, int step, int* status)
{
  const TreeClass C = cls[cls0 + blockIdx.y];
  const int mode = blockIdx.z, n = C.k + C.b, p0 = TB * step;
  const int pb = min (TB, C.k - p0), c0 = TB * blockIdx.x;
  if (pb <= 0 || c0 >= n) return;
  constexpr int LD = TB + 2;
  __shared__ double piv[TB * LD], Rs[TB * LD], Wb[16 * LD], D[16 * 17];
  __shared__ int bad;
  const double* Fm = F + (size_t) mode * fs + C.foff;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (tid == 0) bad = 0;
  // the pivot block (identity past pb) and the rows of P in this tile's
  // columns, every load unconditional
  // (columns already eliminated: F_Pj = -F_jP^T, read from the upper tiles)
  const bool done = c0 < p0;
  double x[16], y[16];
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int r = 4 * q + wave, rr = p0 + min (r, pb - 1);
    x[q] = Fm[(size_t) rr * n + p0 + min (lane, pb - 1)];
    const size_t at = done ? (size_t) (c0 + r) * n + p0 + min (lane, pb - 1)
                           : (size_t) rr * n + min (c0 + lane, n - 1);
    y[q] = Fm[at];
  }
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int r = 4 * q + wave;
    piv[r * LD + lane] = r < pb && lane < pb ? x[q] : r == lane ? 1.0 : 0.0;
    if (done) Rs[lane * LD + r] = lane < pb ? -y[q] : 0.0;
    else Rs[r * LD + lane] = r < pb && c0 + lane < n ? y[q] : 0.0;
  }
  __syncthreads ();
  spd_invert (piv, LD, (pb + 15) / 16, Wb, D, &bad);
  if (tid == 0 && bad && blockIdx.x == 0) atomicMax (status + mode, p0 + bad);
  double* Rg = RW + ((size_t) mode * gridDim.y + blockIdx.y) * 2 * TB * ldw;
  double* Wg = Rg + (size_t) TB * ldw;
  v4d acc[4] = {};
#pragma unroll
  for (int s = 0; s < TB / 4; s++) {
    const double av = piv[(16 * wave + (lane & 15)) * LD + 4 * s + (lane >> 4)];
#pragma unroll
    for (int q = 0; q < 4; q++)
      acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64 (
          av, Rs[(4 * s + (lane >> 4)) * LD + 16 * q + (lane & 15)], acc[q], 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * wave + 4 * r + (lane >> 4), j = c0 + 16 * q + (lane & 15);
      const int jp = j - p0;
      Rg[(size_t) i * ldw + j] = Rs[i * LD + j - c0];
      Wg[(size_t) i * ldw + j] = jp >= 0 && jp < pb ? piv[i * LD + jp] : acc[q][r];
    }
}

// The rest of the step, one 64x64 tile of the front per workgroup:
//   i, j not in P:  F_ij -= F_iP W_j,  F_iP = s_i R_i^T
//   i in P:         F_ij  = W_ij
//   j in P:         F_ij  = -s_i W_ji
// with s_i = -1 for unknowns already eliminated (i < p0), +1 otherwise: the
// matrix stays symmetric up to that sign, so only upper tiles are formed.
// R and W are padded to whole tiles, so every load is unconditional and
// issued before the products (46 -> 25 us a step at 96 fronts of 370, 17 with upper tiles only).
__global__ __launch_bounds__(256) void k_tree_update (
    const TreeClass* __restrict__ cls, int cls0, double* F, size_t fs,
    const double* __restrict__ RW, int ldw, int step, int nt)
{
  const TreeClass C = cls[cls0 + blockIdx.y];
  const int mode = blockIdx.z, n = C.k + C.b, p0 = TB * step;
  const int pb = min (TB, C.k - p0);
  // upper tile blockIdx.x of nt (nt + 1) / 2, by rows
  int ti = 0, tj = blockIdx.x;
  while (tj >= nt - ti) { tj -= nt - ti; ti++; }
  const int i0 = TB * ti, j0 = TB * (ti + tj);
  if (pb <= 0 || i0 >= n || j0 >= n) return;
  constexpr int LD = TB + 2;
  __shared__ double Rs[TB * LD], Ws[TB * LD];
  const double* Rg = RW + ((size_t) mode * gridDim.y + blockIdx.y) * 2 * TB * ldw;
  const double* Wg = Rg + (size_t) TB * ldw;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wi = 32 * (wave & 1), wj = 32 * (wave >> 1);
  double* Fm = F + (size_t) mode * fs + C.foff;
  double x[16], y[16], f[16], wt[16];
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const size_t r = (size_t) (4 * q + wave) * ldw;
    x[q] = Rg[r + i0 + lane];
    y[q] = Wg[r + j0 + lane];
  }
  const bool tp = j0 < p0 + pb && j0 + TB > p0;        // the tile holds columns of P
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int i = i0 + wi + 16 * (q >> 3) + 4 * (q & 3) + (lane >> 4),
              j = j0 + wj + 16 * ((q >> 2) & 1) + (lane & 15);
    f[q] = Fm[(size_t) min (i, n - 1) * n + min (j, n - 1)];
    wt[q] = tp ? Wg[(size_t) min (max (j - p0, 0), TB - 1) * ldw + i] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int r = 4 * q + wave;
    Rs[r * LD + lane] = i0 + lane < p0 ? -x[q] : x[q];
    Ws[r * LD + lane] = y[q];
  }
  __syncthreads ();
  v4d acc[2][2] = {};
  const int ks = (pb + 3) / 4;
  for (int s = 0; s < ks; s++) {
    const double* ra = Rs + (4 * s + (lane >> 4)) * LD + wi + (lane & 15);
    const double* wb = Ws + (4 * s + (lane >> 4)) * LD + wj + (lane & 15);
    const double a0 = ra[0], a1 = ra[16], b0 = wb[0], b1 = wb[16];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64 (a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64 (a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64 (a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64 (a1, b1, acc[1][1], 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int il = wi + 16 * (q >> 3) + 4 * (q & 3) + (lane >> 4),
              jl = wj + 16 * ((q >> 2) & 1) + (lane & 15);
    const int i = i0 + il, j = j0 + jl;
    if (i >= n || j >= n) continue;
    const bool ip = i >= p0 && i < p0 + pb, jp = j >= p0 && j < p0 + pb;
    const double v = ip   ? Ws[(i - p0) * LD + jl]
                     : jp ? (i < p0 ? wt[q] : -wt[q])
                          : f[q] - acc[q >> 3][(q >> 2) & 1][q & 3];
    Fm[(size_t) i * n + j] = v;
  }
}

// Operators of a level in fragment order.  Forward: rows B, k steps over K,
// entry E[kk][row].  Backward: rows K, k steps over [K | B], entries
// A_KK^-1[row][j] and -E[row][j-k].
__global__ __launch_bounds__(256) void k_tree_operators (
    const TreeClass* __restrict__ cls, int cls0, const double* __restrict__ F, size_t fs,
    double* ops, size_t os)
{
  const TreeClass C = cls[cls0 + blockIdx.y];
  const int mode = blockIdx.z, n = C.k + C.b;
  const size_t nf = (size_t) ((C.b + 15) / 16) * C.mfp * 128,
               nb = (size_t) ((C.k + 15) / 16) * C.mbp * 128;
  const double* Fm = F + (size_t) mode * fs + C.foff;
  double* O = ops + (size_t) mode * os;
  for (size_t e = (size_t) blockIdx.x * 256 + threadIdx.x; e < nf + nb;
       e += (size_t) gridDim.x * 256) {
    const bool fw = e < nf;
    const size_t q = fw ? e : e - nf;
    const int np = fw ? C.mfp : C.mbp;
    const int h = (int) (q & 1), l = (int) ((q >> 1) & 63), pair = (int) ((q >> 7) % np),
              rb = (int) ((q >> 7) / np);
    const int row = 16 * rb + (l & 15), kk = 4 * (2 * pair + h) + (l >> 4);
    double v = 0.0;
    if (fw) {
      if (row < C.b && kk < C.k) v = Fm[(size_t) kk * n + C.k + row];
      O[C.mf + q] = v;
    } else {
      if (row < C.k && kk < n)
        v = upper_tile (row, kk) ? Fm[(size_t) row * n + kk] : Fm[(size_t) kk * n + row];
      O[C.mb + q] = kk < C.k ? v : -v;
    }
  }
}

// ---------------------------------------------------------------------------
// Solve: one launch per level and direction
// ---------------------------------------------------------------------------
struct TreeArgs {
  const TreeItem* item;
  int nitem, nmodes, xcd;
  const int *gk, *gb, *tgt;
  const double* ops;
  size_t os;
  const double* in;                    // [mode][nr][nsp] by position
  double *rhs, *v, *cb;                // [mode][nr][nmax] by node, [..][nsp], [..][slots]
  double* sum;                         // solution added to here as well (or null)
  int nmax, nsp, nr;
  size_t slots;
  const int* nsolve;
};

enum { T_UP = 0, T_DOWN = 1, T_ROOT = 2 };

// UP: forward product of a level, DOWN: backward; ROOT: backward of the
// root, which gathers its v_K itself (no forward product: no boundary).
// A level is bound by its chain of dependent loads, not by its bytes: the
// work item; then the operator's fragments, the right-hand sides and the
// parts' contributions (W neighbouring values each); DOWN one more, the
// solution at the boundary nodes.  Every load of a round is issued before
// any of it is used.
template <int DIR, int W>
__device__ __forceinline__ void tree_level_body (const TreeArgs& T)
{
  extern __shared__ double sm[];
  // a mode's work stays on one XCD where the modes fill all eight: its
  // tiles of one class then share the operators in that L2
  int mode, item;
  if (T.xcd) {
    const int q = blockIdx.x >> 3;
    mode = 8 * (q / T.nitem) + (blockIdx.x & 7);
    item = q % T.nitem;
    if (mode >= T.nmodes) return;
  } else {
    mode = blockIdx.x / T.nitem;
    item = blockIdx.x % T.nitem;
  }
  const TreeItem it = T.item[item];
  const int nr = T.nr, ns = T.nsolve[mode];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane (tid >> 6);
  const int k = it.k, n = it.k + it.b;
  const int K = DIR == T_DOWN ? n : k, rows = DIR == T_UP ? it.b : k;
  const int np = (K + 7) / 8;
  const int ncol = it.nf * nr, ldx = ncol | 1;
  // wavefront: k steps [q0, q1) of the row blocks rw, rw + step, ...
  const int kw = it.kw, kp = wave & (kw - 1), step = 4 / kw, rw = wave / kw;
  const int turns = (it.nrb + step - 1) / step;
  const double2* A = (const double2*) (T.ops + (size_t) mode * T.os + it.op) +
                     (size_t) (it.rb0 + rw) * np * 64 + lane;
  const int q0 = np * kp / kw, q1 = np * (kp + 1) / kw;
  constexpr int U = 8;
  double2 a[U];
#pragma unroll
  for (int u = 0; u < U; u++)
    a[u] = rw < it.nrb && q0 + u < q1 ? A[(size_t) (q0 + u) * 64] : make_double2 (0.0, 0.0);
  // the column operand [k rows padded to 8][ldx]; G entries a thread in
  // flight (entry e: row e % K of column e / K, by a float quotient that is
  // exact for K * 16 < 2^16 entries)
  const size_t mrow = (size_t) mode * nr;
  const int Kp = np * 8, ne = K * ncol;
  const float rK = 1.0f / (float) K;
  constexpr int G = DIR == T_DOWN ? 8 : 6;
  for (int e0 = tid; e0 < ne; e0 += 256 * G) {
    double x[G];
    int g[G], cl[G], kk[G];
    size_t r[G];
#pragma unroll
    for (int u = 0; u < G; u++) {
      const int e = min (e0 + 256 * u, ne - 1);
      cl[u] = (int) (((float) e + 0.5f) * rK);
      kk[u] = e - cl[u] * K;
      const int j = cl[u] / nr;
      r[u] = mrow + cl[u] - j * nr;
      g[u] = j;
    }
    if (DIR == T_DOWN) {
      int node[G];
#pragma unroll
      for (int u = 0; u < G; u++)
        node[u] = T.gb[it.offb + (kk[u] < k ? 0 : g[u] * it.b + kk[u] - k)];
#pragma unroll
      for (int u = 0; u < G; u++) {
        const double* p = kk[u] < k ? T.v + r[u] * T.nsp + it.offk + g[u] * k + kk[u]
                                    : T.rhs + r[u] * T.nmax + min (node[u], ns - 1);
        x[u] = *p;
      }
#pragma unroll
      for (int u = 0; u < G; u++)
        if (kk[u] >= k && node[u] >= ns) x[u] = 0.0;
    } else {
      double2 w[G][W / 2];
#pragma unroll
      for (int u = 0; u < G; u++) {
        x[u] = T.in[r[u] * T.nsp + it.offk + g[u] * k + kk[u]];
        if (it.src) {
          const double2* cb = (const double2*) (T.cb + r[u] * T.slots) +
                              (size_t) (it.offn + g[u] * n + kk[u]) * (W / 2);
#pragma unroll
          for (int q = 0; q < W / 2; q++) w[u][q] = cb[q];
        }
      }
#pragma unroll
      for (int u = 0; u < G; u++) {
        if (it.src)
#pragma unroll
          for (int q = 0; q < W / 2; q++) x[u] += w[u][q].x + w[u][q].y;
        if (DIR == T_UP && it.rb0 == 0 && e0 + 256 * u < ne)
          T.v[r[u] * T.nsp + it.offk + g[u] * k + kk[u]] = x[u];
      }
    }
#pragma unroll
    for (int u = 0; u < G; u++)
      if (e0 + 256 * u < ne) sm[kk[u] * ldx + cl[u]] = x[u];
  }
  for (int e = tid; e < (Kp - K) * ldx; e += 256) sm[K * ldx + e] = 0.0;
  // this lane's outputs: rows 16 rb + 4 i + lane/16 of column lane%16
  // (columns past ncol read a valid one, their results are not stored)
  const int col = min (lane & 15, ncol - 1), oj = col / nr;
  const size_t orow = mrow + col - oj * nr;
  const bool mine = kp == 0 && (lane & 15) < ncol;
  const double* X = sm + (lane >> 4) * ldx + col;
  double* red = sm + (size_t) Kp * ldx;
  __syncthreads ();
  for (int t = 0; t < turns; t++) {
    const int rl = rw + t * step, rb = it.rb0 + rl;
    const bool active = rl < it.nrb, more = rl + step < it.nrb;
    double base[4];
    int to[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = 16 * rb + 4 * i + (lane >> 4);
      const bool ok = active && mine && row < rows;
      to[i] = -1;
      base[i] = 0.0;
      if (DIR == T_UP) {
        if (ok) to[i] = T.tgt[it.offb + oj * it.b + row];
        if (ok && it.src) {
          const double2* c = (const double2*) (T.cb + orow * T.slots) +
                             (size_t) (it.offn + oj * n + k + row) * (W / 2);
          double2 w[W / 2];
#pragma unroll
          for (int q = 0; q < W / 2; q++) w[q] = c[q];
#pragma unroll
          for (int q = 0; q < W / 2; q++) base[i] += w[q].x + w[q].y;
        }
      } else if (ok) {
        to[i] = T.gk[it.offk + oj * k + row];
      }
    }
    v4d acc0 = {}, acc1 = {};
    if (active) {
      const double2* An = A + (size_t) step * np * 64;
      for (int q = q0; q < q1; q += U) {
        double2 b[U];
#pragma unroll
        for (int u = 0; u < U; u++) b[u] = a[u];
        if (q + U < q1) {
#pragma unroll
          for (int u = 0; u < U; u++)
            if (q + U + u < q1) a[u] = A[(size_t) (q + U + u) * 64];
        } else if (more) {             // the next row block's first steps
#pragma unroll
          for (int u = 0; u < U; u++)
            if (q0 + u < q1) a[u] = An[(size_t) (q0 + u) * 64];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          if (q + u < q1) {
            const double* x = X + (size_t) 8 * (q + u) * ldx;
            acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64 (b[u].x, x[0], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64 (b[u].y, x[4 * ldx], acc1, 0, 0, 0);
          }
      }
      A = An;
    }
    v4d acc = acc0 + acc1;
    if (kw > 1) {
      if (t) __syncthreads ();         // the last turn's partial tiles are read
      if (kp)
#pragma unroll
        for (int i = 0; i < 4; i++) red[(wave * 4 + i) * 64 + lane] = acc[i];
      __syncthreads ();
      if (kp == 0)
        for (int p = 1; p < kw; p++)
#pragma unroll
          for (int i = 0; i < 4; i++) acc[i] += red[((wave + p) * 4 + i) * 64 + lane];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (to[i] < 0) continue;
      if (DIR == T_UP) {
        T.cb[orow * T.slots + to[i]] = base[i] - acc[i];
      } else if (to[i] < ns) {
        T.rhs[orow * T.nmax + to[i]] = acc[i];
        if (T.sum) T.sum[orow * T.nmax + to[i]] += acc[i];
      }
    }
  }
}

template <int DIR, int W>
__global__ __launch_bounds__(256) void k_tree_level (TreeArgs T)
{
  tree_level_body<DIR, W> (T);
}
template <int DIR, int W> struct FnTreeLevel {
  __device__ __forceinline__ void operator() (const TreeArgs& T) const
  { tree_level_body<DIR, W> (T); }
};

// Entries of a mode's assembled matrix, each pair (row <= column) summed
// over its elements in the band assembly's order
__global__ __launch_bounds__(256) void k_tree_entries (int npairs, const int* __restrict__ pptr,
                                                       const int* __restrict__ psrc,
                                                       const double* __restrict__ S, double* val)
{
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= npairs) return;
  double s = 0.0;
  for (int c = pptr[p]; c < pptr[p + 1]; c++) s += S[psrc[c]];
  val[p] = s;
}

// out = b - A x for one mode's nr right-hand sides (b by bperm, out by
// operm: the positions of their dissections), accumulated in twice
// the working precision (error-free products and sums); a wavefront per row
__device__ __forceinline__ void k_tree_residual_body (
    int ns, int nmax, int nr, const int* __restrict__ ptr, const int* __restrict__ col,
    const int* __restrict__ pair, const double* __restrict__ val, const double* __restrict__ b,
    int ldb, const int* __restrict__ bperm, const double* __restrict__ x, double* out, int ldo,
    const int* __restrict__ operm)
{
#pragma clang fp contract(off)
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= ns) return;
  auto two_sum = [] (double& s, double& e, double v) {
    const double t = s + v, z = t - s;
    e += (s - (t - z)) + (v - z);
    s = t;
  };
  for (int r = 0; r < nr; r++) {
    double s = 0.0, e = 0.0;
    for (int c = ptr[row] + lane; c < ptr[row + 1]; c += 64) {
      const int j = col[c];
      if (j >= ns) continue;
      const double a = -val[pair[c]], xv = x[(size_t) r * nmax + j], q = a * xv;
      e += __builtin_fma (a, xv, -q);
      two_sum (s, e, q);
    }
    for (int o = 32; o > 0; o >>= 1) {
      const double so = __shfl_xor (s, o, 64), eo = __shfl_xor (e, o, 64);
      two_sum (s, e, so);
      e += eo;
    }
    if (lane == 0) {
      two_sum (s, e, b[(size_t) r * ldb + (bperm ? bperm[row] : row)]);
      out[(size_t) r * ldo + operm[row]] = s + e;
    }
  }
}

__global__ __launch_bounds__(256) void k_tree_residual (
    int ns, int nmax, int nr, const int* __restrict__ ptr, const int* __restrict__ col,
    const int* __restrict__ pair, const double* __restrict__ val, const double* __restrict__ b,
    int ldb, const int* __restrict__ bperm, const double* __restrict__ x, double* out, int ldo,
    const int* __restrict__ operm)
{
  k_tree_residual_body (ns, nmax, nr, ptr, col, pair, val, b, ldb, bperm, x, out, ldo, operm);
}
struct FnTreeResidual {
  template <typename... A> __device__ __forceinline__ void operator() (A... a) const
  { k_tree_residual_body (a...); }
};
struct FnTreeKeep {
  __device__ __forceinline__ void operator() (double* to, const double* from, int n) const
  {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) to[i] = from[i];
  }
};

// h on the device, unless it is there already
template <typename V> int upload (V** d, const std::vector<V>& h)
{
  if (*d || h.empty ()) return SX_OK;
  V* p = nullptr;
  SX_HIP (dev_malloc (&p, sizeof (V) * h.size ()));
  const hipError_t e = hipMemcpy (p, h.data (), sizeof (V) * h.size (), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void) hipFree (p);
    return hip_fail (e, "hipMemcpy");
  }
  *d = p;
  return SX_OK;
}

}  // namespace

// A mesh's plan for one mode count and share with its tables on the device
struct TreeDev {
  TreePlan P;
  int nmodes = 0, share = 1;
  bool ok = false, slower = false;     // slower: the band solve is the faster one
  TreeClass* cls = nullptr;
  TreeChild* child = nullptr;
  TreeItem* item = nullptr;
  int *map = nullptr, *gk = nullptr, *gb = nullptr, *tgt = nullptr, *perm = nullptr;
};

void tree_free (TreeDev* t)
{
  if (!t) return;
  void* p[] = {t->cls, t->child, t->item, t->map, t->gk, t->gb, t->tgt, t->perm};
  for (void* q : p) if (q) (void) hipFree (q);
  delete t;
}

// The environment variables that choose a band layout keep the band solve.
static bool band_forced ()
{
  for (const char* v : {"SX_BAND_TWIST", "SX_BAND_UNIT", "SX_BAND_SPLIT", "SX_BAND_SWEEP",
                        "SX_BAND_BLOCK", "SX_BAND_LL", "SX_PANEL_NR"})
    if (std::getenv (v)) return true;
  return false;
}

// The band solve stays for systems outside the dissection's bounds: bands
// past 768 (refused as before by the band solve), a mesh tree_plan does not
// suit, operators of more than 24 GB, and more classes than a grid holds.  always: also under a variable
// that chooses a band layout.
constexpr size_t TREE_OPS_MAX = (size_t) 3 << 30;      // doubles
constexpr int TREE_GRID_MAX = 65535;   // classes and modes are y and z of the set-up's grids
// More than TREE_FEW_MODES modes: also where the band solve is estimated
// faster (up to 32 modes its twisted and split sweeps lost everywhere
// measured; with many its chain costs little next to the fronts' many
// workgroups).  Whole solves, band / dissection: 5x5 elements N_P=6, 128
// modes 40 / 53 us; 8x8 N_P=8, 128 modes 80 / 91 us; uniform 12x24 N_P=6, 256
// modes, which stays, 411 / 315 us.
constexpr double TREE_BAND = 0.95;

int tree_prepare (sx_mesh* m, int nmodes, TreeDev** out, bool always, int share)
{
  *out = nullptr;
  if ((!always && band_forced ()) || m->nband > 768) return SX_OK;
  std::lock_guard<std::mutex> lock (m->tree_mu);
  TreeDev* t = nullptr;
  for (TreeDev* q : m->trees)
    if (q->nmodes == nmodes && q->share == share) t = q;
  if (!t) {
    t = new TreeDev;
    t->nmodes = nmodes;
    t->share = share;
    m->trees.push_back (t);
    size_t f = 0;
    t->ok = tree_plan (m, nmodes, share, t->P);
    int ncls = 0;
    for (const TreeLevel& L : t->P.lev) {
      f = std::max (f, L.fsize);
      ncls = std::max (ncls, L.ncls);
    }
    t->ok = t->ok && t->P.ops * nmodes <= TREE_OPS_MAX && f * nmodes <= TREE_OPS_MAX &&
            ncls <= TREE_GRID_MAX && nmodes <= TREE_GRID_MAX;
    if (!t->ok) t->P = TreePlan ();
    t->slower = nmodes > TREE_FEW_MODES && band_us (m, nmodes) < TREE_BAND * t->P.est_us;
  }
  if (!t->ok || (t->slower && !always)) return SX_OK;
  // (the tables of a plan whose upload failed are tried again)
  int rc;
  if ((rc = upload (&t->cls, t->P.cls)) || (rc = upload (&t->child, t->P.child)) ||
      (rc = upload (&t->item, t->P.item)) || (rc = upload (&t->map, t->P.map)) ||
      (rc = upload (&t->gk, t->P.gk)) || (rc = upload (&t->gb, t->P.gb)) ||
      (rc = upload (&t->tgt, t->P.tgt)) || (rc = upload (&t->perm, t->P.perm)))
    return rc;
  *out = t;
  return SX_OK;
}

// Scratch of a factorisation of nm modes: the front matrices of two levels
// and a step's rows
struct Scratch { size_t f0, f1, rw; };
static Scratch scratch (const TreePlan& P)
{
  Scratch z {0, 0, 0};
  for (size_t j = 0; j < P.lev.size (); j++) {
    const TreeLevel& L = P.lev[j];
    size_t& f = j & 1 ? z.f1 : z.f0;
    f = std::max (f, L.fsize);
    z.rw = std::max (z.rw, (size_t) L.ncls * 2 * TB * ((L.nmax + TB - 1) / TB * TB));
  }
  return z;
}

size_t tree_scratch (const TreeDev* t, int nm)
{
  const Scratch z = scratch (t->P);
  return (z.f0 + z.f1 + z.rw) * nm;
}

size_t tree_ops (const TreeDev* t) { return t->P.ops; }
size_t tree_slots (const TreeDev* t) { return t->P.slots; }

// Factorisation of nm modes: the levels from the elements to the root (Sel:
// the condensed element matrices [nm][nclass][next][next]) into ops
// [nm][tree_ops]; buf: tree_scratch doubles.  status[mode] > 0: a pivot was
// not positive.
static int factor (const TreeDev* t, const sx_mesh* m, int nm, const int* d_nsolve,
                   const double* Sel, double* ops, double* buf, hipStream_t st, int* d_status)
{
  const TreePlan& P = t->P;
  const int nl = (int) P.lev.size ();
  const Scratch z = scratch (P);
  const size_t fmax[2] = {z.f0, z.f1};
  double* F[2] = {buf, buf + fmax[0] * nm};
  double* RW = F[1] + fmax[1] * nm;
  for (int j = nl - 1; j >= 0; j--) {
    const TreeLevel& L = P.lev[j];
    const int nt = (L.nmax + TB - 1) / TB, ldw = nt * TB;
    const size_t n2 = (size_t) L.nmax * L.nmax;
    double* Fj = F[j & 1];
    const dim3 gb ((unsigned) std::min<size_t> ((n2 + 255) / 256, 1024), L.ncls, nm);
    hipLaunchKernelGGL (k_tree_assemble, gb, dim3 (256), 0, st, t->cls, L.cls0, t->child, t->map,
                        Sel, m->next, m->nclass, F[(j + 1) & 1],
                        j + 1 < nl ? P.lev[j + 1].fsize : (size_t) 0, Fj, L.fsize, d_nsolve,
                        m->nsolve);
    for (int step = 0; TB * step < L.kmax; step++) {
      hipLaunchKernelGGL (k_tree_panel, dim3 (nt, L.ncls, nm), dim3 (256), 0, st, t->cls, L.cls0,
                          Fj, L.fsize, RW, ldw, step, d_status);
      hipLaunchKernelGGL (k_tree_update, dim3 (nt * (nt + 1) / 2, L.ncls, nm), dim3 (256), 0, st, t->cls,
                          L.cls0, Fj, L.fsize, RW, ldw, step, nt);
    }
    hipLaunchKernelGGL (k_tree_operators, gb, dim3 (256), 0, st, t->cls, L.cls0, Fj, L.fsize,
                        ops, P.ops);
  }
  SX_HIP (hipGetLastError ());
  return SX_OK;
}

// The arguments of a level's launch that the plan gives
struct LevelLaunch { int dir, W, blocks; size_t lds; };
static LevelLaunch level_launch (const TreeDev* t, TreeArgs& T, int j, int down, int nm, int nr)
{
  const TreePlan& P = t->P;
  const TreeLevel& L = P.lev[j];
  const int q = nr / 2 - 1;
  T.gk = t->gk; T.gb = t->gb; T.tgt = t->tgt;
  T.os = P.ops;
  T.nsp = P.nsolve; T.slots = P.slots; T.nr = nr;
  T.nmodes = nm;
  T.xcd = nm >= 32 || (nm >= 8 && nm % 8 == 0);
  T.item = t->item + (down ? L.it_b[q] : L.it_f[q]);
  T.nitem = down ? L.nit_b[q] : L.nit_f[q];
  return {down ? (j ? T_DOWN : T_ROOT) : T_UP, P.W,
          T.nitem * (T.xcd ? (nm + 7) / 8 * 8 : nm), down ? L.lds_b[q] : L.lds_f[q]};
}

// f (DIR, W) with the launch's kernel instance
template <typename F> static int tree_instance (const LevelLaunch& l, F f)
{
  auto dir = [&] (auto w) {
    return l.dir == T_UP     ? f (std::integral_constant<int, T_UP> {}, w)
           : l.dir == T_DOWN ? f (std::integral_constant<int, T_DOWN> {}, w)
                             : f (std::integral_constant<int, T_ROOT> {}, w);
  };
  return l.W == 4 ? dir (std::integral_constant<int, 4> {}) : dir (std::integral_constant<int, 8> {});
}

// The launches of a solve: up to the root's children, down from the root
static int sweep (const TreeDev* t, TreeArgs T, int nm, int nr, hipStream_t st)
{
  const int nl = (int) t->P.lev.size ();
  auto level = [&] (int j, int down) {
    const LevelLaunch l = level_launch (t, T, j, down, nm, nr);
    if (!l.blocks) return (int) SX_OK;
    return tree_instance (l, [&] (auto d, auto w) {
      auto kern = k_tree_level<decltype (d)::value, decltype (w)::value>;
      if (int rc = lds_limit ((const void*) kern, l.lds)) return rc;
      hipLaunchKernelGGL (kern, dim3 (l.blocks), dim3 (256), l.lds, st, T);
      SX_HIP (hipGetLastError ());
      return (int) SX_OK;
    });
  };
  for (int j = nl - 1; j > 0; j--)
    if (int rc = level (j, 0)) return rc;
  for (int j = 0; j < nl; j++)
    if (int rc = level (j, 1)) return rc;
  return SX_OK;
}

static TreeArgs tree_args (const sx_msys* s)
{
  TreeArgs T {};
  T.ops = s->d_tops;
  T.in = s->d_tb; T.rhs = s->d_rhs; T.v = s->d_tv; T.cb = s->d_tc;
  T.nmax = s->nmax;
  T.nsolve = s->d_nsolve;
  return T;
}

// The same launches recorded into a batch's plan, the roots of all its
// systems in one phase (trees of up to TREE_PLAN_LEVELS levels end level)
constexpr int TREE_PLAN_LEVELS = 5;
static void plan_levels (BatchPlan& P, const TreeDev* t, const TreeArgs& args, int nm)
{
  const int nl = (int) t->P.lev.size (), root = P.phase + std::max (nl, TREE_PLAN_LEVELS) - 1;
  auto level = [&] (int j, int down) {
    TreeArgs T = args;
    const LevelLaunch l = level_launch (t, T, j, down, nm, 2);
    P.phase = down ? root + j : root - j;
    if (!l.blocks) return (int) SX_OK;
    return tree_instance (l, [&] (auto d, auto w) {
      batch_rec<256, FnTreeLevel<decltype (d)::value, decltype (w)::value>> (
          P, dim3 (l.blocks), 256, l.lds, T);
      return (int) SX_OK;
    });
  };
  for (int j = nl - 1; j > 0; j--) level (j, 0);
  for (int j = 0; j < nl; j++) level (j, 1);
  P.phase = root + std::max (nl, TREE_PLAN_LEVELS);
}

// Refinement of a singular mode's solution (pure Neumann, its last unknown
// dropped: condition ~1e5 against the constant vector, so two eliminations
// in working precision end ~2e-11 of the pressure apart).  One correction
// from a residual in twice the working precision, formed with the entries
// the band assembly rounds to, leaves the exact solution of the assembled
// system to rounding, after a dissection and after a band solve alike.  The
// correction runs on a dissection of that mode alone, cut for one mode
// (fewer levels).
struct TreeSing {
  int mode = 0;
  TreeDev* t = nullptr;
  double *ops = nullptr, *val = nullptr, *r = nullptr, *dx = nullptr, *v = nullptr, *cb = nullptr,
         *b = nullptr;                 // band solves: the right-hand sides kept
};

// row lists of the assembled matrix (both triangles), once per mesh
static int sing_rows (sx_mesh* m)
{
  std::lock_guard<std::mutex> lock (m->tree_mu);
  if (m->d_sptr) return SX_OK;
  std::vector<int> ptr (m->nsolve + 1, 0), col, pr;
  for (int p = 0; p < m->npairs; p++) {
    const int a = m->pmn[2 * p], b = m->pmn[2 * p + 1];
    ptr[a + 1]++;
    if (a != b) ptr[b + 1]++;
  }
  for (int i = 0; i < m->nsolve; i++) ptr[i + 1] += ptr[i];
  col.resize (ptr[m->nsolve]);
  pr.resize (ptr[m->nsolve]);
  std::vector<int> at (ptr.begin (), ptr.end () - 1);
  for (int p = 0; p < m->npairs; p++) {
    const int a = m->pmn[2 * p], b = m->pmn[2 * p + 1];
    col[at[a]] = b;
    pr[at[a]++] = p;
    if (a != b) { col[at[b]] = a; pr[at[b]++] = p; }
  }
  int rc;
  if ((rc = upload (&m->d_scol, col)) || (rc = upload (&m->d_spair, pr)) ||
      (rc = upload (&m->d_sptr, ptr)))
    return rc;
  return SX_OK;
}

void tree_sing_free (TreeSing* g)
{
  if (!g) return;
  for (double* p : {g->ops, g->val, g->r, g->dx, g->v, g->cb, g->b}) if (p) (void) hipFree (p);
  delete g;
}

// The workspace of solves with nr right-hand sides per mode by plan t (null:
// none) and of the singular mode's refinement, added to what G replaces
int tree_grow (Grow& G, sx_msys* s, TreeDev* t, int nr)
{
  const size_t n = (size_t) s->nmodes * nr;
  int rc;
  if (t && ((rc = G.add (&s->d_tb, n * t->P.nsolve)) || (rc = G.add (&s->d_tv, n * t->P.nsolve)) ||
            (rc = G.add (&s->d_tc, n * t->P.slots))))
    return rc;
  if (TreeSing* g = s->sing) {
    const TreePlan& P = g->t->P;
    if ((rc = G.add (&g->b, (size_t) nr * s->nmax)) || (rc = G.add (&g->dx, (size_t) nr * s->nmax)) ||
        (rc = G.add (&g->v, (size_t) nr * P.nsolve)) || (rc = G.add (&g->cb, nr * P.slots)) ||
        (rc = G.add (&g->r, (size_t) nr * P.nsolve)))
      return rc;
  }
  return SX_OK;
}

const int* tree_perm (const sx_msys* s) { return s->tree->perm; }

int tree_factor (sx_msys* s, const double* Sel, double* buf, hipStream_t st, int* d_status)
{
  return factor (s->tree, s->m, s->nmodes, s->d_nsolve, Sel, s->d_tops, buf, st, d_status);
}

int tree_for_batch (sx_msys* s, const double* Sel, hipStream_t st, int* d_status, Held& h)
{
  // (64 uneven problems of one mode: 309 us at 4, 318 at 8, 359 at 32, 360
  // with the systems' own cuts.  Systems of 4 and more modes keep their own:
  // batches of those were not measured)
  constexpr int BATCH_SHARE = 4;
  TreeDev* t = nullptr;
  if (int rc = tree_prepare (s->m, s->nmodes, &t, true, std::max (1, BATCH_SHARE / s->nmodes)))
    return rc;
  if (!t || t == s->tree) return SX_OK;
  const size_t n = (size_t) s->nmodes * s->rhs_cap;
  Held now;
  Grow G;
  DevTmp buf;
  int rc;
  if ((rc = G.add (&now.ops, std::max<size_t> (t->P.ops * s->nmodes, 2))) ||
      (rc = G.add (&now.tb, n * t->P.nsolve)) || (rc = G.add (&now.tv, n * t->P.nsolve)) ||
      (rc = G.add (&now.tc, n * t->P.slots)))
    return rc;
  SX_HIP (dev_malloc (&buf.p, sizeof (double) * tree_scratch (t, s->nmodes)));
  // (the arrays are now's once installed)
  if ((rc = factor (t, s->m, s->nmodes, s->d_nsolve, Sel, G.items[0].p, (double*) buf.p, st,
                    d_status)))
    return rc;
  SX_HIP (hipStreamSynchronize (st));
  if ((rc = G.install (s))) return rc;
  now.tree = t;
  h = now;
  return SX_OK;
}

int tree_sing_setup (sx_msys* s, const double* Sel, hipStream_t st, int* d_status)
{
  sx_mesh* m = s->m;
  for (int md = 0; md < s->nmodes; md++) {
    if (s->nsolve[md] == m->nsolve || s->nsolve[md] < 1) continue;
    TreeDev* t = nullptr;
    if (int rc = tree_prepare (m, 1, &t, true)) return rc;
    if (!t) return SX_OK;
    TreeSing* g = s->sing = new TreeSing;
    g->mode = md;
    g->t = t;
    const double* S = Sel + (size_t) md * m->nclass * m->next * m->next;
    // (the scratch is the later workspace's allocation g->val: entries past
    // the matrix's are free once the factor is done)
    const size_t nb = std::max<size_t> (tree_scratch (t, 1), m->npairs);
    SX_HIP (dev_malloc (&g->ops, sizeof (double) * std::max<size_t> (t->P.ops, 2)));
    SX_HIP (dev_malloc (&g->val, sizeof (double) * nb));
    if (int rc = factor (t, m, 1, s->d_nsolve + md, S, g->ops, g->val, st, d_status + md)) return rc;
    if (int rc = sing_rows (m)) return rc;
    hipLaunchKernelGGL (k_tree_entries, dim3 ((m->npairs + 255) / 256), dim3 (256), 0, st,
                        m->npairs, m->d_pptr, m->d_psrc, S, g->val);
    SX_HIP (hipGetLastError ());
    Grow G;
    int rc = tree_grow (G, s, nullptr, 2);
    return rc ? rc : G.install (s);    // at most mode 0 has a zero constant
  }
  return SX_OK;
}

// A refinement's right-hand sides as they were before the solve, by node
// (band solves) or by position of the solve's dissection
struct Kept { const double* b; int ld; const int* perm; };
static Kept kept (const sx_msys* s, int nr, bool tree)
{
  const TreeSing* g = s->sing;
  if (!tree) return {g->b, s->nmax, nullptr};
  const int nsp = s->tree->P.nsolve;
  return {s->d_tb + (size_t) g->mode * nr * nsp, nsp, s->tree->perm};
}
static double* sing_x (const sx_msys* s, int nr)
{
  return s->d_rhs + (size_t) s->sing->mode * nr * s->nmax;
}
static TreeArgs sing_args (const sx_msys* s, int nr)
{
  const TreeSing* g = s->sing;
  TreeArgs T {};
  T.ops = g->ops;
  T.in = g->r; T.rhs = g->dx; T.v = g->v; T.cb = g->cb;
  T.sum = sing_x (s, nr);
  T.nmax = s->nmax;
  T.nsolve = s->d_nsolve + g->mode;
  return T;
}

static int refine (const sx_msys* s, int nr, bool tree, hipStream_t st)
{
  const TreeSing* g = s->sing;
  const sx_mesh* m = s->m;
  const int ns = s->nsolve[g->mode];
  const Kept k = kept (s, nr, tree);
  hipLaunchKernelGGL (k_tree_residual, dim3 ((ns + 3) / 4), dim3 (256), 0, st, ns, s->nmax, nr,
                      m->d_sptr, m->d_scol, m->d_spair, g->val, k.b, k.ld, k.perm, sing_x (s, nr),
                      g->r, g->t->P.nsolve, g->t->perm);
  SX_HIP (hipGetLastError ());
  return sweep (g->t, sing_args (s, nr), 1, nr, st);
}

int sing_keep (const sx_msys* s, int nr, hipStream_t st)
{
  SX_HIP (hipMemcpyAsync (s->sing->b, sing_x (s, nr), sizeof (double) * nr * s->nmax,
                          hipMemcpyDeviceToDevice, st));
  return SX_OK;
}

int sing_refine (const sx_msys* s, int nr, hipStream_t st) { return refine (s, nr, false, st); }

// The same recorded (two right-hand sides per mode)
static void plan_refine (BatchPlan& P, const sx_msys* s, bool tree)
{
  const TreeSing* g = s->sing;
  const sx_mesh* m = s->m;
  const int ns = s->nsolve[g->mode], nr = 2;
  const Kept k = kept (s, nr, tree);
  batch_rec<256, FnTreeResidual> (P, dim3 ((ns + 3) / 4), 256, 0, ns, s->nmax, nr,
                                  (const int*) m->d_sptr, (const int*) m->d_scol,
                                  (const int*) m->d_spair, (const double*) g->val, k.b, k.ld,
                                  k.perm, (const double*) sing_x (s, nr), g->r,
                                  g->t->P.nsolve, (const int*) g->t->perm);
  P.phase++;
  plan_levels (P, g->t, sing_args (s, nr), 1);
}

int plan_sing_keep (BatchPlan& P, const sx_msys* s)
{
  const int n = 2 * s->nmax;
  batch_rec<256, FnTreeKeep> (P, dim3 ((n + 255) / 256), 256, 0, s->sing->b,
                              (const double*) sing_x (s, 2), n);
  P.phase++;
  return SX_OK;
}

int plan_sing_refine (BatchPlan& P, const sx_msys* s)
{
  plan_refine (P, s, false);
  return SX_OK;
}

// A system's solve recorded into a batch's plan
int plan_tree_solve (BatchPlan& P, const sx_msys* s)
{
  plan_levels (P, s->tree, tree_args (s), s->nmodes);
  if (s->sing) plan_refine (P, s, true);
  return SX_OK;
}

// Solve of the nr (2, 4, 6) right-hand sides per mode from d_tb to d_rhs.
int tree_solve (const sx_msys* s, int nr, hipStream_t st)
{
  if (nr < 2 || nr > 6 || (nr & 1) || nr > s->rhs_cap) {
    set_error ("tree solve: 2, 4 or 6 reserved right-hand sides per mode");
    return SX_ERR_ARG;
  }
  s->last_kernel = 4;
  s->last_nr = nr;
  const TreeDev* t = s->tree;
  if (int rc = sweep (t, tree_args (s), s->nmodes, nr, st)) return rc;
  return s->sing ? refine (s, nr, true, st) : (int) SX_OK;
}

}  // namespace sx
