// Waveguide mode solver on the device: the subspace iteration of pjz's
// mode() (src/pjz/_mode.py:99-142) over the operator of a 2-D cross-section
// (_operator, src/pjz/_mode.py:22-50), run to convergence inside one launch,
// so the host never synchronises inside the loop (a torch version of the same
// loop is bound by ~30 launches and one host read per iteration).
//
// Per iteration, four passes over the vectors:
//   1. x = y R1^-1, summing the Gram matrix of x as the rows are written;
//   2. x = x R2^-1 (1 and 2 are CholeskyQR2: Gram matrices in double,
//      Cholesky and the triangular inverse on one lane);
//   3. y = A x, first stencil pass: the scalar fields b = (-(d-y u0) +
//      d-x u1) / eps_z and c = d+x u0 + d+y u1;
//   4. second stencil pass, the vector update, summing w_k = <x_k, y_k>,
//      |y_k|^2, |x_k|^2 (so err_k = |y_k - w_k x_k|) and the Gram matrix of
//      y, which gives the next iteration's R1.
// Vectors are (2, XX, YY, MM) with the MM modes innermost, as pjz lays them
// out; the periodic differences wrap in x and y (jnp.roll in pjz).  Every
// pass is a stride loop over rows or cells, so any cross-section size works;
// fields live in global memory and the sums go through LDS.
//
// Three kernels run that iteration:
//  - k_mode_tile: the state in registers and LDS, up to 6 modes and rows that
//    fit a workgroup (see there): the usual case.  It stops as the two below
//    do, by the section's size.
//  - k_mode_subspace: one workgroup per frequency; the frequency stops once
//    its residuals are all <= tol.  Small sections (a few thousand cells).
//  - k_mode_grid: `gpf` workgroups per frequency in one cooperative launch,
//    the passes split across them and separated by grid barriers, partial
//    sums exchanged through a workspace; every workgroup reduces the partials
//    itself in a fixed order, so all hold the same R^-1 and the same stop
//    decision.  All frequencies iterate together until the largest residual
//    of all is <= tol, which is pjz's own test (it takes the max over
//    frequencies and modes).  Large sections, where one CU per frequency
//    bounds the first kernel.
#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <type_traits>

#include "fdtd_common.h"
#include "waits.h"

namespace pjz {

namespace cg = cooperative_groups;

constexpr int kModeThreads = 512;
constexpr int kModeWaves = kModeThreads / 64;
// Cells x modes from which on all frequencies iterate until the last has
// converged; below, each stops by itself.
constexpr long long kModeJointWork = 16384;
constexpr int kModeMaxShare = 32;  // grid kernel: most workgroups per frequency

struct ModeArgs {
  int XX, YY, max_iters;
  float tol;
  const float* eps;    // (3, XX, YY): eps_x, eps_y, eps_z (propagation along z)
  const float* omega;  // (ww)
  const float* shift;  // (ww)
  float* x;            // (ww, 2, XX, YY, MM): start vectors in, final basis out
  float* y;            // workspace, like x: A x
  float* bc;           // workspace, like x: the b and c scalar fields
  float* w;            // (ww, MM)
  float* err;          // (ww, MM)
  int* iters;          // (ww)
  double* partial;     // grid kernel: (ww, gpf, NQ + NPAIR) partial sums
  int gpf;             // grid kernel: workgroups per frequency
};

template <int MM>
struct ModeLds {
  static constexpr int NPAIR = MM * (MM + 1) / 2;  // Gram entries (upper triangle)
  static constexpr int NQ = 3 * MM;                // <x,y>, <y,y>, <x,x> per mode
  static constexpr int NALL = NQ + NPAIR;
  double red[kModeWaves][NALL];
  double sum[NALL];    // [NQ Rayleigh sums | NPAIR Gram entries]
  double R[MM * MM];   // Cholesky factor, upper (G = R^T R)
  double Ri[MM * MM];  // its inverse, upper
  int go;
};

// Sums acc[0..P) over the workgroup into out[0..P) (LDS): wavefront
// reductions, one LDS row per wave, one barrier, the cross-wave sums, one
// barrier.  Fixed order, so results do not depend on timing.
template <int MM, int P>
__device__ __forceinline__ void block_sum(const double (&acc)[P], ModeLds<MM>& L, double* out) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    double v = acc[p];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) L.red[wv][p] = v;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < P; q += kModeThreads) {
    double t = 0.0;
    for (int w = 0; w < kModeWaves; ++w) t += L.red[w][q];
    out[q] = t;
  }
  __syncthreads();
}

// Index of Gram entry (a, b), a <= b, in the row-by-row upper triangle.
template <int MM>
__device__ constexpr int tri(int a, int b) { return a * MM - a * (a - 1) / 2 + (b - a); }

// acc[off + tri(a, b)] += v[a] v[b] for a <= b (the loops unroll completely,
// so every register index is a constant).
template <int MM, int P>
__device__ __forceinline__ void add_gram(double (&acc)[P], int off, const float (&v)[MM]) {
#pragma unroll
  for (int a = 0; a < MM; ++a) {
#pragma unroll
    for (int b = a; b < MM; ++b) acc[off + tri<MM>(a, b)] += (double)v[a] * (double)v[b];
  }
}

// On one lane: R with G = R^T R for the Gram matrix in g (upper triangle),
// and Ri = R^-1, into LDS.  The caller synchronises.
template <int MM>
__device__ __forceinline__ void chol_inv(const double* g, ModeLds<MM>& L) {
  double* R = L.R;
  double* Ri = L.Ri;
  for (int i = 0; i < MM * MM; ++i) R[i] = Ri[i] = 0.0;
  for (int j = 0; j < MM; ++j) {
    double d = g[tri<MM>(j, j)];
    for (int k = 0; k < j; ++k) d -= R[k * MM + j] * R[k * MM + j];
    // A start vector inside the span of the others (degenerate input only)
    // keeps a tiny pivot instead of a NaN.
    R[j * MM + j] = sqrt(d > 1e-300 ? d : 1e-300);
    for (int i = j + 1; i < MM; ++i) {
      double t = g[tri<MM>(j, i)];
      for (int k = 0; k < j; ++k) t -= R[k * MM + j] * R[k * MM + i];
      R[j * MM + i] = t / R[j * MM + j];
    }
  }
  for (int j = 0; j < MM; ++j) {
    Ri[j * MM + j] = 1.0 / R[j * MM + j];
    for (int i = j - 1; i >= 0; --i) {
      double t = 0.0;
      for (int k = i + 1; k <= j; ++k) t += R[i * MM + k] * Ri[k * MM + j];
      Ri[i * MM + j] = -t / R[i * MM + i];
    }
  }
}

// One row times Ri (upper triangular).
template <int MM>
__device__ __forceinline__ void row_ri(float (&v)[MM], const ModeLds<MM>& L) {
  float o[MM];
#pragma unroll
  for (int k = 0; k < MM; ++k) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j <= k; ++j) t += (double)v[j] * L.Ri[j * MM + k];
    o[k] = (float)t;
  }
#pragma unroll
  for (int k = 0; k < MM; ++k) v[k] = o[k];
}

// A thread's share of a pass: items t0, t0 + stride, ... (one workgroup:
// threadIdx.x and the block size; the grid kernel: the frequency's threads).
struct Share {
  int t0, stride;
};

// acc[off..] += Gram matrix of the rows of v in this share.
template <int MM, int P>
__device__ __forceinline__ void gram_rows(const float* __restrict__ v, int n, Share sh,
                                          double (&acc)[P], int off) {
  for (int r = sh.t0; r < n; r += sh.stride) {
    float row[MM];
#pragma unroll
    for (int k = 0; k < MM; ++k) row[k] = v[r * MM + k];
    add_gram<MM>(acc, off, row);
  }
}

// dst = src Ri for the rows of this share (dst may alias src); with GRAM the
// Gram matrix of the new rows goes into acc.
template <int MM, bool GRAM, int P>
__device__ __forceinline__ void ri_rows(const float* src, float* dst, int n, Share sh,
                                        const ModeLds<MM>& L, double (&acc)[P]) {
  for (int r = sh.t0; r < n; r += sh.stride) {
    float v[MM];
#pragma unroll
    for (int k = 0; k < MM; ++k) v[k] = src[r * MM + k];
    row_ri<MM>(v, L);
#pragma unroll
    for (int k = 0; k < MM; ++k) dst[r * MM + k] = v[k];
    if constexpr (GRAM) add_gram<MM>(acc, 0, v);
  }
}

// First stencil pass of y = A x (_operator, src/pjz/_mode.py:22-50): the
// scalar fields b = (-(d-y u0) + d-x u1) / eps_z (backward differences) and
// c = d+x u0 + d+y u1 (forward differences), periodic in x and y.
template <int MM>
__device__ __forceinline__ void op_pass1(const float* __restrict__ x, float* __restrict__ bc,
                                         const float* __restrict__ eps, int XX, int YY,
                                         Share sh) {
  const int P = XX * YY, cells = P * MM;
  const float* ez = eps + 2 * P;
  for (int e = sh.t0; e < cells; e += sh.stride) {
    const int p = e / MM, k = e - p * MM;
    const int i = p / YY, j = p - i * YY;
    const int im = i == 0 ? XX - 1 : i - 1, ip = i == XX - 1 ? 0 : i + 1;
    const int jm = j == 0 ? YY - 1 : j - 1, jp = j == YY - 1 ? 0 : j + 1;
    const float* x0 = x;
    const float* x1 = x + cells;
    const float u0 = x0[e], u1 = x1[e];
    bc[e] = (-(u0 - x0[(i * YY + jm) * MM + k]) + (u1 - x1[(im * YY + j) * MM + k])) / ez[p];
    bc[cells + e] = (x0[(ip * YY + j) * MM + k] - u0) + (x1[(i * YY + jp) * MM + k] - u1);
  }
}

// Whether the second stencil pass also sums the Gram matrix of y: its
// 3 MM + MM (MM + 1) / 2 double accumulators fit in registers up to 6 modes;
// above, a separate pass sums the Gram matrix.
template <int MM>
constexpr bool kFuseGram = MM <= 6;

// Second stencil pass, one cell (both components, all modes) per item, with
// the same grouping of the float operations as _operator: y = A x, and into
// acc the Rayleigh sums (x.y, y.y, x.x per mode) and, when P has room for it,
// the Gram matrix of y.
template <int MM, int P>
__device__ __forceinline__ void op_pass2(const float* __restrict__ x, float* __restrict__ y,
                                         const float* __restrict__ bc,
                                         const float* __restrict__ eps, int XX, int YY,
                                         float om2, float s, Share sh, double (&acc)[P]) {
  const int PC = XX * YY, cells = PC * MM;
  const float* ex = eps;
  const float* ey = eps + PC;
  const float* bb = bc;
  const float* cc = bc + cells;
  for (int p = sh.t0; p < PC; p += sh.stride) {
    const int i = p / YY, j = p - i * YY;
    const int im = i == 0 ? XX - 1 : i - 1, ip = i == XX - 1 ? 0 : i + 1;
    const int jm = j == 0 ? YY - 1 : j - 1, jp = j == YY - 1 ? 0 : j + 1;
    const float exv = ex[p], eyv = ey[p];
    float x0[MM], x1[MM], y0[MM], y1[MM];
#pragma unroll
    for (int k = 0; k < MM; ++k) {
      const int e = p * MM + k;
      const float b = bb[e], c = cc[e];
      x0[k] = x[e];
      x1[k] = x[cells + e];
      const float a0 = (om2 * eyv - s) * x0[k], a1 = (om2 * exv - s) * x1[k];
      const float b0 = -(bb[(i * YY + jp) * MM + k] - b) * eyv;
      const float b1 = (bb[(ip * YY + j) * MM + k] - b) * exv;
      y0[k] = (a0 + b0) + (c - cc[(im * YY + j) * MM + k]);
      y1[k] = (a1 + b1) + (c - cc[(i * YY + jm) * MM + k]);
      y[e] = y0[k];
      y[cells + e] = y1[k];
      acc[k] += (double)x0[k] * y0[k] + (double)x1[k] * y1[k];
      acc[MM + k] += (double)y0[k] * y0[k] + (double)y1[k] * y1[k];
      acc[2 * MM + k] += (double)x0[k] * x0[k] + (double)x1[k] * x1[k];
    }
    if constexpr (P > 3 * MM) {
      add_gram<MM>(acc, 3 * MM, y0);
      add_gram<MM>(acc, 3 * MM, y1);
    }
  }
}

// Residuals of one frequency from its Rayleigh sums s[0..3 MM); writes w and
// err when `out`; returns max err (NaN if any residual is NaN).
template <int MM>
__device__ __forceinline__ double residuals(const double* s, float* w, float* err, bool out) {
  double emax = 0.0;
  bool nan = false;
  for (int k = 0; k < MM; ++k) {
    const double xy = s[k], yy = s[MM + k], xx = s[2 * MM + k];
    const double e2 = yy - 2.0 * xy * xy + xy * xy * xx;
    const bool bad = !(e2 == e2);
    const double e = sqrt(e2 > 0.0 ? e2 : 0.0);
    nan |= bad;
    emax = e > emax ? e : emax;
    if (out) {
      w[k] = (float)xy;
      err[k] = bad ? __builtin_nanf("") : (float)e;
    }
  }
  return nan ? __builtin_nan("") : emax;
}

// --------------------------------------------------------------- one workgroup

// The stencil's second pass with all its sums into L.sum (Rayleigh sums, then
// the Gram matrix of y), in one pass or two.
template <int MM>
__device__ __forceinline__ void op_pass2_sums(const float* __restrict__ x, float* __restrict__ y,
                                              const float* __restrict__ bc,
                                              const float* __restrict__ eps, int XX, int YY,
                                              float om2, float s, int n, ModeLds<MM>& L) {
  constexpr int NQ = ModeLds<MM>::NQ, NPAIR = ModeLds<MM>::NPAIR;
  const Share sh{(int)threadIdx.x, kModeThreads};
  if constexpr (kFuseGram<MM>) {
    double acc[NQ + NPAIR];
#pragma unroll
    for (int q = 0; q < NQ + NPAIR; ++q) acc[q] = 0.0;
    op_pass2<MM>(x, y, bc, eps, XX, YY, om2, s, sh, acc);
    block_sum<MM>(acc, L, L.sum);
  } else {
    {
      double acc[NQ];
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
      op_pass2<MM>(x, y, bc, eps, XX, YY, om2, s, sh, acc);
      block_sum<MM>(acc, L, L.sum);
    }
    double acc[NPAIR];
#pragma unroll
    for (int q = 0; q < NPAIR; ++q) acc[q] = 0.0;
    gram_rows<MM>(y, n, sh, acc, 0);
    block_sum<MM>(acc, L, L.sum + NQ);
  }
}

template <int MM>
__global__ __launch_bounds__(kModeThreads) void k_mode_subspace(ModeArgs a) {
  __shared__ ModeLds<MM> L;
  constexpr int NQ = ModeLds<MM>::NQ, NPAIR = ModeLds<MM>::NPAIR;
  const int f = blockIdx.x;
  const int n = 2 * a.XX * a.YY;  // rows of the (n, MM) matrices
  const long long off = (long long)f * n * MM;
  float* x = a.x + off;
  float* y = a.y + off;
  float* bc = a.bc + off;
  const float om = a.omega[f];
  const float om2 = om * om;
  const float s = a.shift[f];
  const Share sh{(int)threadIdx.x, kModeThreads};
  // y = A x0 and its Gram matrix; then R^-1 for the first QR.
  op_pass1<MM>(x, bc, a.eps, a.XX, a.YY, sh);
  __syncthreads();
  op_pass2_sums<MM>(x, y, bc, a.eps, a.XX, a.YY, om2, s, n, L);
  if (threadIdx.x == 0) chol_inv<MM>(L.sum + NQ, L);
  __syncthreads();
  int it = 0;
  bool go = true;  // max err > tol; err starts at +inf
  while (it < a.max_iters && go) {
    // CholeskyQR2 of y: x = y R1^-1 (with the Gram matrix of that x), then
    // x = x R2^-1.
    {
      double acc[NPAIR];
#pragma unroll
      for (int q = 0; q < NPAIR; ++q) acc[q] = 0.0;
      ri_rows<MM, (MM <= 7)>(y, x, n, sh, L, acc);
      if constexpr (MM > 7) {
        // Above 7 modes the Gram sum takes a pass of its own (registers);
        // each thread reads back only the rows it wrote.
        gram_rows<MM>(x, n, sh, acc, 0);
      }
      block_sum<MM>(acc, L, L.sum + NQ);
      if (threadIdx.x == 0) chol_inv<MM>(L.sum + NQ, L);
      __syncthreads();
      double none[1];
      ri_rows<MM, false>(x, x, n, sh, L, none);
      __syncthreads();
    }
    // y = A x with the Rayleigh sums and the Gram matrix of the new y.
    op_pass1<MM>(x, bc, a.eps, a.XX, a.YY, sh);
    __syncthreads();
    op_pass2_sums<MM>(x, y, bc, a.eps, a.XX, a.YY, om2, s, n, L);
    if (threadIdx.x == 0) {
      const double emax = residuals<MM>(L.sum, a.w + f * MM, a.err + f * MM, true);
      // pjz continues while max(err) > tol, which a NaN ends.
      L.go = emax > (double)a.tol;
      // R^-1 of the new y for the next iteration's first QR step.
      chol_inv<MM>(L.sum + NQ, L);
    }
    __syncthreads();
    go = L.go;
    ++it;
  }
  if (threadIdx.x == 0) {
    a.iters[f] = it;
    if (it == 0) {
      for (int k = 0; k < MM; ++k) {
        a.w[f * MM + k] = 0.0f;
        a.err[f * MM + k] = __builtin_inff();
      }
    }
  }
}

// ------------------------------------------------------------------ the grid

// Writes P of this workgroup's sums (L.sum[off..off+P)) into its partial row.
__device__ __forceinline__ void put_partial(double* partial, long long row, int stride,
                                            const double* sums, int off, int P) {
  for (int q = threadIdx.x; q < P; q += kModeThreads)
    partial[row * stride + off + q] = sums[off + q];
}

// out[off + q] = sum over the frequency's gpf partial rows of entry off + q,
// in workgroup order, so every workgroup gets the same bits.
__device__ __forceinline__ void reduce_partials(const double* partial, int f, int gpf,
                                                int stride, int off, int P, double* out) {
  for (int q = threadIdx.x; q < P; q += kModeThreads) {
    double t = 0.0;
    for (int j = 0; j < gpf; ++j) t += partial[((long long)f * gpf + j) * stride + off + q];
    out[off + q] = t;
  }
}

// The grid kernel's second stencil pass with its sums: partial rows of all
// NQ + NPAIR sums, grid barrier, then every workgroup reduces its frequency's
// into L.sum.  On entry the previous partials are no longer read.
template <int MM>
__device__ __forceinline__ void grid_pass2(cg::grid_group& grid, const ModeArgs& a,
                                           const float* x, float* y, const float* bc, float om2,
                                           float s, int n, int f, long long prow, Share sh,
                                           ModeLds<MM>& L) {
  constexpr int NQ = ModeLds<MM>::NQ, NPAIR = ModeLds<MM>::NPAIR, NALL = ModeLds<MM>::NALL;
  if constexpr (kFuseGram<MM>) {
    double acc[NALL];
#pragma unroll
    for (int q = 0; q < NALL; ++q) acc[q] = 0.0;
    op_pass2<MM>(x, y, bc, a.eps, a.XX, a.YY, om2, s, sh, acc);
    block_sum<MM>(acc, L, L.sum);
    put_partial(a.partial, prow, NALL, L.sum, 0, NALL);
  } else {
    double acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
    op_pass2<MM>(x, y, bc, a.eps, a.XX, a.YY, om2, s, sh, acc);
    block_sum<MM>(acc, L, L.sum);
    put_partial(a.partial, prow, NALL, L.sum, 0, NQ);
    // Rows (Gram sum) and cells (stencil) are shared out differently, so
    // all of y must be written before its Gram sum.
    grid.sync();
    double accg[NPAIR];
#pragma unroll
    for (int q = 0; q < NPAIR; ++q) accg[q] = 0.0;
    gram_rows<MM>(y, n, sh, accg, 0);
    block_sum<MM>(accg, L, L.sum + NQ);
    put_partial(a.partial, prow, NALL, L.sum, NQ, NPAIR);
  }
  grid.sync();
  reduce_partials(a.partial, f, a.gpf, NALL, 0, NALL, L.sum);
  __syncthreads();
}

template <int MM>
__global__ __launch_bounds__(kModeThreads) void k_mode_grid(ModeArgs a) {
  __shared__ ModeLds<MM> L;
  constexpr int NQ = ModeLds<MM>::NQ, NPAIR = ModeLds<MM>::NPAIR, NALL = ModeLds<MM>::NALL;
  cg::grid_group grid = cg::this_grid();
  const int gpf = a.gpf;
  const int ww = gridDim.x / gpf;
  const int f = blockIdx.x / gpf, part = blockIdx.x - f * gpf;
  const long long prow = (long long)f * gpf + part;  // this workgroup's partial row
  const int n = 2 * a.XX * a.YY;
  const long long off = (long long)f * n * MM;
  float* x = a.x + off;
  float* y = a.y + off;
  float* bc = a.bc + off;
  const float om = a.omega[f];
  const float om2 = om * om;
  const float s = a.shift[f];
  const Share sh{part * kModeThreads + (int)threadIdx.x, gpf * kModeThreads};

  op_pass1<MM>(x, bc, a.eps, a.XX, a.YY, sh);
  grid.sync();
  grid_pass2<MM>(grid, a, x, y, bc, om2, s, n, f, prow, sh, L);
  if (threadIdx.x == 0) chol_inv<MM>(L.sum + NQ, L);
  __syncthreads();
  int it = 0;
  bool go = true;  // max err > tol over all frequencies; err starts at +inf
  while (it < a.max_iters && go) {
    // x = y R1^-1 with the partial Gram sums of x.  The barrier before the
    // partials are written makes sure every workgroup has finished reading
    // the previous ones (its reduce and the stop test).
    {
      double acc[NPAIR];
#pragma unroll
      for (int q = 0; q < NPAIR; ++q) acc[q] = 0.0;
      ri_rows<MM, (MM <= 7)>(y, x, n, sh, L, acc);
      if constexpr (MM > 7) gram_rows<MM>(x, n, sh, acc, 0);  // own rows only
      block_sum<MM>(acc, L, L.sum + NQ);
      grid.sync();
      put_partial(a.partial, prow, NALL, L.sum, NQ, NPAIR);
      grid.sync();
      reduce_partials(a.partial, f, gpf, NALL, NQ, NPAIR, L.sum);
      __syncthreads();
      if (threadIdx.x == 0) chol_inv<MM>(L.sum + NQ, L);
      __syncthreads();
      double none[1];
      ri_rows<MM, false>(x, x, n, sh, L, none);
    }
    grid.sync();  // x complete before the stencil reads neighbours
    op_pass1<MM>(x, bc, a.eps, a.XX, a.YY, sh);
    grid.sync();
    grid_pass2<MM>(grid, a, x, y, bc, om2, s, n, f, prow, sh, L);
    if (threadIdx.x == 0) {
      // The stop test over all frequencies (their Rayleigh sums from the
      // partials, reduced in the same order everywhere); the own frequency's
      // w and err written by its first workgroup.
      double emax = 0.0;
      bool nan = false;
      for (int g = 0; g < ww; ++g) {
        double sums[NQ];
        for (int q = 0; q < NQ; ++q) {
          double t = 0.0;
          for (int j = 0; j < gpf; ++j) t += a.partial[((long long)g * gpf + j) * NALL + q];
          sums[q] = t;
        }
        const double e = residuals<MM>(sums, a.w + g * MM, a.err + g * MM, g == f && part == 0);
        nan |= !(e == e);
        emax = e > emax ? e : emax;
      }
      L.go = !nan && emax > (double)a.tol;
      chol_inv<MM>(L.sum + NQ, L);
    }
    __syncthreads();
    go = L.go;
    ++it;
  }
  if (threadIdx.x == 0 && part == 0) {
    a.iters[f] = it;
    if (it == 0) {
      for (int k = 0; k < MM; ++k) {
        a.w[f * MM + k] = 0.0f;
        a.err[f * MM + k] = __builtin_inff();
      }
    }
  }
}

// ------------------------------------------------------------- resident tiles
//
// Both kernels above are bound by latency: a 256 x 128 section with 2 modes
// spent 40 us an iteration on 0.5 MB of vectors (five grid barriers, each with
// a cache write-back, and four dependent passes that each wait for L2), the
// 30 x 20 strip with 2 modes 7.5 us (three block sums, two Cholesky
// factorisations on one lane, every pass through L2).  They are now 3.5 us (of
// the launch; the exchange and its waits take about half) and 2.0 us, bound by
// the instructions of eight waves on one compute unit.  Here the state never
// leaves the compute units: a workgroup owns R rows of the section for the
// whole run, x, y and the permittivity live in registers (CPT cells a thread),
// neighbours read x, b and c from LDS, and one exchange an iteration carries
// the sums and the two boundary rows between a frequency's workgroups.
//
// Exchange: every 8-byte word carries 4 bytes of payload and the exchange's
// number, written and read with relaxed device-scope atomics.  A word says by
// itself whether it has arrived, so there is no flag, fence or grid barrier:
// one store and one load latency (0.7-1.2 us measured for 4-32 workgroups,
// against 2-5 us for each grid barrier).  The sums are posted before the rows
// are waited for, so both travel at once (with the other order an iteration at
// 256 x 128 took 1.7 x as long).  Two sets of words alternate: a
// workgroup posts exchange s + 2 only after it has everyone's sums of s + 1,
// which each posts after it has read all of s.  All workgroups are resident at
// the same time (cooperative launch) and post before they wait, so every wait
// ends; where that does not hold, by the clock (waits.h), with NaN for results.
//
// Cholesky QR: the Gram matrix is summed in double over float rows, so one
// pass leaves x orthonormal to the rounding of its floats unless y is close to
// rank deficient.  The second pass runs only when a pivot falls below
// kModeQr2 of its column's norm (the error of one pass is about 1e-16 over
// that ratio); every workgroup sees the same sums and takes the same branch.
constexpr double kModeQr2 = 1e-6;
constexpr int kTileMaxModes = 6;   // registers: 3 MM + MM (MM + 1) / 2 double sums
// Cells a thread (more modes take more registers a cell).
constexpr int tile_max_cells(int mm) { return mm <= 3 ? 4 : 2; }
constexpr int kTileMaxWgs = 256;   // workgroups a frequency
constexpr int kTileMaxGrid = 512;  // workgroups of all frequencies that exchange
constexpr int kTileLds = 60 << 10; // dynamic LDS a workgroup may take

typedef unsigned long long word_t;

__device__ __forceinline__ void post_word(word_t* p, unsigned tag, unsigned v) {
  __hip_atomic_store(p, ((word_t)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word_t read_word(const word_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Polls until load() finds the lane's words, or the workgroup's waits end at
// `*end`; whether they were found.  (Lanes leave one by one: all together, by a
// ballot as in the resident steppers, 120 x 30 took 17% longer.)
template <class F>
__device__ __forceinline__ bool poll_words(unsigned* end, F&& load) {
  int left = kWaitPolls;
  bool found;
  do found = load(); while (!found && --left > 0);
  while (!found) {
    if (wait_over(end)) break;
    found = load();
  }
  return found;
}

struct TileArgs {
  ModeArgs m;
  word_t* box;   // words of the exchanges, cleared before the launch
  int R, joint;  // rows a workgroup; whether all frequencies stop together
  WaitArgs waits;
};

// Words of one exchange set: per frequency and workgroup its first and last
// row of y (2 x 2 components x YY x MM), then per frequency and sum every
// workgroup's double in two words, then one stop word a frequency; last the
// word of waits in vain (of the first set).
struct TileBox {
  size_t row, sum, go, late, total;
};
__host__ __device__ inline TileBox tile_box(int ww, int gpf, int YY, int mm) {
  const size_t nall = 3 * mm + mm * (mm + 1) / 2;
  const size_t n = gpf > 1 ? (size_t)ww * gpf : 0;  // one workgroup exchanges nothing
  TileBox b;
  b.row = 0;
  b.sum = n * 4 * YY * mm;
  b.go = b.sum + n * nall * 2;
  b.late = b.go + ww;
  b.total = b.late + 1;
  return b;
}

inline size_t tile_lds(int R, int YY, int mm) {
  return sizeof(float) * ((size_t)(4 * R + 6) * YY * mm + YY);
}

// A lane's double under the lane map of a DPP control.
template <int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// One stage of the wave reduction: lanes with bit OFF clear keep the first
// half of the M values summed with their partner's, the others the second
// half.  Lanes 32 and 16 apart swap by permlane, nearer ones by DPP (rotate by
// 8; mirror of 8 for OFF = 4; quad permutations), none through LDS.
template <int OFF, int M, int P>
__device__ __forceinline__ void fold(double (&v)[P], bool upper) {
  constexpr int H = (M + 1) / 2;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const double a = v[i], b = M == 1 ? v[i] : (i + H < M ? v[i + H] : 0.0);
    if constexpr (OFF >= 16) {
      const unsigned long long ab = __builtin_bit_cast(unsigned long long, a);
      const unsigned long long bb = __builtin_bit_cast(unsigned long long, b);
      unsigned r[4];
      if constexpr (OFF == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap((unsigned)ab, (unsigned)bb, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(ab >> 32), (unsigned)(bb >> 32),
                                                        false, false);
        r[0] = l[0]; r[1] = h[0]; r[2] = l[1]; r[3] = h[1];
      } else {
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)ab, (unsigned)bb, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(ab >> 32), (unsigned)(bb >> 32),
                                                        false, false);
        r[0] = l[0]; r[1] = h[0]; r[2] = l[1]; r[3] = h[1];
      }
      v[i] = __builtin_bit_cast(double, ((unsigned long long)r[1] << 32) | r[0]) +
             __builtin_bit_cast(double, ((unsigned long long)r[3] << 32) | r[2]);
    } else {
      constexpr int ctrl = OFF == 8 ? 0x128 : OFF == 4 ? 0x141 : OFF == 2 ? 0x4E : 0xB1;
      if constexpr (M == 1) {
        v[i] = a + dpp_double<ctrl>(a);
      } else {
        const double keep = upper ? b : a, send = upper ? a : b;
        v[i] = keep + dpp_double<ctrl>(send);
      }
    }
  }
}

// Sums P values over the wave, in a fixed order, into out[0..P): the values
// are halved at each of the first stages, so P values take about P + 2
// exchanges instead of 6 P.
template <int P>
__device__ __forceinline__ void wave_sums(double (&v)[P], double* out) {
  const int lane = threadIdx.x & 63;
  constexpr int M1 = (P + 1) / 2, M2 = (M1 + 1) / 2, M3 = (M2 + 1) / 2, M4 = (M3 + 1) / 2,
                M5 = (M4 + 1) / 2, M6 = (M5 + 1) / 2;
  static_assert(M6 == 1, "at most 64 sums");
  fold<32, P>(v, lane & 32);
  fold<16, M1>(v, lane & 16);
  fold<8, M2>(v, lane & 8);
  fold<4, M3>(v, lane & 4);
  fold<2, M4>(v, lane & 2);
  fold<1, M5>(v, lane & 1);
  // Which sum this lane holds: first index and count of what it kept.
  int first = 0, count = P;
  constexpr int m[6] = {P, M1, M2, M3, M4, M5};
  bool owner = true;  // one lane of those that hold the same sum
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    const bool up = lane & (32 >> s);
    const int h = (m[s] + 1) / 2;
    if (m[s] == 1) {
      owner &= !up;
    } else if (up) {
      first += h;
      count -= h;
    } else {
      count = count < h ? count : h;
    }
  }
  if (owner && count >= 1) out[first] = v[0];
}

// Ri = R^-1 (upper) for the Gram matrix g = R^T R in registers; returns the
// smallest ratio of a pivot to its column's squared norm.  A start vector
// inside the span of the others keeps a tiny pivot instead of a NaN.
template <int MM>
__device__ __forceinline__ double chol_regs(const double* g, double (&Ri)[MM][MM]) {
  double R[MM][MM];
  double low = 1.0;
#pragma unroll
  for (int j = 0; j < MM; ++j) {
    const double gjj = g[tri<MM>(j, j)];
    double d = gjj;
#pragma unroll
    for (int k = 0; k < j; ++k) d -= R[k][j] * R[k][j];
    if (!(d >= kModeQr2 * gjj)) low = 0.0;
    const double inv = rsqrt(d > 1e-300 ? d : 1e-300);
    Ri[j][j] = inv;
#pragma unroll
    for (int i = j + 1; i < MM; ++i) {
      double t = g[tri<MM>(j, i)];
#pragma unroll
      for (int k = 0; k < j; ++k) t -= R[k][j] * R[k][i];
      R[j][i] = t * inv;
    }
  }
#pragma unroll
  for (int j = 0; j < MM; ++j) {
#pragma unroll
    for (int i = j - 1; i >= 0; --i) {
      double t = 0.0;
#pragma unroll
      for (int k = i + 1; k <= j; ++k) t += R[i][k] * Ri[k][j];
      Ri[i][j] = -t * Ri[i][i];
    }
  }
  return low;
}

template <int MM>
__device__ __forceinline__ void row_ri_regs(float (&v)[MM], const double (&Ri)[MM][MM]) {
  float o[MM];
#pragma unroll
  for (int k = 0; k < MM; ++k) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j <= k; ++j) t += (double)v[j] * Ri[j][k];
    o[k] = (float)t;
  }
#pragma unroll
  for (int k = 0; k < MM; ++k) v[k] = o[k];
}

// EX: workgroups exchange; without, one workgroup a frequency stops by itself
// (a kernel of its own: with the exchange's code in it, unused, a 30 x 20 call
// of 1500 iterations took 3.80 ms instead of 3.60).
template <int MM, int CPT, bool EX>
__global__ __launch_bounds__(kModeThreads) void k_mode_tile(TileArgs ta) {
  constexpr int NQ = ModeLds<MM>::NQ, NPAIR = ModeLds<MM>::NPAIR, NALL = ModeLds<MM>::NALL;
  constexpr int T = kModeThreads;
  const ModeArgs& a = ta.m;
  const int XX = a.XX, YY = a.YY, PC = XX * YY, gpf = EX ? a.gpf : 1;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int f = blockIdx.x / gpf, part = blockIdx.x - f * gpf;
  const int r0 = part * ta.R, R = min(ta.R, XX - r0);  // own rows r0 .. r0 + R - 1
  const int rowlen = YY * MM;
  extern __shared__ float dyn[];
  float* X0 = dyn;                       // rows r0 - 1 .. r0 + R of x, component 0
  float* X1 = X0 + (R + 2) * rowlen;     // component 1
  float* Bf = X1 + (R + 2) * rowlen;     // b, rows r0 .. r0 + R
  float* Cf = Bf + (R + 1) * rowlen;     // c, rows r0 - 1 .. r0 + R - 1
  float* ezn = Cf + (R + 1) * rowlen;    // eps_z of row r0 + R
  __shared__ double red[kModeWaves][NALL];
  __shared__ double sum[NALL];
  __shared__ int s_go;
  __shared__ unsigned s_end;  // of the workgroup's waits

  if constexpr (EX) {
    // (Without time to wait, a test: a workgroup is missing.)
    if (ta.waits.ticks == 0 && blockIdx.x + 1 == gridDim.x) return;
    if (t == 0) s_end = wait_end(ta.waits);
  }

  const TileBox tb = tile_box(gridDim.x / gpf, gpf, YY, MM);
  const long long n = 2LL * PC;
  float* xg = a.x + (long long)f * n * MM;
  const float om = a.omega[f], om2 = om * om, s = a.shift[f];

  // Own cells: place in the tile and the neighbours' columns.
  float x[CPT][2][MM], y[CPT][2][MM];
  float ka0[CPT], ka1[CPT], exv[CPT], eyv[CPT], ezv[CPT];
  int lr[CPT], jj[CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int p = c * T + t;
    lr[c] = p < R * YY ? p / YY : -1;
    jj[c] = p - (lr[c] < 0 ? 0 : lr[c]) * YY;
    const int g = lr[c] < 0 ? 0 : (r0 + lr[c]) * YY + jj[c];
    exv[c] = a.eps[g];
    eyv[c] = a.eps[PC + g];
    ezv[c] = a.eps[2 * PC + g];
    ka0[c] = om2 * eyv[c] - s;
    ka1[c] = om2 * exv[c] - s;
#pragma unroll
    for (int k = 0; k < MM; ++k) {
      x[c][0][k] = xg[(long long)g * MM + k];
      x[c][1][k] = xg[((long long)PC + g) * MM + k];
      y[c][0][k] = y[c][1][k] = 0.0f;
    }
  }
  const int up = r0 == 0 ? XX - 1 : r0 - 1, dn = r0 + R == XX ? 0 : r0 + R;
  for (int j = t; j < YY; j += T) ezn[j] = a.eps[2 * PC + dn * YY + j];
  for (int e = t; e < rowlen; e += T) {
    X0[e] = xg[(long long)up * rowlen + e];
    X1[e] = xg[(long long)PC * MM + (long long)up * rowlen + e];
    X0[(R + 1) * rowlen + e] = xg[(long long)dn * rowlen + e];
    X1[(R + 1) * rowlen + e] = xg[(long long)PC * MM + (long long)dn * rowlen + e];
  }
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    if (lr[c] < 0) continue;
    const int o = (lr[c] + 1) * rowlen + jj[c] * MM;
#pragma unroll
    for (int k = 0; k < MM; ++k) {
      X0[o + k] = x[c][0][k];
      X1[o + k] = x[c][1][k];
    }
  }

  unsigned seq = 0;
  // Sums of the wave rows in red over the workgroup: into sum[off .. off + P)
  // with one workgroup, else posted for the frequency's others.
  auto post_sums = [&](auto off_c, auto p_c) {
    constexpr int off = decltype(off_c)::value, P = decltype(p_c)::value;
    __syncthreads();
    if (t < P) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < kModeWaves; ++w) v += red[w][off + t];
      if (gpf == 1) {
        sum[off + t] = v;
      } else {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        word_t* q = ta.box + (seq & 1) * tb.total + tb.sum +
                    (((size_t)f * NALL + off + t) * gpf + part) * 2;
        post_word(q, seq, (unsigned)b);
        post_word(q + 1, seq, (unsigned)(b >> 32));
      }
    }
  };
  // Everyone's posted sums added into sum[off .. off + P); ends with a barrier.
  auto collect_sums = [&](auto off_c, auto p_c) {
    constexpr int off = decltype(off_c)::value, P = decltype(p_c)::value;
    const word_t* sb = ta.box + (seq & 1) * tb.total + tb.sum + (size_t)f * gpf * NALL * 2;
    if (gpf > 1) {
      // Wave wv takes sums wv, wv + 8, ...: lane j reads workgroup j's (and
      // j + 64's, ...) and the wave adds them, in the same order everywhere.
      constexpr int NW = (P + kModeWaves - 1) / kModeWaves;
      double v[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) v[i] = 0.0;
      for (int j = lane; j < gpf; j += 64) {
        word_t lo[NW], hi[NW];
        const bool came = poll_words(&s_end, [&]() __attribute__((always_inline)) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < NW; ++i) {
            const int q = min(wv + i * kModeWaves, P - 1);
            const word_t* p = sb + ((size_t)(off + q) * gpf + j) * 2;
            lo[i] = read_word(p);
            hi[i] = read_word(p + 1);
          }
#pragma unroll
          for (int i = 0; i < NW; ++i)
            ok &= (unsigned)(lo[i] >> 32) == seq && (unsigned)(hi[i] >> 32) == seq;
          return ok;
        });
        // (A wait in vain: NaN, which ends the run.)
#pragma unroll
        for (int i = 0; i < NW; ++i)
          v[i] += came ? __builtin_bit_cast(double, (hi[i] << 32) | (lo[i] & 0xffffffffu))
                       : __builtin_nan("");
      }
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        double w[1] = {v[i]};
        const int q = wv + i * kModeWaves;
        fold<32, 1>(w, false);
        fold<16, 1>(w, false);
        fold<8, 1>(w, false);
        fold<4, 1>(w, false);
        fold<2, 1>(w, false);
        fold<1, 1>(w, false);
        if (lane == 0 && q < P) sum[off + q] = w[0];
      }
    }
    __syncthreads();
  };

  int it = 0;
  bool go = true;
  for (;;) {
    __syncthreads();
    // b (own cells and row r0 + R) and c (own cells and row r0 - 1).
    float bv[CPT][MM], cv[CPT][MM];
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      if (lr[c] < 0) continue;
      const int row = (lr[c] + 1) * rowlen, j = jj[c];
      const int jm = (j == 0 ? YY - 1 : j - 1) * MM, jp = (j == YY - 1 ? 0 : j + 1) * MM;
#pragma unroll
      for (int k = 0; k < MM; ++k) {
        const float u0 = x[c][0][k], u1 = x[c][1][k];
        bv[c][k] = (-(u0 - X0[row + jm + k]) + (u1 - X1[row - rowlen + j * MM + k])) / ezv[c];
        cv[c][k] = (X0[row + rowlen + j * MM + k] - u0) + (X1[row + jp + k] - u1);
        Bf[row - rowlen + j * MM + k] = bv[c][k];
        Cf[row + j * MM + k] = cv[c][k];
      }
    }
    for (int e = t; e < 2 * YY; e += T) {
      const bool is_c = e >= YY;
      const int j = is_c ? e - YY : e;
      const int jm = (j == 0 ? YY - 1 : j - 1) * MM, jp = (j == YY - 1 ? 0 : j + 1) * MM;
      const int row = is_c ? 0 : (R + 1) * rowlen;
#pragma unroll
      for (int k = 0; k < MM; ++k) {
        const float u0 = X0[row + j * MM + k], u1 = X1[row + j * MM + k];
        if (is_c)
          Cf[j * MM + k] = (X0[rowlen + j * MM + k] - u0) + (X1[jp + k] - u1);
        else
          Bf[R * rowlen + j * MM + k] =
              (-(u0 - X0[row + jm + k]) + (u1 - X1[row - rowlen + j * MM + k])) / ezn[j];
      }
    }
    __syncthreads();
    // y = A x, its sums, and its boundary rows to the neighbours.
    ++seq;
    double acc[NALL];
#pragma unroll
    for (int q = 0; q < NALL; ++q) acc[q] = 0.0;
    word_t* rb = ta.box + (seq & 1) * tb.total + tb.row + (size_t)f * gpf * 4 * rowlen;
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      if (lr[c] < 0) continue;
      const int brow = lr[c] * rowlen, j = jj[c];
      const int jm = (j == 0 ? YY - 1 : j - 1) * MM, jp = (j == YY - 1 ? 0 : j + 1) * MM;
#pragma unroll
      for (int k = 0; k < MM; ++k) {
        const float x0 = x[c][0][k], x1 = x[c][1][k], b = bv[c][k], cc = cv[c][k];
        const float a0 = ka0[c] * x0, a1 = ka1[c] * x1;
        const float b0 = -(Bf[brow + jp + k] - b) * eyv[c];
        const float b1 = (Bf[brow + rowlen + j * MM + k] - b) * exv[c];
        const float y0 = (a0 + b0) + (cc - Cf[brow + j * MM + k]);
        const float y1 = (a1 + b1) + (cc - Cf[brow + rowlen + jm + k]);
        y[c][0][k] = y0;
        y[c][1][k] = y1;
        acc[k] += (double)x0 * y0 + (double)x1 * y1;
        acc[MM + k] += (double)y0 * y0 + (double)y1 * y1;
        acc[2 * MM + k] += (double)x0 * x0 + (double)x1 * x1;
      }
      add_gram<MM>(acc, NQ, y[c][0]);
      add_gram<MM>(acc, NQ, y[c][1]);
      if (gpf > 1) {
        if (lr[c] == 0) {
          word_t* q = rb + (size_t)(part * 2 + 0) * 2 * rowlen + j * MM;
#pragma unroll
          for (int k = 0; k < MM; ++k) {
            post_word(q + k, seq, __float_as_uint(y[c][0][k]));
            post_word(q + rowlen + k, seq, __float_as_uint(y[c][1][k]));
          }
        }
        if (lr[c] == R - 1) {
          word_t* q = rb + (size_t)(part * 2 + 1) * 2 * rowlen + j * MM;
#pragma unroll
          for (int k = 0; k < MM; ++k) {
            post_word(q + k, seq, __float_as_uint(y[c][0][k]));
            post_word(q + rowlen + k, seq, __float_as_uint(y[c][1][k]));
          }
        }
      }
    }
    wave_sums<NALL>(acc, red[wv]);
    post_sums(std::integral_constant<int, 0>(), std::integral_constant<int, NALL>());
    // The neighbours' rows of y, as they are, into the tile's edge rows (x is
    // not read there again before it is made from them).
    if (gpf > 1) {
      const int pu = part == 0 ? gpf - 1 : part - 1, pd = part == gpf - 1 ? 0 : part + 1;
      for (int e = t; e < 4 * YY; e += T) {
        const int side = e / (2 * YY), comp = (e / YY) & 1, j = e - (e / YY) * YY;
        const word_t* q = rb + ((size_t)((side ? pd * 2 : pu * 2 + 1) * 2 + comp) * YY + j) * MM;
        float* d = (comp ? X1 : X0) + (side ? (R + 1) * rowlen : 0) + j * MM;
        word_t v[MM];
        const bool came = poll_words(&s_end, [&]() __attribute__((always_inline)) {
          bool ok = true;
#pragma unroll
          for (int k = 0; k < MM; ++k) v[k] = read_word(q + k);
#pragma unroll
          for (int k = 0; k < MM; ++k) ok &= (unsigned)(v[k] >> 32) == seq;
          return ok;
        });
#pragma unroll
        for (int k = 0; k < MM; ++k)
          d[k] = came ? __uint_as_float((unsigned)v[k]) : __builtin_nanf("");
      }
    }
    collect_sums(std::integral_constant<int, 0>(), std::integral_constant<int, NALL>());
    // The stop test: while the largest residual is above tol, which a NaN ends
    // (the square of the residual against tol's: no square root).
    if (it > 0) {
      bool above = false, nan = false;
      for (int k = 0; k < MM; ++k) {
        const double xy = sum[k], yy = sum[MM + k], xx = sum[2 * MM + k];
        const double e2 = yy - 2.0 * xy * xy + xy * xy * xx;
        nan |= !(e2 == e2);
        above |= e2 > (double)a.tol * (double)a.tol;
      }
      go = above && !nan;
      if (EX && ta.joint && gridDim.x > (unsigned)gpf) {
        // All frequencies: one word each, numbered by the iteration.
        const int ww = gridDim.x / gpf;
        word_t* gb = ta.box + (it & 1) * tb.total + tb.go;
        if (part == 0 && t == 0) post_word(gb + f, it, (above ? 1 : 0) | (nan ? 2 : 0));
        if (t == 0) s_go = 0;
        __syncthreads();
        int got = 0;
        for (int g = t; g < ww; g += T) {
          word_t v;
          const bool came = poll_words(&s_end, [&]() __attribute__((always_inline)) {
            v = read_word(gb + g);
            return (unsigned)(v >> 32) == (unsigned)it;
          });
          got |= came ? (int)(unsigned)v : 2;
        }
        if (got) atomicOr(&s_go, got);
        __syncthreads();
        go = s_go == 1;
        __syncthreads();
      }
    }
    if (it >= a.max_iters || !go) break;
    ++it;
    // x = y R^-1 for the own cells and the edge rows.
    double Ri[MM][MM];
    const double low = chol_regs<MM>(sum + NQ, Ri);
    const bool twice = MM > 1 && low == 0.0;
    const int edges = gpf > 1 ? 4 * YY : 0;
    auto edge_rows = [&](const double (&M)[MM][MM]) {
      for (int e = t; e < edges; e += T) {
        const int side = e / (2 * YY), comp = (e / YY) & 1, j = e - (e / YY) * YY;
        float* d = (comp ? X1 : X0) + (side ? (R + 1) * rowlen : 0) + j * MM;
        float v[MM];
#pragma unroll
        for (int k = 0; k < MM; ++k) v[k] = d[k];
        row_ri_regs<MM>(v, M);
#pragma unroll
        for (int k = 0; k < MM; ++k) d[k] = v[k];
      }
    };
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int k = 0; k < MM; ++k) x[c][h][k] = y[c][h][k];
        row_ri_regs<MM>(x[c][h], Ri);
      }
    }
    edge_rows(Ri);
    if (twice) {
      double g[NPAIR];
#pragma unroll
      for (int q = 0; q < NPAIR; ++q) g[q] = 0.0;
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        if (lr[c] < 0) continue;
        add_gram<MM>(g, 0, x[c][0]);
        add_gram<MM>(g, 0, x[c][1]);
      }
      ++seq;
      wave_sums<NPAIR>(g, red[wv] + NQ);
      post_sums(std::integral_constant<int, NQ>(), std::integral_constant<int, NPAIR>());
      collect_sums(std::integral_constant<int, NQ>(), std::integral_constant<int, NPAIR>());
      chol_regs<MM>(sum + NQ, Ri);
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        row_ri_regs<MM>(x[c][0], Ri);
        row_ri_regs<MM>(x[c][1], Ri);
      }
      edge_rows(Ri);
    }
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      if (lr[c] < 0) continue;
      const int o = (lr[c] + 1) * rowlen + jj[c] * MM;
#pragma unroll
      for (int k = 0; k < MM; ++k) {
        X0[o + k] = x[c][0][k];
        X1[o + k] = x[c][1][k];
        if (gpf == 1 && lr[c] == R - 1) {
          X0[jj[c] * MM + k] = x[c][0][k];
          X1[jj[c] * MM + k] = x[c][1][k];
        }
        if (gpf == 1 && lr[c] == 0) {
          X0[(R + 1) * rowlen + jj[c] * MM + k] = x[c][0][k];
          X1[(R + 1) * rowlen + jj[c] * MM + k] = x[c][1][k];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    if (lr[c] < 0) continue;
    const long long g = (long long)(r0 + lr[c]) * YY + jj[c];
#pragma unroll
    for (int k = 0; k < MM; ++k) {
      xg[g * MM + k] = x[c][0][k];
      xg[(PC + g) * MM + k] = x[c][1][k];
    }
  }
  __syncthreads();
  const bool late = EX && s_end == kLate;
  if (late) {
    if (t == 0) {
      xg[(long long)r0 * rowlen] = __builtin_nanf("");
      tell_late(ta.waits);
    }
  }
  if (part == 0 && t == 0) {
    a.iters[f] = it;
    if (late) {
      for (int k = 0; k < MM; ++k) a.w[f * MM + k] = a.err[f * MM + k] = __builtin_nanf("");
    } else if (it > 0) {
      residuals<MM>(sum, a.w + f * MM, a.err + f * MM, true);
    } else {
      for (int k = 0; k < MM; ++k) {
        a.w[f * MM + k] = 0.0f;
        a.err[f * MM + k] = __builtin_inff();
      }
    }
  }
}

// ------------------------------------------------------------------ host side

// Rows a workgroup and workgroups a frequency of the tile kernel, from the
// sizes alone (the workspace is sized by it); R = 0 where it does not apply:
// more than kTileMaxModes modes, rows too long for a workgroup, or more
// workgroups than a device holds at once.
struct TilePlan {
  int R, gpf;
};

TilePlan tile_plan(int ww, int XX, int YY, int mm) {
  const TilePlan none{0, 0};
  const int most_cells = tile_max_cells(mm) * kModeThreads;  // of a workgroup
  if (mm > kTileMaxModes || YY > most_cells) return none;
  const long long cells = (long long)XX * YY;
  // One workgroup up to 1024 cells (2 modes: 30 x 20 2.1 us an iteration
  // against 3.0 on two, 40 x 30 3.2 against 3.2 on three), above that one per
  // 512 (60 x 40: 3.4 us, one per 1024 3.8, one per 2048 4.7; 256 x 128: 3.4,
  // 3.9, 5.4), at most 128 (512 x 128, 1 mode: 2.6 us, with 64 2.9).
  long long gpf = cells <= 1024 ? 1 : std::min<long long>({128, XX, (cells + 511) / 512});
  long long R = std::min<long long>((XX + gpf - 1) / gpf, most_cells / YY);
  while (R > 0 && tile_lds((int)R, YY, mm) > (size_t)kTileLds) --R;
  if (R < 1) return none;
  gpf = (XX + R - 1) / R;
  if (gpf > kTileMaxWgs || (gpf > 1 && gpf * ww > kTileMaxGrid)) return none;
  return {(int)R, (int)gpf};
}

size_t tile_words(int ww, int XX, int YY, int mm) {
  const TilePlan p = tile_plan(ww, XX, YY, mm);
  return p.R > 0 ? 2 * tile_box(ww, p.gpf, YY, mm).total : 0;
}

// Workgroups per frequency for the grid kernel, or 0 to use one workgroup:
// about one workgroup per 8192 cells x modes, at most kModeMaxShare (grid
// barriers cost more as the grid grows), and only when the whole grid fits on
// the device at once (a cooperative launch needs every workgroup resident).
template <int MM>
static int grid_share(int ww, int XX, int YY) {
  const long long work = (long long)XX * YY * MM;
  if (work < kModeJointWork) return 0;
  int gpf = (int)std::min<long long>(kModeMaxShare, (work + 8191) / 8192);
  int dev = 0, cus = 0, coop = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess ||
      !coop ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &per_cu, reinterpret_cast<const void*>(&k_mode_grid<MM>), kModeThreads, 0) !=
          hipSuccess)
    return 0;
  const long long slots = (long long)cus * per_cu;
  while (gpf > 1 && (long long)gpf * ww > slots) gpf /= 2;
  return gpf >= 2 && (long long)gpf * ww <= slots ? gpf : 0;
}

size_t mode_workspace_floats(int ww, int XX, int YY, int mm, bool tile) {
  // y and bc, then (256-byte aligned) the grid kernel's partial sums:
  // kModeMaxShare rows of NQ + NPAIR doubles per frequency.
  // The tile kernel's exchange words take the same memory, in some sections
  // more: a workspace without it is left to the other kernels.
  const size_t nall = 3 * (size_t)mm + (size_t)mm * (mm + 1) / 2;
  const size_t others =
      2 * (size_t)ww * 2 * XX * YY * mm + 64 + (size_t)ww * kModeMaxShare * nall * 2;
  return tile ? std::max(others, 2 * tile_words(ww, XX, YY, mm) + 64) : others;
}

// The tile kernel where it applies; *done says whether it runs.
template <int MM, int CPT>
static hipError_t launch_tile(const ModeArgs& a, int ww, TilePlan p, float* ws, hipStream_t s,
                              const WaitWords& waits, bool* done) {
  TileArgs ta;
  ta.waits = {};
  ta.m = a;
  ta.m.gpf = p.gpf;
  ta.R = p.R;
  // Small sections stop frequency by frequency, large ones together.
  ta.joint = (long long)a.XX * a.YY * MM >= kModeJointWork;
  ta.box = reinterpret_cast<word_t*>((reinterpret_cast<uintptr_t>(ws) + 255) & ~uintptr_t(255));
  const void* kernel = reinterpret_cast<const void*>(&k_mode_tile<MM, CPT, true>);
  const size_t lds = tile_lds(p.R, a.YY, MM);
  const bool coop = p.gpf > 1 || (ta.joint && ww > 1);
  if (coop) {
    if (!waits.report) return hipSuccess;
    // Every workgroup has to be resident at once.  A small section's launch
    // can be recorded into a graph, which a cooperative one might not.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (!ta.joint && (hipStreamIsCapturing(s, &cap) != hipSuccess ||
                      cap != hipStreamCaptureStatusNone))
      return hipSuccess;
    int dev = 0, cus = 0, ok = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&ok, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !ok ||
        !whole_device(s, cus) ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kModeThreads, lds) !=
            hipSuccess ||
        (long long)p.gpf * ww > (long long)cus * per_cu)
      return hipSuccess;
    hipError_t e = launch_zero(reinterpret_cast<float*>(ta.box),
                               4 * tile_box(ww, p.gpf, a.YY, MM).total, s);
    if (e != hipSuccess) return e;
    // 60 s, as the resident steppers' launches, and 0.1 ms an iteration (of
    // 2-8 us).
    const double ms = waits.no_time ? 0.0 : 60e3 + 0.1 * a.max_iters;
    ta.waits.ticks = (unsigned)std::min(ms * (100e3 / kWaitTick), 1e9);
    ta.waits.stalled =
        reinterpret_cast<unsigned*>(ta.box + tile_box(ww, p.gpf, a.YY, MM).late);
    ta.waits.report = waits.report;
    void* args[] = {&ta};
    e = waits.refused() ? hipErrorCooperativeLaunchTooLarge
                        : hipLaunchCooperativeKernel(kernel, dim3(ww * p.gpf), dim3(kModeThreads),
                                                     args, (unsigned)lds, s);
    // A refused launch leaves it to the other kernels.
    *done = e == hipSuccess;
    if (!*done) (void)hipGetLastError();
    return hipSuccess;
  }
  *done = true;
  hipLaunchKernelGGL((k_mode_tile<MM, CPT, false>), dim3(ww), dim3(kModeThreads), lds, s, ta);
  return hipGetLastError();
}

template <int MM>
static hipError_t launch_mode_mm(ModeArgs a, int ww, float* ws, bool tile, const WaitWords& waits,
                                 hipStream_t s) {
  if constexpr (MM <= kTileMaxModes) {
    const TilePlan p = tile_plan(ww, a.XX, a.YY, MM);
    if (tile && p.R > 0) {
      bool done = false;
      const int cells = p.R * a.YY;
      const hipError_t e =
          cells <= kModeThreads ? launch_tile<MM, 1>(a, ww, p, ws, s, waits, &done)
          : cells <= 2 * kModeThreads
              ? launch_tile<MM, 2>(a, ww, p, ws, s, waits, &done)
              : launch_tile<MM, tile_max_cells(MM)>(a, ww, p, ws, s, waits, &done);
      if (done || e != hipSuccess) return e;
    }
  }
  const int gpf = grid_share<MM>(ww, a.XX, a.YY);
  if (gpf > 0) {
    a.gpf = gpf;
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&k_mode_grid<MM>),
                                      dim3(ww * gpf), dim3(kModeThreads), args, 0, s);
  }
  hipLaunchKernelGGL((k_mode_subspace<MM>), dim3(ww), dim3(kModeThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_mode(int ww, int XX, int YY, int mm, const float* eps, const float* omega,
                       const float* shift, float* x, float* w, float* err, int* iters,
                       int max_iters, float tol, float* ws, bool tile, const WaitWords& waits,
                       hipStream_t s) {
  ModeArgs a;
  a.XX = XX;
  a.YY = YY;
  a.max_iters = max_iters;
  a.tol = tol;
  a.eps = eps;
  a.omega = omega;
  a.shift = shift;
  a.x = x;
  const size_t vec = (size_t)ww * 2 * XX * YY * mm;
  a.y = ws;
  a.bc = ws + vec;
  const uintptr_t pbase = (reinterpret_cast<uintptr_t>(ws + 2 * vec) + 255) & ~uintptr_t(255);
  a.partial = reinterpret_cast<double*>(pbase);
  a.gpf = 1;
  a.w = w;
  a.err = err;
  a.iters = iters;
  switch (mm) {
    case 1: return launch_mode_mm<1>(a, ww, ws, tile, waits, s);
    case 2: return launch_mode_mm<2>(a, ww, ws, tile, waits, s);
    case 3: return launch_mode_mm<3>(a, ww, ws, tile, waits, s);
    case 4: return launch_mode_mm<4>(a, ww, ws, tile, waits, s);
    case 5: return launch_mode_mm<5>(a, ww, ws, tile, waits, s);
    case 6: return launch_mode_mm<6>(a, ww, ws, tile, waits, s);
    case 7: return launch_mode_mm<7>(a, ww, ws, tile, waits, s);
    case 8: return launch_mode_mm<8>(a, ww, ws, tile, waits, s);
    case 9: return launch_mode_mm<9>(a, ww, ws, tile, waits, s);
    case 10: return launch_mode_mm<10>(a, ww, ws, tile, waits, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pjz
