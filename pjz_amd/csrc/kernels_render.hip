// pjz's permittivity render (src/pjz/_epsilon.py:10-108) on the device:
// layered 2-D profiles magnified 2m x 2m -> (3, xx, yy, zz) Yee-cell eps by
// Farjadpour et al.'s diagonal sub-pixel average, with the exact reverse pass
// for the layers and the interface positions.
//
//   forward:  k_render_stats    per (component, layer, pixel): mean, mean of
//                               the inverse and the two in-plane moments of
//                               the component's half-cell-shifted 2m x 2m
//                               tile (:12-16, 26-45)
//             k_render_shares   per (z grid, layer, z): the layer's share of
//                               the cell and its z moment (:47-61, 75-87)
//             k_render_combine  per (component, x, y, z): the moments mixed
//                               by the shares into 1 / (p aoi + (1 - p) /
//                               avg) or the plain average (:63-99);
//                               k_render_combine_cells past 4 layers
//   backward: k_render_bwd_cells   dL/dstats, summed over z, and dL/d(z share,
//                                  z-moment share), summed over the pixels of
//                                  a workgroup, in one pass over the cells;
//                                  k_render_bwd_all_cells past 4 layers
//             k_render_sum_parts   the workgroups' share sums added
//             k_render_bwd_pos     dL/d(interface positions)
//             k_render_bwd_layers  dL/d(layer sub-pixels), gathered through
//                                  the shifts' edge replication
// Layouts (fp32): layers (ll, SX = 2m xx, SY = 2m yy); stats (3, 4, ll, xx,
// yy) with the four moments (mean, mean of inverse, x moment, y moment),
// then each layer's share of each cell (k_render_shares); eps (3, xx, yy,
// zz).  Grid bounds gs, ge are (zz, 2): column 0 for the x
// and y components, column 1 for z (:18-24).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fdtd_common.h"

namespace pjz {

namespace {

struct RenderDims {
  int ll, m, xx, yy, zz, simple;
};

__device__ inline size_t stat_at(const RenderDims& d, int a, int q, int l, int x, int y) {
  return ((((size_t)a * 4 + q) * d.ll + l) * d.xx + x) * (size_t)d.yy + y;
}

// Source sub-pixel a component's shifted sub-pixel (i, j) reads: components
// not along x are shifted by m sub-pixels in x (edge-replicated at the
// start), likewise in y (:12-16).
__device__ inline int src_x(int a, int i, int m) { return a != 0 ? max(i - m, 0) : i; }
__device__ inline int src_y(int a, int j, int m) { return a != 1 ? max(j - m, 0) : j; }

__global__ __launch_bounds__(256) void k_render_stats(RenderDims d, const float* __restrict__ L,
                                                      float* __restrict__ st) {
  // 3 ll xx yy < 2^31 (the arrays' bound of the C ABI): 32-bit indices
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned np = (unsigned)d.xx * d.yy;
  if (i >= 3u * d.ll * np) return;
  const unsigned al = i / np, p = i - al * np;
  const int x = p / (unsigned)d.yy, y = p - x * (unsigned)d.yy;
  const int a = al / (unsigned)d.ll, l = al - a * (unsigned)d.ll;
  const int n = 2 * d.m, SX = n * d.xx, SY = n * d.yy;
  const float* Ll = L + (size_t)l * SX * SY;
  float s = 0.0f, si = 0.0f, sx = 0.0f, sy = 0.0f;
  for (int di = 0; di < n; ++di) {
    const float wx = (di - (d.m - 0.5f)) / (float)(n * n);
    const int r = src_x(a, n * x + di, d.m);
    for (int dj = 0; dj < n; ++dj) {
      const float wy = (dj - (d.m - 0.5f)) / (float)(n * n);
      const float v = Ll[(size_t)r * SY + src_y(a, n * y + dj, d.m)];
      s += v;
      si += 1.0f / v;
      sx += v * wx;
      sy += v * wy;
    }
  }
  const float inv = 1.0f / (float)(n * n);
  st[stat_at(d, a, 0, l, x, y)] = s * inv;
  st[stat_at(d, a, 1, l, x, y)] = si * inv;
  // mean of 12 (2m) v w (:35-37)
  st[stat_at(d, a, 2, l, x, y)] = 12.0f * n * sx * inv;
  st[stat_at(d, a, 3, l, x, y)] = 12.0f * n * sy * inv;
}

// Layer l's share u of cell z (grid column col) and its z moment
// uz = u zc / (dz^2 / 12) (:47-61, 75-87), with what the reverse pass needs.
struct Share {
  float u, uz, p0, p1, gs, ge;
};

__device__ inline Share layer_share(const RenderDims& d, const float* __restrict__ pos,
                                    const float* __restrict__ gsa, const float* __restrict__ gea,
                                    int l, int z, int col) {
  Share s;
  s.gs = gsa[2 * z + col];
  s.ge = gea[2 * z + col];
  const float lo = l == 0 ? -INFINITY : pos[l - 1];
  const float hi = l == d.ll - 1 ? INFINITY : pos[l];
  s.p0 = fminf(fmaxf(lo, s.gs), s.ge);
  s.p1 = fminf(fmaxf(hi, s.gs), s.ge);
  const float dz = s.ge - s.gs;
  s.u = (s.p1 - s.p0) / dz;
  const float zc = (s.p0 + s.p1) / 2 - (s.gs + s.ge) / 2;
  s.uz = s.u * zc / (dz * dz / 12.0f);
  return s;
}

// The share table: (u, uz) of every layer and cell for both z grids,
// table[((col * ll + l) * zz + z) * 2 + {0, 1}], after the 12 ll xx yy
// moments in the stats array.
__global__ __launch_bounds__(256) void k_render_shares(RenderDims d, const float* __restrict__ pos,
                                                       const float* __restrict__ gsa,
                                                       const float* __restrict__ gea,
                                                       float* __restrict__ tab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * d.ll * d.zz) return;
  const int z = i % d.zz, l = (i / d.zz) % d.ll, col = i / (d.zz * d.ll);
  const Share sh = layer_share(d, pos, gsa, gea, l, z, col);
  tab[2 * i] = sh.u;
  tab[2 * i + 1] = sh.uz;
}

__device__ inline const float* share_at(const RenderDims& d, const float* tab, int a, int l,
                                        int z) {
  return tab + (((a == 2 ? 1 : 0) * d.ll + l) * (size_t)d.zz + z) * 2;
}

// Mixed sums of one output cell and its value.
struct Mix {
  float A, B, g0, g1, g2, out, pii, iT, iA;
};

constexpr int kRenderMaxLayers = 16;
static_assert(kRenderMaxLayers == PJZ_FDTD_RENDER_MAX_LAYERS, "layer bound of the C ABI");

// The moment along the component's own axis (selected, not indexed: an array
// here goes to scratch memory).
__device__ __forceinline__ float own_moment(float g0, float g1, float g2, int a) {
  return a == 0 ? g0 : (a == 1 ? g1 : g2);
}

// Finishes a cell from its mixed sums (:89-99).
__device__ inline void mix_finish(Mix& r, int simple, int a) {
  if (simple) {
    r.out = r.A;
    r.pii = r.iT = r.iA = 0.0f;
    return;
  }
  const float T = r.g0 * r.g0 + r.g1 * r.g1 + r.g2 * r.g2;
  const float g0 = r.g0, g1 = r.g1, g2 = r.g2;
  const float ga = own_moment(g0, g1, g2, a);
  r.pii = ga * ga / (T == 0.0f ? 1.0f : T);  // (:92-95)
  r.iT = T == 0.0f ? 0.0f : 1.0f / T;
  r.iA = 1.0f / r.A;
  r.out = 1.0f / (r.pii * r.B + (1.0f - r.pii) * r.iA);  // (:97)
}

// Cotangents of a cell's mixed sums A, B, G = (g0, g1, g2) from g = dL/d(out).
struct MixGrad {
  float gA, gB, gG[3];
};

__device__ __forceinline__ MixGrad mix_grad(int simple, const Mix& r, int a, float g) {
  MixGrad t;
  if (simple) {
    t.gA = g;
    t.gB = t.gG[0] = t.gG[1] = t.gG[2] = 0.0f;
    return t;
  }
  // out = 1 / D, D = pii B + (1 - pii) / A, pii = G_a^2 / T (T = sum G_k^2,
  // no gradient through T where T = 0, where every G_k and pii are 0):
  // dpii/dG_k = (2 G_a [k = a] - 2 pii G_k) / T.
  const float gD = -g * r.out * r.out;
  t.gA = gD * (1.0f - r.pii) * (-r.iA * r.iA);
  t.gB = gD * r.pii;
  const float gp = gD * (r.B - r.iA) * (2.0f * r.iT);
  const float g0 = r.g0, g1 = r.g1, g2 = r.g2;
  const float ga = own_moment(g0, g1, g2, a);
  t.gG[0] = gp * ((a == 0 ? ga : 0.0f) - r.pii * r.g0);
  t.gG[1] = gp * ((a == 1 ? ga : 0.0f) - r.pii * r.g1);
  t.gG[2] = gp * ((a == 2 ? ga : 0.0f) - r.pii * r.g2);
  return t;
}

// The cell kernels of more than 4 layers (k_render_combine_cells,
// k_render_bwd_all_cells; fewer go by classes, below): a wave walks over
// pixels of one component with its lanes on z, so the output (or its
// cotangent) is read and written in whole rows of zz floats and the layers'
// shares of the lane's cells stay in registers.  The 4 LL moments of 16
// pixels at a time come in as 16 lanes of as many loads and reach all lanes
// by readlane.  C cells a lane cover the z range [z0, z0 + 64 C); taller
// stacks take several launches.  The kernels these replaced gave each
// (component, z, pixel) a thread: they read the cotangent with the pixels on
// the lanes (one float of every 512-byte row) and divided 64-bit indices per
// cell.  384 x 384 x 128 cells, 3 layers: combine 342 -> 135 us, the
// two reverse passes 972 + 622 -> 315 us in one.
constexpr int kRenderWaves = 4;  // waves of a workgroup

template <int LL, int C>
struct Shares {
  float u[C][LL], uz[C][LL];
};

template <int LL, int C>
__device__ inline void load_shares(Shares<LL, C>& S, const RenderDims& d, const float* tab, int a,
                                   int z0, int lane) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int z = min(z0 + 64 * c + lane, d.zz - 1);
#pragma unroll
    for (int l = 0; l < LL; ++l) {
      const float* sh = share_at(d, tab, a, min(l, d.ll - 1), z);
      S.u[c][l] = l < d.ll ? sh[0] : 0.0f;
      S.uz[c][l] = l < d.ll ? sh[1] : 0.0f;
    }
  }
}

// Moments of pixels p .. p + 15 (lane & 15) of component a; 0 past the last
// layer, the last pixel repeated past the end.
template <int LL>
__device__ inline void load_moments(float (&m)[LL][4], const RenderDims& d,
                                    const float* __restrict__ st, int a, int p, int np, int lane) {
  const int q0 = min(p + (lane & 15), np - 1);
#pragma unroll
  for (int l = 0; l < LL; ++l)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      m[l][q] = l < d.ll ? st[(((size_t)a * 4 + q) * d.ll + l) * np + q0] : 0.0f;
}

__device__ inline float from_lane(float v, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

template <int LL, int C>
__device__ inline void mix_sums(Mix& r, const float (&m)[LL][4], const Shares<LL, C>& S, int c) {
  r.A = r.B = r.g0 = r.g1 = r.g2 = 0.0f;
#pragma unroll
  for (int l = 0; l < LL; ++l) {
    r.A += m[l][0] * S.u[c][l];
    r.B += m[l][1] * S.u[c][l];
    r.g0 += m[l][2] * S.u[c][l];
    r.g1 += m[l][3] * S.u[c][l];
    r.g2 += m[l][0] * S.uz[c][l];
  }
}

// The 16-pixel groups [g0, g1) of a wave: gpw consecutive ones.
struct GroupRange {
  int g0, g1;
};
__device__ inline GroupRange wave_groups(int np, int gpw) {
  const int wave = blockIdx.x * kRenderWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = (np + 15) / 16;
  return {min(wave * gpw, n), min(wave * gpw + gpw, n)};
}

// Up to 4 layers, the cell kernels work by classes of cells.  Along z, a pixel's
// cells that no interface touches have one of LL share vectors (by how many
// interfaces lie below them), so their value and its derivatives are those of
// (pixel, class): a wave evaluates 16 pixels x 4 classes at once, one on each
// lane, instead of every cell.  A cell that an interface touches, ends included
// (where the clip's derivative is a half), is a class of its own.  What is left
// per cell is its read or write.  384 x 384 x 128 cells, 3 layers: combine
// 135 us (bound by three divisions a cell) -> 46 (226 MB written), reverse 315 -> 94.
constexpr int kPure = 4;  // classes of untouched cells, the first of a wave's list

template <int C>
struct Classes {
  int at[C];  // class of the lane's cells
  int nsp;    // cells with a class of their own
};

// Classes of the cells z0 + 64 c + lane; list[k] becomes a cell of class k, or
// -1.  Called by whole workgroups, a list a wave.
template <int C>
__device__ __forceinline__ Classes<C> cell_classes(const RenderDims& d, const float* __restrict__ pos,
                                          const float* __restrict__ gsa,
                                          const float* __restrict__ gea, int col, int z0, int lane,
                                          int* list) {
  Classes<C> K;
  K.nsp = 0;
  for (int k = lane; k < kPure + 64 * C; k += 64) list[k] = -1;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int z = z0 + 64 * c + lane, zc = min(z, d.zz - 1);
    const float gs = gsa[2 * zc + col], ge = gea[2 * zc + col];
    // (Cells whose height, or its square in the z moment, is no positive number
    // have no such share vector: what they are must not become a class's value.)
    const float dz = ge - gs;
    bool own = !(dz > 0.0f && dz < INFINITY && dz * dz / 12.0f > 0.0f);
    int below = 0;
    for (int l = 0; l + 1 < d.ll; ++l) {
      own |= !(pos[l] < gs || pos[l] > ge);
      below += pos[l] < gs ? 1 : 0;
    }
    own &= z < d.zz;
    const unsigned long long m = __ballot(own);
    const int before = __popcll(m & ((1ull << lane) - 1));
    K.at[c] = own ? kPure + K.nsp + before : below;
    K.nsp += __popcll(m);
    if (z < d.zz) list[K.at[c]] = z;
  }
  __syncthreads();
  return K;
}

// Shares of cell z (clamped to the stack) of component a.
template <int LL>
struct CellShares {
  float u[LL], uz[LL];
};
template <int LL>
__device__ __forceinline__ CellShares<LL> cell_shares(const RenderDims& d, const float* tab, int a, int z) {
  CellShares<LL> S;
#pragma unroll
  for (int l = 0; l < LL; ++l) {
    const float* sh = share_at(d, tab, a, min(l, d.ll - 1), max(z, 0));
    S.u[l] = l < d.ll ? sh[0] : 0.0f;
    S.uz[l] = l < d.ll ? sh[1] : 0.0f;
  }
  return S;
}

template <int LL>
__device__ __forceinline__ Mix class_mix(const float (&m)[LL][4], const CellShares<LL>& S,
                                         int simple, int a) {
  float A = 0.0f, B = 0.0f, g0 = 0.0f, g1 = 0.0f, g2 = 0.0f;
#pragma unroll
  for (int l = 0; l < LL; ++l) {
    A += m[l][0] * S.u[l];
    B += m[l][1] * S.u[l];
    g0 += m[l][2] * S.u[l];
    g1 += m[l][3] * S.u[l];
    g2 += m[l][0] * S.uz[l];
  }
  Mix r{A, B, g0, g1, g2, A, 0.0f, 0.0f, 0.0f};
  mix_finish(r, simple, a);
  return r;
}

template <int LL, int C>
__global__ __launch_bounds__(64 * kRenderWaves) void k_render_combine(
    RenderDims d, const float* __restrict__ st, const float* __restrict__ tab,
    const float* __restrict__ pos, const float* __restrict__ gsa, const float* __restrict__ gea,
    float* __restrict__ eps, int gpw, int z0) {
  __shared__ int lists[kRenderWaves][kPure + 64 * C];
  __shared__ __align__(16) float values[kRenderWaves][(kPure + 64 * C) * 16];  // (class, pixel)
  const int a = blockIdx.y, lane = threadIdx.x & 63, np = d.xx * d.yy;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Classes<C> K = cell_classes<C>(d, pos, gsa, gea, a == 2 ? 1 : 0, z0, lane, lists[w]);
  const GroupRange R = wave_groups(np, gpw);
  const CellShares<LL> pure = cell_shares<LL>(d, tab, a, lists[w][lane >> 4]);
  float* const val = values[w];
  for (int g = R.g0; g < R.g1; ++g) {
    float m[LL][4];
    load_moments(m, d, st, a, 16 * g, np, lane);
    val[lane] = class_mix<LL>(m, pure, d.simple, a).out;
    for (int k = 0; k < K.nsp; k += 4) {
      const int z = k + (lane >> 4) < K.nsp ? lists[w][kPure + k + (lane >> 4)] : 0;
      val[(kPure + k) * 16 + lane] =
          class_mix<LL>(m, cell_shares<LL>(d, tab, a, z), d.simple, a).out;
    }
    // The wave's own values: its LDS operations are in order.
    __builtin_amdgcn_wave_barrier();
    const int n = min(16, np - 16 * g);
    float* row = eps + ((size_t)a * np + 16 * g) * d.zz + z0 + lane;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (z0 + 64 * c + lane >= d.zz) continue;
      const float4* v = reinterpret_cast<const float4*>(val + K.at[c] * 16);
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const float4 t = v[i / 4];
        const float o[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i + j < n)
            __builtin_nontemporal_store(o[j], row + (size_t)(i + j) * d.zz + 64 * c);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int LL, int C>
__global__ __launch_bounds__(64 * kRenderWaves) void k_render_combine_cells(
    RenderDims d, const float* __restrict__ st, const float* __restrict__ tab,
    float* __restrict__ eps, int gpw, int z0) {
  const int a = blockIdx.y, lane = threadIdx.x & 63, np = d.xx * d.yy;
  const GroupRange R = wave_groups(np, gpw);
  if (R.g0 >= R.g1) return;
  Shares<LL, C> S;
  load_shares(S, d, tab, a, z0, lane);
  for (int g = R.g0; g < R.g1; ++g) {
    float m[LL][4];
    load_moments(m, d, st, a, 16 * g, np, lane);
    const int n = min(16, np - 16 * g);
    for (int i = 0; i < n; ++i) {
      float t[LL][4];
#pragma unroll
      for (int l = 0; l < LL; ++l)
#pragma unroll
        for (int q = 0; q < 4; ++q) t[l][q] = from_lane(m[l][q], i);
      float* row = eps + ((size_t)a * np + 16 * g + i) * d.zz;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int z = z0 + 64 * c + lane;
        Mix r;
        mix_sums(r, t, S, c);
        mix_finish(r, d.simple, a);
        if (z < d.zz) __builtin_nontemporal_store(r.out, row + z);
      }
    }
  }
}

// Sums 4 values over the 64 lanes: on return row r (16 lanes) of the result
// holds the sum of v[0], v[2], v[1], v[3] for r = 0..3 in each of its lanes.
// gfx950's half and row swaps fold two values into one register per add: 3
// swaps, 3 adds and 4 row rotations for 4 values, against 24 adds one by one.
__device__ inline float swap_add32(float a, float b) {
  const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                  __builtin_bit_cast(unsigned, b), false, false);
  // (copied out first: a bit cast of t[1] itself reads t[0])
  const unsigned lo = t[0], hi = t[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ inline float swap_add16(float a, float b) {
  const auto t = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                  __builtin_bit_cast(unsigned, b), false, false);
  // (copied out first: a bit cast of t[1] itself reads t[0])
  const unsigned lo = t[0], hi = t[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
template <int N>
__device__ inline float row_ror_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                           0, __builtin_bit_cast(int, v), 0x120 + N, 0xf, 0xf, true));
}
__device__ inline float sum4(float v0, float v1, float v2, float v3) {
  float s = swap_add16(swap_add32(v0, v1), swap_add32(v2, v3));
  s = row_ror_add<8>(s);
  s = row_ror_add<4>(s);
  s = row_ror_add<2>(s);
  return row_ror_add<1>(s);
}

// One pass over the cells of a component's pixels for both reductions of the
// reverse pass:
//  - dL/dstats (3, 4, ll, xx, yy): a pixel's cell cotangents times the shares,
//    summed over z across the lanes (sum4; lane 16 r + i of a layer's register
//    keeps pixel i's sum of moment r, stored 16 pixels at a time).  `add`
//    accumulates onto the z ranges of earlier launches.
//  - dL/du, dL/duz of the lane's cells, summed over the wave's pixels in
//    registers (in double once per 16 pixels), over the workgroup in LDS and
//    written to part[((blockIdx.x * 3 + a) * 2 + w) * ll * zz + l * zz + z].
template <int LL, int C>
__global__ __launch_bounds__(64 * kRenderWaves) void k_render_bwd_all_cells(
    RenderDims d, const float* __restrict__ st, const float* __restrict__ tab,
    const float* __restrict__ geps, float* __restrict__ gst, double* __restrict__ part, int gpw,
    int z0, int add) {
  __shared__ double red[kRenderWaves][64];
  const int a = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6, np = d.xx * d.yy;
  const GroupRange R = wave_groups(np, gpw);
  Shares<LL, C> S;
  load_shares(S, d, tab, a, z0, lane);
  double au[C][LL], auz[C][LL];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int l = 0; l < LL; ++l) au[c][l] = auz[c][l] = 0.0;
  // Moment held by this lane's row (sum4's order).
  const int row = lane >> 4, qrow = row == 1 ? 2 : (row == 2 ? 1 : row);
  for (int g = R.g0; g < R.g1; ++g) {
    float m[LL][4], keep[LL], fu[C][LL], fuz[C][LL];
    load_moments(m, d, st, a, 16 * g, np, lane);
#pragma unroll
    for (int l = 0; l < LL; ++l) {
      keep[l] = 0.0f;
#pragma unroll
      for (int c = 0; c < C; ++c) fu[c][l] = fuz[c][l] = 0.0f;
    }
    const int n = min(16, np - 16 * g);
    const float* grow = geps + ((size_t)a * np + 16 * g) * d.zz + z0 + lane;
    float gnext[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
      gnext[c] = z0 + 64 * c + lane < d.zz ? __builtin_nontemporal_load(grow + 64 * c) : 0.0f;
    for (int i = 0; i < n; ++i) {
      float gv[C], t[LL][4], v[LL][4];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        gv[c] = gnext[c];
        gnext[c] = i + 1 < n && z0 + 64 * c + lane < d.zz
                       ? __builtin_nontemporal_load(grow + (size_t)(i + 1) * d.zz + 64 * c)
                       : 0.0f;
      }
#pragma unroll
      for (int l = 0; l < LL; ++l)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          t[l][q] = from_lane(m[l][q], i);
          v[l][q] = 0.0f;
        }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        Mix r;
        mix_sums(r, t, S, c);
        mix_finish(r, d.simple, a);
        const MixGrad k = mix_grad(d.simple, r, a, gv[c]);
#pragma unroll
        for (int l = 0; l < LL; ++l) {
          v[l][0] += k.gA * S.u[c][l] + k.gG[2] * S.uz[c][l];
          v[l][1] += k.gB * S.u[c][l];
          v[l][2] += k.gG[0] * S.u[c][l];
          v[l][3] += k.gG[1] * S.u[c][l];
          fu[c][l] += k.gA * t[l][0] + k.gB * t[l][1] + k.gG[0] * t[l][2] + k.gG[1] * t[l][3];
          fuz[c][l] += k.gG[2] * t[l][0];
        }
      }
#pragma unroll
      for (int l = 0; l < LL; ++l) {
        const float s = sum4(v[l][0], v[l][1], v[l][2], v[l][3]);
        keep[l] = (lane & 15) == i ? s : keep[l];
      }
    }
#pragma unroll
    for (int l = 0; l < LL; ++l) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        au[c][l] += fu[c][l];
        auz[c][l] += fuz[c][l];
      }
      if (l < d.ll && (lane & 15) < n) {
        float* o = gst + (((size_t)a * 4 + qrow) * d.ll + l) * np + 16 * g + (lane & 15);
        *o = add ? *o + keep[l] : keep[l];
      }
    }
  }
  if (!part) return;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int l = 0; l < LL; ++l)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (l >= d.ll) continue;
        red[w][lane] = k == 0 ? au[c][l] : auz[c][l];
        __syncthreads();
        const int z = z0 + 64 * c + lane;
        if (w == 0 && z < d.zz) {
          double s = 0.0;
          for (int j = 0; j < kRenderWaves; ++j) s += red[j][lane];
          part[((((size_t)blockIdx.x * 3 + a) * 2 + k) * d.ll + l) * d.zz + z] = s;
        }
        __syncthreads();
      }
}

// A row's 16 lanes summed, in each of them.
__device__ inline float row_sum(float s) {
  s = row_ror_add<8>(s);
  s = row_ror_add<4>(s);
  s = row_ror_add<2>(s);
  return row_ror_add<1>(s);
}

// Both reductions of the reverse pass by classes (outputs as
// k_render_bwd_all_cells').  A pixel's cotangents are summed over the cells of
// each untouched class (sum4) and taken cell by cell for the others; every
// cotangent of the mixed sums is linear in them, so the rest is done once a
// (pixel, class).  dL/du and dL/duz are formed for the touched cells only: the
// positions' gradient takes no other.
template <int LL, int C>
__global__ __launch_bounds__(64 * kRenderWaves) void k_render_bwd_cells(
    RenderDims d, const float* __restrict__ st, const float* __restrict__ tab,
    const float* __restrict__ pos, const float* __restrict__ gsa, const float* __restrict__ gea,
    const float* __restrict__ geps, float* __restrict__ gst, double* __restrict__ part, int gpw,
    int z0, int add) {
  static_assert(LL <= kPure, "one class a row of lanes");
  __shared__ int lists[kRenderWaves][kPure + 64 * C];
  __shared__ float touched[kRenderWaves][64 * C * 16];         // cotangents (cell, pixel)
  __shared__ double acc[kRenderWaves][64 * C][2 * LL];  // dL/du, dL/duz of touched cells
  const int a = blockIdx.y, lane = threadIdx.x & 63, np = d.xx * d.yy;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Classes<C> K = cell_classes<C>(d, pos, gsa, gea, a == 2 ? 1 : 0, z0, lane, lists[w]);
  for (int q = lane; q < K.nsp * 2 * LL; q += 64) acc[w][q / (2 * LL)][q % (2 * LL)] = 0.0;
  __syncthreads();
  const GroupRange R = wave_groups(np, gpw);
  // Class, then moment, held by this lane's row (sum4's order).
  const int row = lane >> 4, qrow = row == 1 ? 2 : (row == 2 ? 1 : row);
  const CellShares<LL> pure = cell_shares<LL>(d, tab, a, lists[w][qrow]);
  for (int g = R.g0; g < R.g1; ++g) {
    float m[LL][4], gv[16][C];
    load_moments(m, d, st, a, 16 * g, np, lane);
    const int n = min(16, np - 16 * g);
    const float* grow = geps + ((size_t)a * np + 16 * g) * d.zz + z0 + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int c = 0; c < C; ++c)
        gv[i][c] = i < n && z0 + 64 * c + lane < d.zz
                       ? __builtin_nontemporal_load(grow + (size_t)i * d.zz + 64 * c)
                       : 0.0f;
    float keep = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < C; ++c) {
#pragma unroll
        for (int k = 0; k < LL; ++k) v[k] += K.at[c] == k ? gv[i][c] : 0.0f;
        if (K.at[c] >= kPure) touched[w][(K.at[c] - kPure) * 16 + i] = gv[i][c];
      }
      const float s = sum4(v[0], v[1], v[2], v[3]);
      keep = (lane & 15) == i ? s : keep;
    }
    __builtin_amdgcn_wave_barrier();
    float v[LL][4];
    {
      const Mix r = class_mix<LL>(m, pure, d.simple, a);
      const MixGrad k = mix_grad(d.simple, r, a, keep);
#pragma unroll
      for (int l = 0; l < LL; ++l) {
        v[l][0] = k.gA * pure.u[l] + k.gG[2] * pure.uz[l];
        v[l][1] = k.gB * pure.u[l];
        v[l][2] = k.gG[0] * pure.u[l];
        v[l][3] = k.gG[1] * pure.u[l];
      }
    }
    for (int t = 0; t < K.nsp; t += 4) {
      const int e = t + (lane >> 4);
      const bool in = e < K.nsp;
      const CellShares<LL> S = cell_shares<LL>(d, tab, a, in ? lists[w][kPure + e] : 0);
      const Mix r = class_mix<LL>(m, S, d.simple, a);
      const MixGrad k =
          mix_grad(d.simple, r, a, in ? touched[w][(in ? e : 0) * 16 + (lane & 15)] : 0.0f);
#pragma unroll
      for (int l = 0; l < LL; ++l) {
        if (in) {
          v[l][0] += k.gA * S.u[l] + k.gG[2] * S.uz[l];
          v[l][1] += k.gB * S.u[l];
          v[l][2] += k.gG[0] * S.u[l];
          v[l][3] += k.gG[1] * S.u[l];
        }
        const float fu = row_sum(k.gA * m[l][0] + k.gB * m[l][1] + k.gG[0] * m[l][2] +
                                 k.gG[1] * m[l][3]);
        const float fuz = row_sum(k.gG[2] * m[l][0]);
        if (in && (lane & 15) == 0) {
          acc[w][e][2 * l] += fu;
          acc[w][e][2 * l + 1] += fuz;
        }
      }
    }
#pragma unroll
    for (int l = 0; l < LL; ++l) {
      // Summed over the classes (rows); row r then holds moment qrow.
      const float sum = swap_add16(swap_add32(v[l][0], v[l][1]), swap_add32(v[l][2], v[l][3]));
      if (l < d.ll && (lane & 15) < n) {
        float* o = gst + (((size_t)a * 4 + qrow) * d.ll + l) * np + 16 * g + (lane & 15);
        *o = add ? *o + sum : sum;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (!part) return;
  __syncthreads();
  // Entries shared out over the waves.
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int z = z0 + 64 * c + lane;
    for (int q = w; q < 2 * d.ll; q += kRenderWaves) {
      double t = 0.0;
      if (K.at[c] >= kPure)
        for (int j = 0; j < kRenderWaves; ++j) t += acc[j][K.at[c] - kPure][q];
      if (z < d.zz)
        part[((((size_t)blockIdx.x * 3 + a) * 2 + (q & 1)) * d.ll + (q >> 1)) * d.zz + z] = t;
    }
  }
}

// d clip(v, lo, hi) / dv with torch's (and jax's) halves at ties.
__device__ inline float dclip(float v, float lo, float hi) {
  const float m = fmaxf(v, lo);
  const float a = v > lo ? 1.0f : (v == lo ? 0.5f : 0.0f);
  const float b = m < hi ? 1.0f : (m == hi ? 0.5f : 0.0f);
  return a * b;
}

// Adds the workgroups' parts of k_render_bwd_cells: gus[((a * 2 + w) * ll + l)
// * zz + z] (w = 0: dL/du, 1: dL/duz).  64 entries a workgroup, its 16 waves
// taking every 16th part.
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void k_render_sum_parts(
    int n, int nparts, const double* __restrict__ part, double* __restrict__ gus) {
  __shared__ double red[kSumWaves][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int e = blockIdx.x * 64 + lane;
  double t = 0.0;
  if (e < n)
    for (int j = w; j < nparts; j += kSumWaves) t += part[(size_t)j * n + e];
  red[w][lane] = t;
  __syncthreads();
  if (w == 0 && e < n) {
    for (int j = 1; j < kSumWaves; ++j) t += red[j][lane];
    gus[e] = t;
  }
}

// dL/dpos (ll - 1): interface j is layer j's upper bound and layer j+1's
// lower bound.  One workgroup an interface, its lanes over components and z
// (one lane an interface took 86 us at zz = 128, this 8).
__global__ __launch_bounds__(256) void k_render_bwd_pos(RenderDims d, const float* __restrict__ pos,
                                                        const float* __restrict__ gsa,
                                                        const float* __restrict__ gea,
                                                        const double* __restrict__ gus,
                                                        float* __restrict__ gpos) {
  __shared__ double red[256];
  const int j = blockIdx.x;
  auto sum = [&](int w, int a, int l, int z) {
    return gus[(((size_t)a * 2 + w) * d.ll + l) * d.zz + z];
  };
  double acc = 0.0;
  for (int i = threadIdx.x; i < 3 * d.zz; i += blockDim.x) {
    const int a = i / d.zz, z = i - a * d.zz;
    const int col = a == 2 ? 1 : 0;
    const float gs = gsa[2 * z + col], ge = gea[2 * z + col];
    const float dz = ge - gs, c = (gs + ge) / 2, k = 12.0f / (dz * dz * dz);
    const float dp = dclip(pos[j], gs, ge);
    // layer j: hi = pos[j] -> p1;  layer j + 1: lo = pos[j] -> p0
    const Share s1 = layer_share(d, pos, gsa, gea, j, z, col);
    const Share s0 = layer_share(d, pos, gsa, gea, j + 1, z, col);
    acc += ((sum(0, a, j, z) - sum(0, a, j + 1, z)) / dz +
            (sum(1, a, j, z) * (s1.p1 - c) + sum(1, a, j + 1, z) * (c - s0.p0)) * k) * dp;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) gpos[j] = (float)red[0];
}

// dL/dlayers (ll, SX, SY): each source sub-pixel gathers, for every
// component, the shifted sub-pixels that read it (its own position, m on
// from it, or the first m + 1 along a shifted edge; none for the last m of a
// shifted axis) with their tile's moment cotangents: d mean = 1 / n^2,
// d mean of inverse = -1 / (v^2 n^2), d moments = 12 n w / n^2.
// A workgroup takes 256 sub-pixels of one source row: the row's part of the
// index is uniform and nothing is divided but the 32-bit column.  (One lane
// a sub-pixel over a flat 64-bit index, with a division by v^2 for every
// position read: 98 us for 3 x 1536 x 1536 sub-pixels, this 58.)
__global__ __launch_bounds__(256) void k_render_bwd_layers(RenderDims d, const float* __restrict__ L,
                                                           const float* __restrict__ gst,
                                                           float* __restrict__ gL) {
  const int n = 2 * d.m, SX = n * d.xx, SY = n * d.yy, np = d.xx * d.yy;
  const int nblk = (SY + 255) / 256;
  const int rowid = blockIdx.x / nblk;  // (layer, source row)
  const int l = rowid / SX, si = rowid - l * SX;
  const int sj = (blockIdx.x - rowid * nblk) * 256 + (int)threadIdx.x;
  if (sj >= SY) return;
  const size_t i = ((size_t)l * SX + si) * SY + sj;
  const float v = L[i];
  const float inv = 1.0f / (float)(n * n);
  const float iv2 = 1.0f / (v * v);
  const float k12 = 12.0f * n;
  float acc = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    // shifted positions along x reading source row si
    int i0, i1;
    if (a == 0) {
      i0 = i1 = si;
    } else if (si == 0) {
      i0 = 0;
      i1 = min(d.m, SX - 1);
    } else {
      i0 = i1 = si + d.m;
      if (i0 >= SX) continue;
    }
    int j0, j1;
    if (a == 1) {
      j0 = j1 = sj;
    } else if (sj == 0) {
      j0 = 0;
      j1 = min(d.m, SY - 1);
    } else {
      j0 = j1 = sj + d.m;
      if (j0 >= SY) continue;
    }
    const float* g0 = gst + ((size_t)a * 4 * d.ll + l) * np;
    const size_t q = (size_t)d.ll * np;  // from one moment to the next
    for (int ii = i0; ii <= i1; ++ii) {
      const int x = ii / n, di = ii - x * n;
      const float wx = (di - (d.m - 0.5f)) / (float)(n * n);
      for (int jj = j0; jj <= j1; ++jj) {
        const int y = jj / n, dj = jj - y * n;
        const float wy = (dj - (d.m - 0.5f)) / (float)(n * n);
        const float* p = g0 + (size_t)x * d.yy + y;
        acc += (p[0] - p[q] * iv2 + p[2 * q] * k12 * wx + p[3 * q] * k12 * wy) * inv;
      }
    }
  }
  gL[i] = acc;
}

unsigned blocks_for(long long n, int threads = 256) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace

int render_max_layers() { return kRenderMaxLayers; }

size_t render_stats_floats(int ll, int xx, int yy, int zz) {
  return (size_t)12 * ll * xx * yy + (size_t)4 * ll * zz;
}

// Workgroups per component of the cell kernels: their waves take 16-pixel
// groups, about 1366 waves a component (4 a SIMD over the three components)
// where there are as many groups.
struct CellGrid {
  int blocks, gpw;
};
static CellGrid cell_grid(int xx, int yy) {
  const int groups = (xx * yy + 15) / 16;
  const int gpw = (groups + 4 * 342 - 1) / (4 * 342);
  return {(groups + kRenderWaves * gpw - 1) / (kRenderWaves * gpw), gpw};
}

size_t render_workspace_bytes(int ll, int xx, int yy, int zz) {
  return align256(sizeof(float) * (size_t)12 * ll * xx * yy) +
         align256(sizeof(double) * (size_t)cell_grid(xx, yy).blocks * 6 * ll * zz) +
         align256(sizeof(double) * (size_t)6 * ll * zz);
}

// Calls f(LL, C) with the layers a cell kernel is built for (the fewest that
// hold ll: unused ones have share 0) and its cells a lane.  Up to 4 layers go
// by classes, up to 3 with two cells a lane where zz > 64 (4: LDS); more take
// every cell.
template <typename F>
static void cell_variant(int ll, int zz, F&& f) {
  const bool two = zz > 64;
  auto pick = [&](auto LL) {
    if (two) f(LL, std::integral_constant<int, 2>());
    else f(LL, std::integral_constant<int, 1>());
  };
  if (ll == 1) pick(std::integral_constant<int, 1>());
  else if (ll == 2) pick(std::integral_constant<int, 2>());
  else if (ll == 3) pick(std::integral_constant<int, 3>());
  else if (ll == 4) f(std::integral_constant<int, 4>(), std::integral_constant<int, 1>());
  else if (ll <= 8) f(std::integral_constant<int, 8>(), std::integral_constant<int, 1>());
  else f(std::integral_constant<int, 16>(), std::integral_constant<int, 1>());
}

hipError_t render_forward(int ll, int m, int xx, int yy, int zz, int simple, const float* layers,
                          const float* pos, const float* gs, const float* ge, float* eps,
                          float* stats, hipStream_t s) {
  const RenderDims d{ll, m, xx, yy, zz, simple};
  float* tab = stats + (size_t)12 * ll * xx * yy;
  hipLaunchKernelGGL(k_render_stats, dim3(blocks_for(3LL * ll * xx * yy)), dim3(256), 0, s, d,
                     layers, stats);
  hipLaunchKernelGGL(k_render_shares, dim3(blocks_for(2LL * ll * zz)), dim3(256), 0, s, d, pos,
                     gs, ge, tab);
  const CellGrid G = cell_grid(xx, yy);
  cell_variant(ll, zz, [&](auto LL, auto C) {
    for (int z0 = 0; z0 < zz; z0 += 64 * C.value) {
      if constexpr (LL.value <= kPure)
        hipLaunchKernelGGL((k_render_combine<LL.value, C.value>), dim3(G.blocks, 3),
                           dim3(64 * kRenderWaves), 0, s, d, stats, tab, pos, gs, ge, eps, G.gpw,
                           z0);
      else
        hipLaunchKernelGGL((k_render_combine_cells<LL.value, C.value>), dim3(G.blocks, 3),
                           dim3(64 * kRenderWaves), 0, s, d, stats, tab, eps, G.gpw, z0);
    }
  });
  return hipGetLastError();
}

hipError_t render_backward(int ll, int m, int xx, int yy, int zz, int simple, const float* layers,
                           const float* pos, const float* gs, const float* ge,
                           const float* stats, const float* g_eps, float* g_layers, float* g_pos,
                           char* ws, hipStream_t s) {
  const RenderDims d{ll, m, xx, yy, zz, simple};
  const float* tab = stats + (size_t)12 * ll * xx * yy;
  const CellGrid G = cell_grid(xx, yy);
  float* gst = (float*)ws;
  double* part = (double*)(ws + align256(sizeof(float) * (size_t)12 * ll * xx * yy));
  double* gus = (double*)((char*)part + align256(sizeof(double) * (size_t)G.blocks * 6 * ll * zz));
  const bool want_pos = ll > 1 && g_pos;
  cell_variant(ll, zz, [&](auto LL, auto C) {
    for (int z0 = 0; z0 < zz; z0 += 64 * C.value) {
      double* const parts = want_pos ? part : nullptr;
      if constexpr (LL.value <= kPure)
        hipLaunchKernelGGL((k_render_bwd_cells<LL.value, C.value>), dim3(G.blocks, 3),
                           dim3(64 * kRenderWaves), 0, s, d, stats, tab, pos, gs, ge, g_eps, gst,
                           parts, G.gpw, z0, z0 > 0);
      else
        hipLaunchKernelGGL((k_render_bwd_all_cells<LL.value, C.value>), dim3(G.blocks, 3),
                           dim3(64 * kRenderWaves), 0, s, d, stats, tab, g_eps, gst, parts, G.gpw,
                           z0, z0 > 0);
    }
  });
  // ll SX SY < 2^29 (the arrays' bound of the C ABI); a row takes at least
  // one workgroup.
  const int SX = 2 * m * xx, SY = 2 * m * yy;
  hipLaunchKernelGGL(k_render_bwd_layers, dim3((unsigned)ll * SX * ((SY + 255) / 256)), dim3(256),
                     0, s, d, layers, gst, g_layers);
  if (want_pos) {
    const int n = 6 * ll * zz;
    hipLaunchKernelGGL(k_render_sum_parts, dim3((n + 63) / 64), dim3(64 * kSumWaves), 0, s, n,
                       G.blocks, part, gus);
    hipLaunchKernelGGL(k_render_bwd_pos, dim3(ll - 1), dim3(256), 0, s, d, pos, gs, ge, gus,
                       g_pos);
  }
  return hipGetLastError();
}

}  // namespace pjz
