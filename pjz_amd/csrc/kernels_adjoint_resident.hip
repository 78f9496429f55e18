// Resident reverse run: all reversed steps of a segment in one launch, the
// adjoint fields in registers (the counterpart of kernels_resident.hip, whose
// tiling and exchange it uses; resident.h).
//
// The two halves of a reverse step (kernels_adjoint.hip gives them cell by
// cell) have the forward step's shape: lH reads lK = cb lE at x+1, y+1, z+1,
// as H reads E there, and lE reads the new lH at x-1, y-1, z-1, as E reads H.
// So lK takes the place of E in the exchange.  lE, lK and lH live in registers
// (9 a cell), up to 12 cells a lane the accumulator G too and up to 8 cells
// cb; D = E^n - E^(n+1), written by the recompute, is read from memory once,
// and beyond those sizes G and cb pass through the caches each step.  Both
// psi cotangents live in LDS.  Snapshot cotangents are added where lE is made.
//
// Bound by the exchange's latency on small domains and by arithmetic on
// larger ones.  The streaming reverse pair it replaces there is bound by
// latency within a workgroup (7 waves, two barriers a level and plane).
// 128x128x64: 6.5 us a reversed step; the gradient of 600 steps, with the
// resident recompute and the streaming reverse 17.4 ms, takes 11.5.
// 160x160x64, 200 steps: 15.2 ms all streaming, 8.2.
#include "resident.h"

namespace pjz {

struct AdjResArgs {
  float* lE;   // in place: state before and after
  float* lH;
  float* lu;   // psi_H cotangent pair (P apart)
  float* lp;   // psi_E cotangent pair
  float* G;
  const float* D;   // D^begin, 3N a step
  const float* cb;
  const float* zt;
  const float* mask;
  const float* gout;  // snapshot cotangents (nn, 3, wex, wey, wez)
  ResTileArgs t;
  float dt;
  int begin, end;  // reversed: end - 1 down to begin
  unsigned tag0;
  int wx0, wy0, wz0, wex, wey, wez, ostart, ostop, ostep;
};

template <int CPL, int RX, int RY>
__global__ __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_adj_resident(AdjResArgs a) {
  using Tile = ResTile<CPL, RX, RY>;
  using Order = ColOrder<RX, RY>;
  constexpr int C = Tile::C, ED = Tile::ED;
  constexpr bool CBR = C * CPL <= 8, GR = C * CPL <= 12;
  // Columns of D (and of G and cb where they are not kept) in flight.
  constexpr int AHEAD = C * CPL <= 12 ? (C < 8 / CPL ? C : 8 / CPL) : 2 / CPL;
  extern __shared__ float lds[];
  Tile T(a.t, lds);
  T.edges(0);
  const int Z = a.t.Z, N = a.t.N, P = a.t.P, NP = a.t.NP;
  const int zb = T.zb;
  const float dt = a.dt;

  float ikE[CPL], ikEp[CPL], bE[CPL], cE[CPL], ikH[CPL], ikHm[CPL], bH[CPL], cH[CPL];
  bool pml[CPL];
  int pH[CPL], pE[CPL], zc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const int z = min(zb + c, Z - 1);
    ikE[c] = a.zt[IKE * Z + z];
    ikEp[c] = zb + c + 1 < Z ? a.zt[IKE * Z + zb + c + 1] : 0.0f;
    bE[c] = a.zt[BE * Z + z];
    cE[c] = a.zt[CE * Z + z];
    ikH[c] = a.zt[IKH * Z + z];
    ikHm[c] = zb + c > 0 ? a.zt[IKH * Z + min(zb + c - 1, Z - 1)] : 0.0f;
    bH[c] = a.zt[BH * Z + z];
    cH[c] = a.zt[CH * Z + z];
    pml[c] = (zb + c < Z) && (zb + c < a.t.lo || zb + c >= Z - a.t.hi);
    const int pidx = zb + c < a.t.lo ? zb + c : zb + c - (Z - a.t.hi) + a.t.lo;
    pH[c] = 4 * (pml[c] ? pidx * 2 : NP * 4);
    pE[c] = 4 * (pml[c] ? NP * 2 + pidx * 2 : NP * 4);
    zc[c] = 4 * z;
  }

  // A column's three components, from inside the domain (what lies outside is
  // dropped at its use).
  auto fetch = [&](float (&v)[3][CPL], const float* base, int i, int r) {
    const int x = min(opaque_s(T.colx(i)), T.X - 1), y = min(T.coly(r), T.Y - 1);
    const char* const p = reinterpret_cast<const char*>(base + (x * T.Y + y) * Z);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        v[k][c] = *to_global(reinterpret_cast<const float*>(p + 4 * (size_t)N * k +
                                                            (unsigned)opaque_v(zc[c])));
  };

  int valid_mask = 0;  // columns (in lE's order) inside the domain
#pragma unroll
  for (int k = 0; k < C; ++k)
    valid_mask |= (T.colx(Order::x(k)) < T.xe && T.coly(Order::y(k)) < T.Y ? 1 : 0) << k;
  auto is_out = [&](int n) {
    return n >= a.ostart && n < a.ostop && (n - a.ostart) % a.ostep == 0;
  };
  // Adds the cotangent of snapshot n to a column.
  auto inject = [&](float (&v)[3][CPL], int n, int i, int r) {
    const int slot = (n - a.ostart) / a.ostep;
    const int x = opaque_s(T.colx(i)) - a.wx0, y = T.coly(r) - a.wy0;
    if (x >= 0 && x < a.wex && y >= 0 && y < a.wey) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        gcfloat* q = to_global(a.gout) +
                     ((((long long)slot * 3 + k) * a.wex + x) * a.wey + y) * (long long)a.wez;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const int z = zb + c - a.wz0;
          if (z >= 0 && z < a.wez) v[k][c] += q[z];
        }
      }
    }
  };

  T.fill(a.lu, a.lp, P, a.mask, a.t.waits);
  __builtin_amdgcn_sched_barrier(0);
  float le[RX][RY][3][CPL], lk[RX][RY][3][CPL], lh[RX][RY][3][CPL];
  float cbr[CBR ? RX : 1][CBR ? RY : 1][3][CPL], gr[GR ? RX : 1][GR ? RY : 1][3][CPL];
#pragma unroll
  for (int i = 0; i < RX; ++i)
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      T.load(le[i][r], a.lE, N, i, r);
      T.load(lh[i][r], a.lH, N, i, r);
      float cb[3][CPL];
      T.load(cb, a.cb, N, i, r);
      if (is_out(a.end - 1)) inject(le[i][r], a.end - 1, i, r);
      if constexpr (GR) T.load(gr[GR ? i : 0][GR ? r : 0], a.G, N, i, r);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          lk[i][r][k][c] = cb[k][c] * le[i][r][k][c];
          if constexpr (CBR) cbr[CBR ? i : 0][CBR ? r : 0][k][c] = cb[k][c];
        }
    }
  __syncthreads();
  T.pass_low(a.tag0 + 1, lk);

  float dq[AHEAD][3][CPL], gq[GR ? 1 : AHEAD][3][CPL], cbq[CBR ? 1 : AHEAD][3][CPL];
  // Column k of a step's D (and G, cb) on its way into its place of the queue.
  auto request = [&](auto kk, const float* D) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    if constexpr (k < C) {
      fetch(dq[k % AHEAD], D, Order::x(k), Order::y(k));
      if constexpr (!GR) fetch(gq[k % AHEAD], a.G, Order::x(k), Order::y(k));
      if constexpr (!CBR) fetch(cbq[k % AHEAD], a.cb, Order::x(k), Order::y(k));
    }
  };

  // lH of the wave's columns.
  auto h_phase = [&](unsigned tag) {
    f32x2 nlu[CPL], nlp[CPL];
    auto load_psi = [&](int i, int r) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        nlu[c] = *T.psi_at(pH[c], i, r);
        nlp[c] = *T.psi_at(pE[c], i, r);
      }
    };
    load_psi(RX - 1 - Order::x(0), RY - 1 - Order::y(0));
    static_for<C>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      if (k == Order::inner) T.take_low(tag);
      constexpr int i = RX - 1 - Order::x(k), r = RY - 1 - Order::y(k);
      f32x2 lu[CPL], lp[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        lu[c] = nlu[c];
        lp[c] = nlp[c];
      }
      float kxp[2][CPL], kyp[2][CPL];  // lK y, z at x + 1; x, z at y + 1
      if (i < RX - 1) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          kxp[0][c] = lk[i + 1 < RX ? i + 1 : 0][r][1][c];
          kxp[1][c] = lk[i + 1 < RX ? i + 1 : 0][r][2][c];
        }
      } else {
        const float* q = T.low_x() + r * ED;
        lds_get<CPL>(kxp[0], q);
        lds_get<CPL>(kxp[1], q + ED / 2);
      }
      if (r < RY - 1) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          kyp[0][c] = lk[i][r + 1 < RY ? r + 1 : 0][0][c];
          kyp[1][c] = lk[i][r + 1 < RY ? r + 1 : 0][2][c];
        }
      } else {
        const float* q = T.low_y() + i * ED;
        lds_get<CPL>(kyp[0], q);
        lds_get<CPL>(kyp[1], q + ED / 2);
      }
      float vx[CPL], vy[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        vx[c] = pml[c] ? cE[c] * (lp[c].x - lk[i][r][0][c]) : 0.0f;
        vy[c] = pml[c] ? cE[c] * (lp[c].y + lk[i][r][1][c]) : 0.0f;
      }
      const float kxn = lane_next(lk[i][r][0][0]), kyn = lane_next(lk[i][r][1][0]);
      const float vxn = lane_next(vx[0]), vyn = lane_next(vy[0]);
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const int cn = c + 1 < CPL ? c + 1 : 0;
        const float kxz = c + 1 < CPL ? lk[i][r][0][cn] : kxn;
        const float kyz = c + 1 < CPL ? lk[i][r][1][cn] : kyn;
        const float vxz = c + 1 < CPL ? vx[cn] : vxn, vyz = c + 1 < CPL ? vy[cn] : vyn;
        const float K0 = lk[i][r][0][c], K1 = lk[i][r][1][c], K2 = lk[i][r][2][c];
        lh[i][r][0][c] = lh[i][r][0][c] - (ikEp[c] * kyz - ikE[c] * K1) + (kyp[1][c] - K2) -
                         (vyz - vy[c]);
        lh[i][r][1][c] = lh[i][r][1][c] + (ikEp[c] * kxz - ikE[c] * K0) - (kxp[1][c] - K2) -
                         (vxz - vx[c]);
        lh[i][r][2][c] = lh[i][r][2][c] - (kyp[0][c] - K0) + (kxp[0][c] - K1);
#pragma unroll
        for (int q = 0; q < 3; ++q) pin(lh[i][r][q][c]);
        const float u0 = pml[c] ? bH[c] * lu[c].x + dt * lh[i][r][0][c] : 0.0f;
        const float u1 = pml[c] ? bH[c] * lu[c].y - dt * lh[i][r][1][c] : 0.0f;
        *T.psi_at(pH[c], i, r) = f32x2{u0, u1};
      }
      __builtin_amdgcn_sched_barrier(0);
      if (k + 1 < C)
        load_psi(RX - 1 - Order::x(k + 1 < C ? k + 1 : 0), RY - 1 - Order::y(k + 1 < C ? k + 1 : 0));
    });
    T.edges_read();
    T.pass_high(tag, lh);
  };

  // lE, lK, G and the psi_E cotangents; `next`: the snapshot that enters before
  // the next reversed step, or -1.
  auto e_phase = [&](const float* D, int next, unsigned tag) {
    const f32x4* const sg0 = T.sig() + T.w * C;
    f32x4 nsg = sg0[Order::x(0) * RY + Order::y(0)];
    f32x2 nlu[CPL], nlp[CPL];
    auto load_psi = [&](int i, int r) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        nlu[c] = *T.psi_at(pH[c], i, r);
        nlp[c] = *T.psi_at(pE[c], i, r);
      }
    };
    load_psi(Order::x(0), Order::y(0));
    static_for<C>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      if (k == Order::inner) T.take_high(tag);
      constexpr int i = Order::x(k), r = Order::y(k);
      const f32x4 sg = nsg;
      f32x2 lu[CPL], lp[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        lu[c] = nlu[c];
        lp[c] = nlp[c];
      }
      const bool ok = (opaque_s(valid_mask) >> k) & 1;
      float cb[3][CPL], d[3][CPL], g[3][CPL];
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const bool in = ok && zb + c < Z;
          cb[q][c] = CBR ? cbr[CBR ? i : 0][CBR ? r : 0][q][c]
                         : in ? cbq[CBR ? 0 : k % AHEAD][q][c] : 0.0f;
          d[q][c] = in ? dq[k % AHEAD][q][c] : 0.0f;
          g[q][c] = GR ? gr[GR ? i : 0][GR ? r : 0][q][c] : gq[GR ? 0 : k % AHEAD][q][c];
        }
      request(std::integral_constant<int, k + AHEAD>(), D);
      float hm[2][CPL], hdn[2][CPL];  // lH y, z at x - 1; x, z at y - 1
      if (i > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          hm[0][c] = lh[i > 0 ? i - 1 : 0][r][1][c];
          hm[1][c] = lh[i > 0 ? i - 1 : 0][r][2][c];
        }
      } else {
        const float* q = T.high_x() + r * ED;
        lds_get<CPL>(hm[0], q);
        lds_get<CPL>(hm[1], q + ED / 2);
      }
      if (r > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          hdn[0][c] = lh[i][r > 0 ? r - 1 : 0][0][c];
          hdn[1][c] = lh[i][r > 0 ? r - 1 : 0][2][c];
        }
      } else {
        const float* q = T.high_y() + i * ED;
        lds_get<CPL>(hdn[0], q);
        lds_get<CPL>(hdn[1], q + ED / 2);
      }
      float ux[CPL], uy[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        ux[c] = pml[c] ? cH[c] * lu[c].x : 0.0f;
        uy[c] = pml[c] ? cH[c] * lu[c].y : 0.0f;
        const float p0 = pml[c] ? bE[c] * (lp[c].x - lk[i][r][0][c]) : 0.0f;
        const float p1 = pml[c] ? bE[c] * (lp[c].y + lk[i][r][1][c]) : 0.0f;
        *T.psi_at(pE[c], i, r) = f32x2{p0, p1};
      }
      __builtin_amdgcn_sched_barrier(0);
      if (k + 1 < C) {
        const int i1 = Order::x(k + 1 < C ? k + 1 : 0), r1 = Order::y(k + 1 < C ? k + 1 : 0);
        load_psi(i1, r1);
        nsg = sg0[i1 * RY + r1];
      }
      const float hxn = lane_prev(lh[i][r][0][CPL - 1]), hyn = lane_prev(lh[i][r][1][CPL - 1]);
      const float uxn = lane_prev(ux[CPL - 1]), uyn = lane_prev(uy[CPL - 1]);
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const int cp = c > 0 ? c - 1 : 0;
        const float hxz = c > 0 ? lh[i][r][0][cp] : hxn, hyz = c > 0 ? lh[i][r][1][cp] : hyn;
        const float uxz = c > 0 ? ux[cp] : uxn, uyz = c > 0 ? uy[cp] : uyn;
        const float hx = lh[i][r][0][c], hy = lh[i][r][1][c], hz = lh[i][r][2][c];
        const float gx = dt * ((ikH[c] * hy - ikHm[c] * hyz) - (hz - hdn[1][c])) - (uy[c] - uyz);
        const float gy = dt * (-(ikH[c] * hx - ikHm[c] * hxz) + (hz - hm[1][c])) - (ux[c] - uxz);
        const float gz = dt * ((hx - hdn[0][c]) - (hy - hm[0][c]));
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          g[q][c] += le[i][r][q][c] * d[q][c];
          if constexpr (GR) {
            gr[GR ? i : 0][GR ? r : 0][q][c] = g[q][c];
            pin(gr[GR ? i : 0][GR ? r : 0][q][c]);
          }
        }
        // Cells past the domain hold lE = 0 and stay so (their lH neighbours
        // inside it are not zero).
        const bool in = ok && zb + c < Z;
        le[i][r][0][c] = in ? (1.0f - sg.x * cb[0][c]) * le[i][r][0][c] + gx : 0.0f;
        le[i][r][1][c] = in ? (1.0f - sg.y * cb[1][c]) * le[i][r][1][c] + gy : 0.0f;
        le[i][r][2][c] = in ? (1.0f - sg.z * cb[2][c]) * le[i][r][2][c] + gz : 0.0f;
      }
      if constexpr (!GR) {
        if (ok) T.store(a.G, g, N, i, r);
      }
      if (next >= 0) inject(le[i][r], next, i, r);
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          pin(le[i][r][q][c]);
          lk[i][r][q][c] = cb[q][c] * le[i][r][q][c];
          pin(lk[i][r][q][c]);
        }
      __builtin_amdgcn_sched_barrier(0);
    });
    T.edges_read();
    T.pass_low(tag + 1, lk);
  };

  for (int n = a.end - 1; n >= a.begin; --n) {
    const unsigned tag = a.tag0 + (unsigned)(a.end - n);
    const float* const D = a.D + (size_t)(n - a.begin) * 3 * N;
    static_for<AHEAD>([&](auto kk) __attribute__((always_inline)) { request(kk, D); });
    h_phase(tag);
    e_phase(D, n > a.begin && is_out(n - 1) ? n - 1 : -1, tag);
  }
#pragma unroll
  for (int i = 0; i < RX; ++i)
#pragma unroll
    for (int r = 0; r < RY; ++r)
      if (T.valid(i, r)) {
        T.store(a.lE, le[i][r], N, i, r);
        T.store(a.lH, lh[i][r], N, i, r);
        if constexpr (GR) T.store(a.G, gr[GR ? i : 0][GR ? r : 0], N, i, r);
      }
  T.store_psi(a.lu, a.lp, P);
  if (T.late()) {
    // A wait in vain: the wave's first column of the gradient is spoiled.
    if (T.valid(0, 0) && zb < Z) to_global(a.G)[T.offset(0, 0) + zb] = __builtin_nanf("");
    tell_late(a.t.waits);
  }
}

// ------------------------------------------------------------------ host side

// Up to 16 cells a lane: 20 spill 53 registers, and the gradient of 190x200x50
// over 200 steps takes 14.5 ms instead of 12.6 with the streaming reverse.
#define PJZ_ADJ_SHAPES(F)                                                              \
  F(1, 2, 1) F(1, 2, 2) F(1, 3, 2) F(1, 4, 2) F(1, 4, 3) F(1, 4, 4)                     \
  F(2, 1, 1) F(2, 2, 1) F(2, 2, 2) F(2, 3, 2) F(2, 4, 2)

template <int CPL, int RX, int RY>
static hipError_t launch_adj_resident(AdjResArgs& a, const ResPlan& p, hipStream_t s) {
  const void* k = reinterpret_cast<const void*>(&k_adj_resident<CPL, RX, RY>);
  hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
  if (e != hipSuccess) return e;
  void* args[] = {&a};
  return hipLaunchCooperativeKernel(k, dim3(launched_tiles(a.t)), dim3(kResThreads), args,
                                    (unsigned)p.lds, s);
}

bool adjoint_resident_supported(const ResPlan& p) {
#define PJZ_ADJ_HAS(c, x, y) if (p.cpl == c && p.rx == x && p.ry == y) return true;
  PJZ_ADJ_SHAPES(PJZ_ADJ_HAS)
#undef PJZ_ADJ_HAS
  return false;
}

hipError_t run_adjoint_resident(const Geom& g, const pjz_fdtd_problem& p, const float* mask,
                                char* ws, const Layout& L, const ResPlan& plan, const float* D,
                                const float* gout, int begin, int end, unsigned tag0,
                                hipStream_t s) {
  if (L.waits.refused()) return hipErrorCooperativeLaunchTooLarge;
  AdjResArgs a;
  a.lE = (float*)(ws + L.lE_[0]);
  a.lH = (float*)(ws + L.lH_[0]);
  a.lu = (float*)(ws + L.lu_[0]);
  a.lp = (float*)(ws + L.lpE_[0]);
  a.G = (float*)(ws + L.accG);
  a.D = D;
  a.cb = (const float*)(ws + L.cb);
  a.zt = (const float*)(ws + L.zt);
  a.mask = mask;
  a.gout = gout;
  a.t = tile_args(g, plan, (rword_t*)(ws + L.E1), wait_args(L.waits, end - begin));
  a.dt = p.dt;
  a.begin = begin;
  a.end = end;
  a.tag0 = tag0;
  a.wx0 = p.x0; a.wy0 = p.y0; a.wz0 = p.z0;
  a.wex = p.ex; a.wey = p.ey; a.wez = p.ez;
  a.ostart = p.out_start; a.ostop = p.out_stop; a.ostep = p.out_step;
#define PJZ_ADJ_LAUNCH(c, x, y) \
  if (plan.cpl == c && plan.rx == x && plan.ry == y) return launch_adj_resident<c, x, y>(a, plan, s);
  PJZ_ADJ_SHAPES(PJZ_ADJ_LAUNCH)
#undef PJZ_ADJ_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace pjz
