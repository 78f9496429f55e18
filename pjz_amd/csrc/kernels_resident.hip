// Resident stepper: a whole run of steps in one launch, the fields in
// registers.
//
// What bounds the streaming steppers on domains of up to a few million cells
// is not bytes: a launch of a 64^3 domain takes 26 us for two steps of 9 MB
// (8-13 planes in sequence, two barriers each, 36-64 workgroups), and a
// 128x128x64 step of 38 MB 15 us.  The chip's registers (128 MB) hold such a
// domain.  Here a workgroup owns a tile of z columns for the whole run: E, H
// (and, up to 16 cells a lane, cb) live in registers, RX x RY columns a wave
// and CPL cells of a column a lane, so x neighbours and most y neighbours are
// other registers of the same lane and z neighbours a DPP move; the CPML psi
// live in LDS.
//
// Edges: after a half step a wave passes its edge columns (the low edges of
// E, the high edges of H) to the next wave through LDS or, at the tile's
// border, to the next workgroup as self-numbered 8-byte words (resident.h).
// The columns that need no neighbour's edge are computed first, while the
// words travel: a step costs the larger of its arithmetic and two exchange
// latencies (about 1 us each).  A word is rewritten only after its reader
// has posted the answer that the writer waits for (E of step n + 1 at an edge
// needs H of step n + 1 there, which the neighbour posts after it read E of
// step n), so one set of words is enough.  All workgroups are on the chip at
// the same time (cooperative launch, one a compute unit) and post before they
// wait for the answer, so every wait ends; where that does not hold, by the
// clock (waits.h).
//
// Measured, us a step, two-step kernel (the default before) against this:
// 64^3 13.4 -> 2.6 (both exchange latencies: a wave waits 0.74 of its cycles),
// 128x128x64 14.3 -> 4.8, 160x160x64 20.4 -> 6.8, 190x200x50 25.1 -> 10.4,
// 150x140x96 29.0 -> 11.4, 301x187x45 45.0 -> 17.0, 180x150x128 37.2 -> 13.8
// (16-30 cells a lane: the instructions of two waves a SIMD, at 301x187x45
// vector ones in 0.53 of a SIMD's cycles and any in 0.98; cb from the caches).
//
// The arithmetic of a cell is that of the two-step kernel (stream2_parts.h),
// in its order of rounding: results equal that kernel's bit for bit.
// Cells past the domain's end in x, y and z have cb = 0 and start from zero,
// so they stay zero and need no bounds checks.
#include <algorithm>

#include "resident.h"

namespace pjz {

struct ResArgs {
  const float* Ein;  // state before step `begin`: E, H (3N each), psi (4P); null: zeros
  const float* Hin;
  const float* psiin;
  float* Eout;       // state after the last step (or null)
  float* Hout;
  float* psiout;
  const float* cb;
  const float* zt;
  const float* mask;
  const float* sfield;
  const float* swave;
  float* out;        // snapshots (or null)
  float* cap;        // E^n - E^(n+1) at cap + (n - begin) * 3N (CAP kernels)
  float* ckpt;       // states before steps begin, begin + every, ... (or null)
  long long ckpt_stride;  // floats
  int every;
  ResTileArgs t;
  int saxis, spos, squad;
  float dt;
  int begin, end;
  unsigned tag0;     // exchange numbers tag0 + 1 .. tag0 + (end - begin) + 1
  int wx0, wy0, wz0, wex, wey, wez, ostart, ostop, ostep;
  __device__ __forceinline__ void split() {
    apart(Ein, Hin, psiin, Eout, Hout, psiout, cb, zt, mask, sfield, swave, out, cap, ckpt,
          ckpt_stride, every, saxis, spos, squad, dt, begin, end, tag0, wx0, wy0, wz0, wex, wey,
          wez, ostart, ostop, ostep);
    t.split();
  }
};

// Registers: 6 a cell for E and H, 3 more for cb where that still fits; past
// it cb (12 of the 60 bytes a streaming step moves a cell) is read from the
// caches each step, two columns ahead.
template <int CPL, int RX, int RY>
constexpr bool res_keeps_cb() { return CPL * RX * RY <= 16; }

template <int CPL, int RX, int RY, bool CAP>
__global__ __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_resident(ResArgs a) {
  a.split();
  using Tile = ResTile<CPL, RX, RY>;
  using Order = ColOrder<RX, RY>;
  constexpr int C = Tile::C, ED = Tile::ED;
  constexpr bool CBR = res_keeps_cb<CPL, RX, RY>();
  extern __shared__ float lds[];
  Tile T(a.t, lds);
  const int X = a.t.X, Y = a.t.Y, Z = a.t.Z, N = a.t.N, P = a.t.P, NP = a.t.NP;
  const int zb = T.zb;
  const float dt = a.dt;
  const int nsrc = a.saxis == 0 ? T.TY * ED : a.saxis == 1 ? T.TX * ED : T.TX * T.TY * 4;
  float* const srcl = T.own();
  T.edges(nsrc);

  // Per-z coefficients and psi addresses.
  float ikE[CPL], bE[CPL], cE[CPL], ikH[CPL], bH[CPL], cH[CPL];
  bool pml[CPL];
  int pH[CPL], pE[CPL];  // bytes from a column's block
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const int z = min(zb + c, Z - 1);
    ikE[c] = a.zt[IKE * Z + z];
    bE[c] = a.zt[BE * Z + z];
    cE[c] = a.zt[CE * Z + z];
    ikH[c] = a.zt[IKH * Z + z];
    bH[c] = a.zt[BH * Z + z];
    cH[c] = a.zt[CH * Z + z];
    pml[c] = (zb + c < Z) && (zb + c < a.t.lo || zb + c >= Z - a.t.hi);
    const int pidx = zb + c < a.t.lo ? zb + c : zb + c - (Z - a.t.hi) + a.t.lo;
    pH[c] = 4 * (pml[c] ? pidx * 2 : NP * 4);
    pE[c] = 4 * (pml[c] ? NP * 2 + pidx * 2 : NP * 4);
  }

  T.fill(a.psiin, a.psiin ? a.psiin + 2 * (size_t)P : nullptr, P, a.mask, a.t.waits);
  __builtin_amdgcn_sched_barrier(0);
  float e[RX][RY][3][CPL], h[RX][RY][3][CPL], cbr[CBR ? RX : 1][CBR ? RY : 1][3][CPL];
#pragma unroll
  for (int i = 0; i < RX; ++i)
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      if (a.Ein) {
        T.load(e[i][r], a.Ein, N, i, r);
        T.load(h[i][r], a.Hin, N, i, r);
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int c = 0; c < CPL; ++c) e[i][r][k][c] = h[i][r][k][c] = 0.0f;
      }
      if constexpr (CBR) T.load(cbr[i][r], a.cb, N, i, r);
    }
  if (a.saxis < 2) {
    // (row or column, component, z): the plane's field.
    const int len = a.saxis == 0 ? Y : X, first = a.saxis == 0 ? T.by * T.TY : T.xs;
    for (int q = threadIdx.x; q < nsrc; q += kResThreads) {
      const int t = q / ED, k = (q / (ED / 2)) & 1, z = q % (ED / 2);
      const int j = first + t;
      srcl[q] = j < len && z < Z ? a.sfield[((size_t)k * len + j) * Z + z] : 0.0f;
    }
  } else {
    for (int q = threadIdx.x; q < nsrc; q += kResThreads) {
      const int t = q >> 2, k = q & 3;
      const int x = T.tile_x(t), y = T.tile_y(t);
      srcl[q] = x < T.xe && y < Y && k < 2 * a.squad ? a.sfield[(size_t)k * X * Y + x * Y + y] : 0.0f;
    }
  }

  __syncthreads();
  T.pass_low(a.tag0 + 1, e);

  // A column's psi pairs (pair 0: H, 1: E), read a column ahead of their use.
  auto psi_at = [&](int c, int pair, int i, int r) {
    return T.psi_at(pair ? pE[c] : pH[c], i, r);
  };
  auto load_psi = [&](f32x2 (&v)[CPL], int pair, int i, int r) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) v[c] = *psi_at(c, pair, i, r);
  };

  // H half step of the wave's columns.
  auto h_phase = [&](unsigned tag) {
    f32x2 nps[CPL];
    load_psi(nps, 0, RX - 1 - Order::x(0), RY - 1 - Order::y(0));
    static_for<C>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      if (k == Order::inner) T.take_low(tag);
      constexpr int i = RX - 1 - Order::x(k), r = RY - 1 - Order::y(k);
      f32x2 ps[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) ps[c] = nps[c];
      float e1[2][CPL], eup[2][CPL];  // Ey, Ez at x + 1; Ex, Ez at y + 1
      if (i < RX - 1) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          e1[0][c] = e[i + 1 < RX ? i + 1 : 0][r][1][c];
          e1[1][c] = e[i + 1 < RX ? i + 1 : 0][r][2][c];
        }
      } else {
        const float* q = T.low_x() + r * ED;
        lds_get<CPL>(e1[0], q);
        lds_get<CPL>(e1[1], q + ED / 2);
      }
      if (r < RY - 1) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          eup[0][c] = e[i][r + 1 < RY ? r + 1 : 0][0][c];
          eup[1][c] = e[i][r + 1 < RY ? r + 1 : 0][2][c];
        }
      } else {
        const float* q = T.low_y() + i * ED;
        lds_get<CPL>(eup[0], q);
        lds_get<CPL>(eup[1], q + ED / 2);
      }
      const float exn = lane_next(e[i][r][0][0]), eyn = lane_next(e[i][r][1][0]);
      float tEy[CPL], tEx[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const float dzEy = (c + 1 < CPL ? e[i][r][1][c + 1 < CPL ? c + 1 : 0] : eyn) - e[i][r][1][c];
        const float dzEx = (c + 1 < CPL ? e[i][r][0][c + 1 < CPL ? c + 1 : 0] : exn) - e[i][r][0][c];
        const float p0 = pml[c] ? bH[c] * ps[c].x + cH[c] * dzEy : 0.0f;
        const float p1 = pml[c] ? bH[c] * ps[c].y + cH[c] * dzEx : 0.0f;
        *psi_at(c, 0, i, r) = f32x2{p0, p1};
        tEy[c] = ikH[c] * dzEy + p0;
        tEx[c] = ikH[c] * dzEx + p1;
      }
      // Here, not before this column's own wait for its psi.
      __builtin_amdgcn_sched_barrier(0);
      if (k + 1 < C)
        load_psi(nps, 0, RX - 1 - Order::x(k + 1 < C ? k + 1 : 0),
                 RY - 1 - Order::y(k + 1 < C ? k + 1 : 0));
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        h[i][r][0][c] = h[i][r][0][c] - dt * ((eup[1][c] - e[i][r][2][c]) - tEy[c]);
        h[i][r][1][c] = h[i][r][1][c] - dt * (tEx[c] - (e1[1][c] - e[i][r][2][c]));
        h[i][r][2][c] = h[i][r][2][c] -
                        dt * ((e1[0][c] - e[i][r][1][c]) - (eup[0][c] - e[i][r][0][c]));
#pragma unroll
        for (int q = 0; q < 3; ++q) pin(h[i][r][q][c]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    T.edges_read();
    T.pass_high(tag, h);
  };

  // cb of a column from memory, from inside the domain (the selects that make
  // it zero outside stand at its use: here they would wait for the loads).  A
  // lane's two cells come in one load; past the end of an odd row it reads the
  // next row's first cell or, at the end of cb, the psi that follow it.
  const int zc = 4 * min(zb, Z - 1);
  auto load_cb = [&](float (&v)[3][CPL], int i, int r) {
    const int x = min(opaque_s(T.colx(i)), X - 1), y = min(T.coly(r), Y - 1);
    const char* const p = reinterpret_cast<const char*>(a.cb + (x * Y + y) * Z);
    const unsigned at = (unsigned)opaque_v(zc);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      gcfloat* const q = to_global(reinterpret_cast<const float*>(p + 4 * (size_t)N * k + at));
#pragma unroll
      for (int c = 0; c < CPL; ++c) v[k][c] = q[c];
    }
  };

  // Of the columns in E's order: those inside the domain, those with a source.
  int valid_mask = 0, src_mask = 0;
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const int x = T.colx(Order::x(k)), y = T.coly(Order::y(k)), at = a.saxis == 0 ? x : y;
    valid_mask |= (x < T.xe && y < Y ? 1 : 0) << k;
    src_mask |= (a.saxis == 2 || at == a.spos || at == a.spos - 1 ? 1 : 0) << k;
  }

  // E half step.
  auto e_phase = [&](int n, unsigned tag, float w0, float w1) {
    // Columns of cb in flight, by the registers that are left.
    constexpr int AHEAD = C * CPL <= 20 ? 6 / CPL : C * CPL <= 25 ? 4 / CPL : C * CPL <= 30 ? 2 : 1;
    float cbq[AHEAD][3][CPL];
    f32x2 nps[CPL];
    const f32x4* const sg0 = T.sig() + T.w * C;
    f32x4 nsg = sg0[Order::x(0) * RY + Order::y(0)];
    load_psi(nps, 1, Order::x(0), Order::y(0));
    // A z-plane source: J of every column of the wave, column t on lane t (read
    // in the columns themselves, each would wait for LDS).
    float jxs = 0.0f, jys = 0.0f;
    if (a.saxis == 2) {
      const f32x4 s = reinterpret_cast<const f32x4*>(srcl)[T.w * C + min(T.lane, C - 1)];
      jxs = s.x * w0;
      jys = s.y * w0;
      if (a.squad > 1) {
        jxs += s.z * w1;
        jys += s.w * w1;
      }
    }
    if constexpr (!CBR) {
#pragma unroll
      for (int k = 0; k < AHEAD && k < C; ++k) load_cb(cbq[k], Order::x(k), Order::y(k));
    }
    static_for<C>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      if (k == Order::inner) T.take_high(tag);
      constexpr int i = Order::x(k), r = Order::y(k);
      const f32x4 sg = nsg;
      f32x2 ps[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) ps[c] = nps[c];
      float cb[3][CPL];
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
          cb[q][c] = CBR ? cbr[CBR ? i : 0][CBR ? r : 0][q][c]
                         : ((opaque_s(valid_mask) >> k) & 1) && zb + c < Z ? cbq[k % AHEAD][q][c]
                                                                           : 0.0f;
      if constexpr (!CBR) {
        if (k + AHEAD < C)
          load_cb(cbq[k % AHEAD], Order::x(k + AHEAD < C ? k + AHEAD : 0),
                  Order::y(k + AHEAD < C ? k + AHEAD : 0));
      }
      float hm[2][CPL], hdn[2][CPL];  // Hy, Hz at x - 1; Hx, Hz at y - 1
      if (i > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          hm[0][c] = h[i > 0 ? i - 1 : 0][r][1][c];
          hm[1][c] = h[i > 0 ? i - 1 : 0][r][2][c];
        }
      } else {
        const float* q = T.high_x() + r * ED;
        lds_get<CPL>(hm[0], q);
        lds_get<CPL>(hm[1], q + ED / 2);
      }
      if (r > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          hdn[0][c] = h[i][r > 0 ? r - 1 : 0][0][c];
          hdn[1][c] = h[i][r > 0 ? r - 1 : 0][2][c];
        }
      } else {
        const float* q = T.high_y() + i * ED;
        lds_get<CPL>(hdn[0], q);
        lds_get<CPL>(hdn[1], q + ED / 2);
      }
      const float hxn = lane_prev(h[i][r][0][CPL - 1]), hyn = lane_prev(h[i][r][1][CPL - 1]);
      float cx[CPL], cy[CPL], cz[CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const float dzHy = h[i][r][1][c] - (c > 0 ? h[i][r][1][c > 0 ? c - 1 : 0] : hyn);
        const float dzHx = h[i][r][0][c] - (c > 0 ? h[i][r][0][c > 0 ? c - 1 : 0] : hxn);
        const float p0 = pml[c] ? bE[c] * ps[c].x + cE[c] * dzHy : 0.0f;
        const float p1 = pml[c] ? bE[c] * ps[c].y + cE[c] * dzHx : 0.0f;
        *psi_at(c, 1, i, r) = f32x2{p0, p1};
        const float tHy = ikE[c] * dzHy + p0;
        const float tHx = ikE[c] * dzHx + p1;
        cx[c] = (h[i][r][2][c] - hdn[1][c]) - tHy;
        cy[c] = tHx - (h[i][r][2][c] - hm[1][c]);
        cz[c] = (h[i][r][1][c] - hm[0][c]) - (h[i][r][0][c] - hdn[0][c]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (k + 1 < C) {
        const int i1 = Order::x(k + 1 < C ? k + 1 : 0), r1 = Order::y(k + 1 < C ? k + 1 : 0);
        load_psi(nps, 1, i1, r1);
        nsg = sg0[i1 * RY + r1];
      }
      // J as in add_source2: two components, to the axes that they belong to.
      if ((opaque_s(src_mask) >> k) & 1) {
        float ju[CPL], jv[CPL];
        if (a.saxis < 2) {
          const float wv = (a.saxis == 0 ? T.colx(i) : T.coly(r)) == a.spos ? w0 : w1;
          const float* s = srcl + opaque_s((a.saxis == 0 ? T.wy * RY + r : T.wx * RX + i) * ED) + zb;
#pragma unroll
          for (int c = 0; c < CPL; ++c) {
            ju[c] = s[c] * wv;
            jv[c] = s[ED / 2 + c] * wv;
          }
        } else {
          const float jx = read_lane(jxs, i * RY + r), jy = read_lane(jys, i * RY + r);
#pragma unroll
          for (int c = 0; c < CPL; ++c) {
            ju[c] = zb + c == a.spos ? jx : 0.0f;
            jv[c] = zb + c == a.spos ? jy : 0.0f;
          }
        }
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          cx[c] += a.saxis == 0 ? 0.0f : ju[c];
          cy[c] += a.saxis == 0 ? ju[c] : (a.saxis == 1 ? 0.0f : jv[c]);
          cz[c] += a.saxis == 2 ? 0.0f : jv[c];
        }
      }
      float d[3][CPL];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const float o0 = e[i][r][0][c], o1 = e[i][r][1][c], o2 = e[i][r][2][c];
        // The streaming kernels' rounding: cb K rounded, then one fma.
        e[i][r][0][c] = __builtin_fmaf(o0, 1.0f - sg.x * cb[0][c], cb[0][c] * cx[c]);
        e[i][r][1][c] = __builtin_fmaf(o1, 1.0f - sg.y * cb[1][c], cb[1][c] * cy[c]);
        e[i][r][2][c] = __builtin_fmaf(o2, 1.0f - sg.z * cb[2][c], cb[2][c] * cz[c]);
#pragma unroll
        for (int q = 0; q < 3; ++q) pin(e[i][r][q][c]);
        if constexpr (CAP) {
          d[0][c] = o0 - e[i][r][0][c];
          d[1][c] = o1 - e[i][r][1][c];
          d[2][c] = o2 - e[i][r][2][c];
        }
      }
      if constexpr (CAP) {
        if (T.owned(i, r)) {
          gfloat* q = to_global(a.cap) + (size_t)(n - a.begin) * 3 * N + T.offset(i, r) + zb;
#pragma unroll
          for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int c = 0; c < CPL; ++c)
              if (zb + c < Z) __builtin_nontemporal_store(d[m][c], q + m * N + c);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    T.edges_read();
    T.pass_low(tag + 1, e);
  };

  // The state in registers and LDS to E, H (3N each) and psi (4P).
  auto store_state = [&](float* E, float* H, float* ps) {
#pragma unroll
    for (int i = 0; i < RX; ++i)
#pragma unroll
      for (int r = 0; r < RY; ++r)
        if (T.owned(i, r)) {
          T.store(E, e[i][r], N, i, r);
          T.store(H, h[i][r], N, i, r);
        }
    T.store_psi(ps, ps + 2 * (size_t)P, P);
  };

  float w0 = uniform_load(a.swave, 2 * a.begin), w1 = uniform_load(a.swave, 2 * a.begin + 1);
  int to_ckpt = a.ckpt ? 0 : -1;
  for (int n = a.begin; n < a.end; ++n) {
    const unsigned tag = a.tag0 + 1 + (n - a.begin);
    if (to_ckpt == 0) {
      float* q = a.ckpt + (long long)((n - a.begin) / a.every) * a.ckpt_stride;
      store_state(q, q + 3 * (size_t)N, q + 6 * (size_t)N);
      to_ckpt = a.every;
    }
    --to_ckpt;
    h_phase(tag);
    const int m = min(n + 1, a.end - 1);  // the next step's waveform row
    const float u0 = uniform_load(a.swave, 2 * m), u1 = uniform_load(a.swave, 2 * m + 1);
    e_phase(n, tag, w0, w1);
    w0 = u0;
    w1 = u1;
    // Never taken (every >= 0).  Without a write the compiler cannot rule out
    // here, the capturing kernels keep both versions of a step's fields live:
    // 157 spilled registers instead of 13 at 30 cells a lane.
    if constexpr (CAP) {
      if (__builtin_expect(a.every < 0, 0))
        e[0][0][0][0] = e[0][0][1][0] = e[0][0][2][0] = 0.0f;
    }
    if (a.out && n >= a.ostart && n < a.ostop && (n - a.ostart) % a.ostep == 0) {
      const int slot = (n - a.ostart) / a.ostep;
#pragma unroll
      for (int i = 0; i < RX; ++i)
#pragma unroll
        for (int r = 0; r < RY; ++r) {
          const int x = opaque_s(T.colx(i)) - a.wx0, y = T.coly(r) - a.wy0;
          if (x >= 0 && x < a.wex && y >= 0 && y < a.wey && T.owned(i, r)) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              gfloat* q = to_global(a.out) +
                          ((((long long)slot * 3 + k) * a.wex + x) * a.wey + y) * (long long)a.wez;
#pragma unroll
              for (int c = 0; c < CPL; ++c) {
                const int z = zb + c - a.wz0;
                if (z >= 0 && z < a.wez) q[z] = e[i][r][k][c];
              }
            }
          }
        }
    }
  }
  if (a.Eout) store_state(a.Eout, a.Hout, a.psiout);
  if (T.late()) {
    // A wait in vain: the wave's first column of what it wrote is spoiled.
    const float nan = __builtin_nanf("");
    if (T.owned(0, 0) && zb < Z) {
      const int o = T.offset(0, 0) + zb;
      if (a.Eout) to_global(a.Eout)[o] = nan;
      if (CAP) to_global(a.cap)[o] = nan;
      const int x = T.colx(0) - a.wx0, y = T.coly(0) - a.wy0, z = zb - a.wz0;
      if (a.out && x >= 0 && x < a.wex && y >= 0 && y < a.wey && z >= 0 && z < a.wez)
        for (int n = max(a.begin, a.ostart); n < min(a.end, a.ostop); ++n)
          if ((n - a.ostart) % a.ostep == 0)
            to_global(a.out)[((((long long)((n - a.ostart) / a.ostep) * 3) * a.wex + x) * a.wey +
                              y) * (long long)a.wez + z] = nan;
    }
    tell_late(a.t.waits);
  }
}

// ------------------------------------------------------------------ host side

namespace {

// The kernels: columns a wave.
struct ResShape {
  int cpl, rx, ry;
};
#define PJZ_RES_SHAPES(F)                                                                   \
  F(1, 2, 1) F(1, 2, 2) F(1, 3, 2) F(1, 4, 2) F(1, 4, 3) F(1, 4, 4) F(1, 5, 4) F(1, 5, 5)   \
  F(1, 6, 5) F(1, 8, 4)                                                                     \
  F(2, 1, 1) F(2, 2, 1) F(2, 2, 2) F(2, 3, 2) F(2, 4, 2) F(2, 5, 2) F(2, 4, 3) F(2, 5, 3)   \
  F(2, 4, 4)
constexpr ResShape kShapes[] = {
#define PJZ_RES_ROW(c, x, y) {c, x, y},
    PJZ_RES_SHAPES(PJZ_RES_ROW)
#undef PJZ_RES_ROW
};

size_t res_lds(const Geom& g, int saxis, int cpl, int tx, int ty, int wx, int wy, bool alias) {
  const size_t ed = 2 * 64 * cpl;
  const size_t nsrc = saxis == 0 ? ty * ed : saxis == 1 ? tx * ed : (size_t)tx * ty * 4;
  const size_t edge = (size_t)(wx * ty + wy * tx) * ed;
  const size_t psi = ((size_t)tx * ty * (g.NP * 4 + 2) + 3) & ~(size_t)3;
  return sizeof(float) * (psi + (size_t)tx * ty * 4 + nsrc + edge * (alias ? 1 : 2));
}

}  // namespace

// The best tiling of X x Y columns whose words take at most `room` bytes.
static ResPlan best_tiling(const Geom& g, int X, int saxis, int cus, size_t room) {
  ResPlan best{};
  if (g.Z > 128) return best;
  const int cpl = g.Z <= 64 ? 1 : 2;
  // Cost of a step: the columns a wave computes, one after the other.
  int cost = 0;
  for (const ResShape& s : kShapes) {
    if (s.cpl != cpl) continue;
    for (int wx = 1; wx <= kResWaves; wx *= 2) {
      ResPlan p{s.cpl, s.rx, s.ry, wx, kResWaves / wx, 0, 0, false, 0};
      p.ntx = (X + p.tx() - 1) / p.tx();
      p.nty = (g.Y + p.ty() - 1) / p.ty();
      if ((long long)p.ntx * p.nty > cus) continue;
      p.lds = res_lds(g, saxis, cpl, p.tx(), p.ty(), p.wx, p.wy, false);
      if (p.lds > kResLds) {
        p.alias = true;
        p.lds = res_lds(g, saxis, cpl, p.tx(), p.ty(), p.wx, p.wy, true);
        if (p.lds > kResLds) continue;
      }
      // More than half of a compute unit's LDS: one workgroup each.
      p.lds = std::max(p.lds, kResLds / 2 + 1024);
      if (p.words() * sizeof(rword_t) > room) continue;
      const int c = 64 * s.rx * s.ry + 2 * (s.rx + s.ry) + (p.alias ? 8 : 0) + p.tx() + p.ty();
      if (!best.rx || c < cost) {
        best = p;
        cost = c;
      }
    }
  }
  return best;
}

ResPlan resident_plan(const Geom& g, int saxis, int cus) {
  // The words take the place of the second set of E and H.
  return best_tiling(g, g.X, saxis, cus, 2 * align256(sizeof(float) * 3 * (size_t)g.N));
}

// By the tiling's cells a lane, from the measurements at the head of this file
// (tilings of two cells a lane past 25 were slower when it was fitted: 16.8 at
// 30 cells, now 13.8): past 16 cells cb comes from memory, two cells a lane past
// 30 spill.
double resident_step_us(const ResPlan& p) {
  const int c = p.cpl * p.rx * p.ry;
  return c <= 16 ? 2.5 + 0.3 * c : p.cpl == 2 && c > 30 ? 21.0 : 1.0 + 0.53 * c;
}

// Slabs cost their ghost columns, and every `steps` steps a launch each (35 us
// with the start of its waves) and one pass over the state.  Taken where that
// is estimated below 0.85 of the streaming steppers' rate, measured as 80-90
// cells/ns at zz = 96, 94-113 at 128 and 110 at 64 (by the lanes in
// use).  Measured, us a step: 220x200x96 48.9 -> 32.8, 260x196x96 55.0 -> 34.0,
// 300x300x64 52.2 -> 29.6, 256x341x64 52.0 -> 33.6, 128x341x128 59.2 -> 39.0,
// 512x512x64 148 -> 110; 256x256x128 in three slabs 75.7 against 74.5 (before
// kernel arguments had registers of their own), which this estimate leaves
// alone.
SlabPlan slab_plan(const Geom& g, int saxis, int cus) {
  SlabPlan best{};
  if (g.Z > 128) return best;
  const double cells = (double)g.N;
  double cost = 0.85 * cells / (g.Z <= 64 ? 110e3 / 64 * g.Z : 0.85e3 * g.Z);
  const double pass = cells * (60.0 + 32.0 * g.NP / g.Z) / 4.5e6;  // us
  for (int n = 2; n <= 6; ++n) {
    const int own = (g.X + n - 1) / n;
    for (int k = 6; k <= 20; k += 2) {
      if (own < 2 * k) break;
      // The widest slab: an inner one where there are any.
      const ResPlan t = best_tiling(g, own + (n > 2 ? 2 : 1) * k, saxis, cus, (size_t)1 << 30);
      if (!t.rx) break;
      const double c = n * resident_step_us(t) + (n * 35.0 + pass) / k;
      if (c < cost) {
        cost = c;
        best = {t, n, k};
      }
    }
  }
  return best;
}

hipError_t run_slabs(const Geom& g, const pjz_fdtd_problem& p, const float* mask, const Src& src,
                     const OutWin& win, char* ws, const Layout& L, const SlabPlan& plan,
                     rword_t* words, const StepRange& r, int* done, hipStream_t s) {
  hipError_t e = launch_zero((float*)words, slab_words(plan) * 2, s);
  float* psi = (float*)(ws + L.psi);
  const size_t P4 = (size_t)PSI_SET * g.X * g.Y * g.NP;
  auto state = [&](int set) {
    return ResState{(float*)(ws + (set ? L.E1 : L.E0)), (float*)(ws + (set ? L.H1 : L.H0)),
                    psi + set * P4};
  };
  const int own = (g.X + plan.n - 1) / plan.n;
  unsigned tags = 0;
  for (int b = r.begin; b < r.end && e == hipSuccess; b += plan.steps) {
    const int end = std::min(b + plan.steps, r.end);
    for (int i = 0; i < plan.n && e == hipSuccess; ++i) {
      ResRun q{b, end, state(*r.cur), state(1 - *r.cur), nullptr, nullptr, 1, tags};
      if (r.capture) q.capture = r.capture + (size_t)(b - r.begin) * 3 * g.N;
      q.words = words;
      q.own0 = i * own;
      q.own1 = std::min(q.own0 + own, g.X);
      q.xs = std::max(q.own0 - plan.steps, 0);
      q.xe = std::min(q.own1 + plan.steps, g.X);
      if (q.own0 >= q.own1) continue;
      tags += resident_tags(end - b);
      // The tiling of the widest slab, as many of its tiles as this one takes.
      ResPlan t = plan.tile;
      t.ntx = (q.xe - q.xs + t.tx() - 1) / t.tx();
      e = run_resident(g, p, mask, src, win, ws, L, t, q, s);
    }
    if (e != hipSuccess) break;
    *r.cur = 1 - *r.cur;
    *done = end;
  }
  return e;
}

template <int CPL, int RX, int RY, bool CAP>
static hipError_t launch_resident(ResArgs& a, const ResPlan& p, hipStream_t s) {
  const void* k = reinterpret_cast<const void*>(&k_resident<CPL, RX, RY, CAP>);
  hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
  if (e != hipSuccess) return e;
  void* args[] = {&a};
  return hipLaunchCooperativeKernel(k, dim3(launched_tiles(a.t)), dim3(kResThreads), args,
                                    (unsigned)p.lds, s);
}

hipError_t run_resident(const Geom& g, const pjz_fdtd_problem& p, const float* mask,
                        const Src& src, const OutWin& win, char* ws, const Layout& L,
                        const ResPlan& plan, const ResRun& r, hipStream_t s) {
  if (L.waits.refused()) return hipErrorCooperativeLaunchTooLarge;
  ResArgs a;
  a.Ein = r.in.E;
  a.Hin = r.in.H;
  a.psiin = r.in.psi;
  a.Eout = r.out.E;
  a.Hout = r.out.H;
  a.psiout = r.out.psi;
  a.cb = (const float*)(ws + L.cb);
  a.zt = (const float*)(ws + L.zt);
  a.mask = mask;
  a.sfield = src.field;
  a.swave = src.wave;
  a.out = win.out;
  a.cap = r.capture;
  a.ckpt = r.ckpt;
  a.ckpt_stride = (long long)(ckpt_stride(L) / sizeof(float));
  a.every = r.every;
  a.t = tile_args(g, plan, r.words ? r.words : (rword_t*)(ws + L.E1),
                  wait_args(L.waits, r.end - r.begin));
  if (r.xe > 0) {
    a.t.xs = r.xs;
    a.t.xe = r.xe;
    a.t.own0 = r.own0;
    a.t.own1 = r.own1;
  }
  a.saxis = src.axis; a.spos = src.pos; a.squad = src.quad;
  a.dt = p.dt;
  a.begin = r.begin;
  a.end = r.end;
  a.tag0 = r.tag0;
  a.wx0 = win.x0; a.wy0 = win.y0; a.wz0 = win.z0;
  a.wex = win.ex; a.wey = win.ey; a.wez = win.ez;
  a.ostart = p.out_start; a.ostop = p.out_stop; a.ostep = p.out_step;
#define PJZ_RES_LAUNCH(c, x, y)                                               \
  if (plan.cpl == c && plan.rx == x && plan.ry == y) {                        \
    if (!r.capture) return launch_resident<c, x, y, false>(a, plan, s);       \
    if constexpr (tiling_captures(c, x, y))                                   \
      return launch_resident<c, x, y, true>(a, plan, s);                      \
  }
  PJZ_RES_SHAPES(PJZ_RES_LAUNCH)
#undef PJZ_RES_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace pjz
