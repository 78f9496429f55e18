// Parts of the resident steppers (kernels_resident.hip, forward, and
// kernels_adjoint_resident.hip, reverse): the tiling of a domain over the
// compute units and the exchange of edge columns between workgroups.
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>

#include "stream_common.h"
#include "waits.h"

namespace pjz {

// 64-bit exchange words: 4 bytes of payload and the exchange's number, written
// and read with relaxed device-scope atomics.  A word says by itself whether
// it has arrived, so there is no flag, fence or grid barrier: a store and a
// load latency an exchange.
typedef unsigned long long rword_t;

// A value the compiler cannot trace: addresses made from it are computed where
// they are used, not once for all columns before the step loop (which would
// take the registers that the fields need).
__device__ __forceinline__ int opaque_v(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ int opaque_s(int v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return v;
}
// A kernel argument in registers of its own.  Arguments arrive in groups of up
// to 16 registers; where such a group is spilled, each use of one of its values
// reloads all of it (k_resident<2,5,3>: 7200 reloaded registers, apart 700;
// 220x200x96 in slabs, 800 steps: 29.8 -> 26.8 ms).
template <class T>
__device__ __forceinline__ void apart(T& v) {
  if constexpr (std::is_pointer_v<T>) {
    unsigned long long w;
    asm volatile("s_mov_b64 %0, %1" : "=s"(w) : "s"(v));
    // (The compiler knows that an argument points to global memory; of the
    // copy it is told.)
    v = (T)(__attribute__((address_space(1))) std::remove_pointer_t<T>*)w;
  } else {
    T w;
    if constexpr (sizeof(T) == 8) asm volatile("s_mov_b64 %0, %1" : "=s"(w) : "s"(v));
    else asm volatile("s_mov_b32 %0, %1" : "=s"(w) : "s"(v));
    v = w;
  }
}
template <class T, class... Ts>
__device__ __forceinline__ void apart(T& v, Ts&... vs) {
  apart(v);
  apart(vs...);
}
// Pins a result where it is computed: the compiler would otherwise move the
// updates of all columns past the next branch, with their inputs live.
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ float read_lane(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// f(0), .. f(N - 1) with constant arguments (past the size at which the
// compiler unrolls a loop over register arrays).
template <class F, int... K>
__device__ __forceinline__ void static_for_seq(std::integer_sequence<int, K...>, F&& f) {
  (f(std::integral_constant<int, K>()), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(std::make_integer_sequence<int, N>(), f);
}

// Word `off + lane` of a tile's edges (off uniform).
__device__ __forceinline__ rword_t* edge_word(rword_t* base, int off, int lane) {
  return (rword_t*)((char*)(base + opaque_s(off)) + (unsigned)opaque_v(8 * lane));
}

// The value is copied first: paired with the tag in place, every edge value
// would hold a second register for the whole run.
__device__ __forceinline__ void post_edge(rword_t* p, unsigned tag, float v) {
  pin(v);
  __hip_atomic_store(p, ((rword_t)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

template <int CPL>
__device__ __forceinline__ void lds_put(float* p, const float (&v)[CPL]) {
  if constexpr (CPL == 2) *reinterpret_cast<f32x2*>(p) = f32x2{v[0], v[1]};
  else p[0] = v[0];
}
template <int CPL>
__device__ __forceinline__ void lds_get(float (&v)[CPL], const float* p) {
  if constexpr (CPL == 2) {
    const f32x2 t = *reinterpret_cast<const f32x2*>(p);
    v[0] = t.x;
    v[1] = t.y;
  } else {
    v[0] = p[0];
  }
}

// The columns of a wave in the order they are computed: first those that need
// no other wave's edge.  E needs the low neighbours; H, mirrored, the high.
template <int RX, int RY>
struct ColOrder {
  static constexpr int inner = (RX - 1) * (RY - 1);
  static constexpr int x(int k) {
    return k < inner ? 1 + k / (RY > 1 ? RY - 1 : 1) : (k - inner < RX ? k - inner : 0);
  }
  static constexpr int y(int k) {
    return k < inner ? 1 + k % (RY > 1 ? RY - 1 : 1) : (k - inner < RX ? 0 : k - inner - RX + 1);
  }
};

constexpr int kResWaves = 8;  // two waves a SIMD, 256 registers a lane each
constexpr int kResThreads = 64 * kResWaves;
constexpr size_t kResLds = 160 << 10;

// A domain's tiling: kResWaves = WX * WY waves a workgroup, RX x RY columns a
// wave, ntx x nty workgroups, one a compute unit.
struct ResPlan {
  int cpl, rx, ry;  // the kernel's template arguments; rx = 0: not resident
  int wx, wy;
  int ntx, nty;
  bool alias;       // one set of edge buffers for E and H (LDS is short)
  size_t lds;       // bytes
  int tx() const { return rx * wx; }
  int ty() const { return ry * wy; }
  int tiles() const { return ntx * nty; }
  // Words of a tile's edges: E and H, 2 components of tx + ty columns.
  size_t words() const { return (size_t)tiles() * 4 * (tx() + ty()) * 64 * cpl; }
};

// A workgroup's tile as one of its waves sees it: where its columns lie, and
// the passing of edges.  Low edges are those of E (lK in the reverse run),
// which the waves below and to the left read; high edges those of H.  At x
// edges components 1 and 2 are passed, at y edges 0 and 2.
//
// A run may cover a slab of x only: columns [xs, xe), of which it writes (state,
// snapshots, changes of E) its own, [own0, own1).
struct ResTileArgs {
  int X, Y, Z, N, P, lo, hi, NP;
  int xs, xe, own0, own1;
  int wx, wy, ntx, nty, alias;
  rword_t* words;
  WaitArgs waits;
  __device__ __forceinline__ void split() {
    apart(X, Y, Z, N, P, lo, hi, NP, xs, xe, own0, own1, wx, wy, ntx, nty, alias, words,
          waits.ticks, waits.stalled, waits.report);
  }
};

template <int CPL, int RX, int RY>
struct ResTile {
  static constexpr int C = RX * RY;
  static constexpr int ED = 2 * 64 * CPL;  // floats (or words) of an edge column
  // Whether the tile, and in its tile the wave, has a neighbour on a side.  Bits
  // of one register, tested where they are used: as booleans they took a pair of
  // scalar registers each, and what that spilled was reloaded lane by lane.
  enum Place {
    TILE_XLO = 1, TILE_XHI = 2, TILE_YLO = 4, TILE_YHI = 8,
    WAVE_XLO = 16, WAVE_XHI = 32, WAVE_YLO = 64, WAVE_YHI = 128,
    ALIAS = 256  // one set of edge buffers
  };
  __device__ __forceinline__ bool is(int p) const { return (opaque_s(place) & p) != 0; }
  int lane, w, wx, wy, WX, WY, TX, TY, bx, by, xs, xe, own0, own1, x0, y0, zb, X, Y, Z, NP, PS;
  float* lds;
  int er, hr, sx, sy;  // see edges()
  rword_t* mine;
  int ox, oy, oh, fx, fy;
  int place;  // bits of Place

  __device__ __forceinline__ ResTile(const ResTileArgs& a, float* lds_) {
    lane = threadIdx.x & 63;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WX = a.wx;
    WY = a.wy;
    // Quotients of uniform values are computed on the vector unit: back to
    // scalar registers, or all that follows from them takes vector registers.
    wx = __builtin_amdgcn_readfirstlane(w % WX);
    wy = __builtin_amdgcn_readfirstlane(w / WX);
    TX = RX * WX;
    TY = RY * WY;
    X = a.X;
    Y = a.Y;
    Z = a.Z;
    NP = a.NP;
    const int nt = a.ntx * a.nty;
    // Consecutive workgroups go round-robin over the 8 XCDs; neighbouring
    // tiles go to one XCD where the count allows it.
    int tile = blockIdx.x;
    if ((nt & 7) == 0) tile = (tile & 7) * (nt >> 3) + (tile >> 3);
    bx = __builtin_amdgcn_readfirstlane(tile / a.nty);
    by = __builtin_amdgcn_readfirstlane(tile % a.nty);
    xs = a.xs + bx * TX;
    xe = a.xe;
    own0 = a.own0;
    own1 = a.own1;
    x0 = xs + wx * RX;
    y0 = by * TY + wy * RY;
    zb = lane * CPL;
    lds = lds_;
    PS = NP * 4 + 2;
    // A tile's words: low x edge (TY columns), low y (TX), high x, high y.
    // Of the neighbours' (as offsets from this tile's): the low edges from +x
    // and +y, the high ones from -x and -y.
    const size_t tw = (size_t)2 * (TX + TY) * ED;
    mine = a.words + (size_t)tile * tw;
    ox = wy * RY * ED;
    oy = TY * ED + wx * RX * ED;
    oh = (TX + TY) * ED;
    fx = (int)(a.nty * tw);
    fy = (int)tw;
    place = __builtin_amdgcn_readfirstlane(
            (bx > 0 ? TILE_XLO : 0) | (bx + 1 < a.ntx ? TILE_XHI : 0) |
            (by > 0 ? TILE_YLO : 0) | (by + 1 < a.nty ? TILE_YHI : 0) |
            (wx > 0 ? WAVE_XLO : 0) | (wx < WX - 1 ? WAVE_XHI : 0) |
            (wy > 0 ? WAVE_YLO : 0) | (wy < WY - 1 ? WAVE_YHI : 0) | (a.alias ? ALIAS : 0));
  }

  // LDS: psi as (column, pair, PML cell, 2) and, per column, a zero pair for
  // the lanes outside the PML (so every lane's address steps alike); absorber
  // values and in their fourth place, for the wave's first column, the end of
  // its waits; `more` floats of the kernel's own; edge buffers.
  __device__ __forceinline__ f32x4* sig() const {
    return reinterpret_cast<f32x4*>(lds + ((TX * TY * PS + 3) & ~3));
  }
  __device__ __forceinline__ unsigned* waits() const {
    return reinterpret_cast<unsigned*>(lds + opaque_s(((TX * TY * PS + 3) & ~3) + w * C * 4 + 3));
  }
  __device__ __forceinline__ float* own() const {
    return reinterpret_cast<float*>(sig() + TX * TY);
  }
  // Edge slot s of a direction lies between waves s - 1 and s.  Low edges are
  // read from slot w + 1 and written to slot w, high ones read from w and
  // written to w + 1; slots 1 .. WX (low) and 0 .. WX - 1 (high) exist, the
  // outer one holding the neighbouring workgroup's edge.  (Float offsets,
  // uniform: the lane's address is made where it is used.)
  __device__ __forceinline__ void edges(int more) {
    const int eoff = (int)(own() - lds) + more;
    const int hoff = eoff + (is(ALIAS) ? 0 : (WX * TY + WY * TX) * ED);
    sx = (wx * TY + wy * RY) * ED;
    sy = (WX * TY + wy * TX + wx * RX) * ED;
    er = eoff;
    hr = hoff;
  }
  __device__ __forceinline__ float* slot(int off) const { return lds + opaque_s(off) + zb; }
  __device__ __forceinline__ float* low_x() const { return slot(er + sx); }
  __device__ __forceinline__ float* low_y() const { return slot(er + sy); }
  __device__ __forceinline__ float* high_x() const { return slot(hr + sx); }
  __device__ __forceinline__ float* high_y() const { return slot(hr + sy); }

  __device__ __forceinline__ int colx(int i) const { return x0 + i; }
  __device__ __forceinline__ int coly(int r) const { return y0 + r; }
  __device__ __forceinline__ bool valid(int i, int r) const {
    return opaque_s(colx(i)) < xe && opaque_s(coly(r)) < Y;
  }
  __device__ __forceinline__ bool owned(int i, int r) const {
    const int x = opaque_s(colx(i));
    return x >= own0 && x < own1 && opaque_s(coly(r)) < Y;
  }
  __device__ __forceinline__ int offset(int i, int r) const {
    return (opaque_s(colx(i)) * Y + coly(r)) * Z;
  }
  // Column t of the tile's psi and absorber blocks: column t % C of wave t / C.
  __device__ __forceinline__ int tile_x(int t) const {
    return xs + (t / C) % WX * RX + t % C / RY;
  }
  __device__ __forceinline__ int tile_y(int t) const {
    return by * TY + (t / C) / WX * RY + t % C % RY;
  }

  // Three components of a column from arrays N apart.
  __device__ __forceinline__ void load(float (&v)[3][CPL], const float* p, int N, int i,
                                       int r) const {
    const bool ok = valid(i, r);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        v[k][c] = ok && zb + c < Z ? to_global(p)[k * N + offset(i, r) + zb + c] : 0.0f;
  }
  __device__ __forceinline__ void store(float* p, const float (&v)[3][CPL], int N, int i,
                                        int r) const {
    const int o = offset(i, r) + zb;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (zb + c < Z) to_global(p)[k * N + o + c] = v[k][c];
  }
  // A psi block's entry m = lane + 64 j: where it lies in the arrays.
  __device__ __forceinline__ int psi_entry(int m, int P, bool& second) const {
    second = m >= NP * 2;
    return (m & 1) * P + ((m - (second ? NP * 2 : 0)) >> 1);
  }
  // The wave's psi (a pair of arrays P apart each; null: zeros) and the tile's
  // absorber to LDS.  All of a wave's columns are requested at once: entry by
  // entry over the tile, the loads' latencies added up to 40 us a launch.
  __device__ __forceinline__ void fill(const float* psi0, const float* psi1, int P,
                                       const float* mask, const WaitArgs& wa) const {
    for (int j = 0; 64 * j < NP * 4; ++j) {
      const int m = min(lane + 64 * j, NP * 4 - 1);
      bool second;
      const int at = psi_entry(m, P, second);
      const float* const p = second ? psi1 : psi0;
      float v[C];
      static_for<C>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value, i = k / RY, r = k % RY;
        v[k] = psi0 && valid(i, r) ? to_global(p)[at + (opaque_s(colx(i)) * Y + coly(r)) * NP]
                                   : 0.0f;
        // (Bounds the scalar registers that the columns' addresses take.)
        if constexpr (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      });
      static_for<C>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        lds[(w * C + k) * PS + m] = v[k];
      });
    }
    if (lane < 2 * C) lds[(w * C + (lane >> 1)) * PS + NP * 4 + (lane & 1)] = 0.0f;
    const float end = __uint_as_float(wait_end(wa));
    for (int t = threadIdx.x; t < TX * TY; t += kResThreads) {
      const int x = tile_x(t), y = tile_y(t);
      f32x4 s = {0.0f, 0.0f, 0.0f, end};
      if (x < xe && y < Y) {
        const int m = x * Y + y, XY = X * Y;
        s = f32x4{mask[m], mask[XY + m], mask[2 * XY + m], end};
      }
      sig()[t] = s;
    }
  }
  // The wave's own psi back to memory (no barrier: nobody else's).
  __device__ __forceinline__ void store_psi(float* psi0, float* psi1, int P) const {
    for (int j = 0; 64 * j < NP * 4; ++j) {
      const int m = lane + 64 * j;
      if (m >= NP * 4) break;
      bool second;
      const int at = psi_entry(m, P, second);
      float* const p = second ? psi1 : psi0;
      static_for<C>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value, i = k / RY, r = k % RY;
        if (owned(i, r))
          to_global(p)[at + (opaque_s(colx(i)) * Y + coly(r)) * NP] = lds[(w * C + k) * PS + m];
        __builtin_amdgcn_sched_barrier(0);
      });
    }
  }
  // A column's psi pair, from the lane's address in a column's block.
  __device__ __forceinline__ f32x2* psi_at(int lane_bytes, int i, int r) const {
    const int b = lane_bytes + opaque_s((w * C + i * RY + r) * PS * 4);
    return reinterpret_cast<f32x2*>(reinterpret_cast<char*>(lds) + b);
  }

  // A column's two edge values: to LDS, or as words.
  __device__ __forceinline__ void put_edge(float* p, int k, const float (&u)[CPL],
                                           const float (&v)[CPL]) const {
    lds_put<CPL>(p + k * ED, u);
    lds_put<CPL>(p + k * ED + ED / 2, v);
  }
  __device__ __forceinline__ void post(int off, unsigned tag, const float (&u)[CPL],
                                       const float (&v)[CPL]) const {
    rword_t* const q = edge_word(mine, off, lane);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      post_edge(q + 64 * c, tag, u[c]);
      post_edge(q + ED / 2 + 64 * c, tag, v[c]);
    }
  }
  // Passes the wave's edges on: through LDS within the workgroup, as words to
  // its neighbours.
  __device__ __forceinline__ void pass_low(unsigned tag, const float (&e)[RX][RY][3][CPL]) const {
    if (is(WAVE_XLO)) {
#pragma unroll
      for (int r = 0; r < RY; ++r) put_edge(slot(er + sx - TY * ED), r, e[0][r][1], e[0][r][2]);
    } else if (is(TILE_XLO)) {
#pragma unroll
      for (int r = 0; r < RY; ++r) post(ox + r * ED, tag, e[0][r][1], e[0][r][2]);
    }
    if (is(WAVE_YLO)) {
#pragma unroll
      for (int i = 0; i < RX; ++i) put_edge(slot(er + sy - TX * ED), i, e[i][0][0], e[i][0][2]);
    } else if (is(TILE_YLO)) {
#pragma unroll
      for (int i = 0; i < RX; ++i) post(oy + i * ED, tag, e[i][0][0], e[i][0][2]);
    }
  }
  __device__ __forceinline__ void pass_high(unsigned tag, const float (&h)[RX][RY][3][CPL]) const {
    if (is(WAVE_XHI)) {
#pragma unroll
      for (int r = 0; r < RY; ++r)
        put_edge(slot(hr + sx + TY * ED), r, h[RX - 1][r][1], h[RX - 1][r][2]);
    } else if (is(TILE_XHI)) {
#pragma unroll
      for (int r = 0; r < RY; ++r)
        post(oh + ox + r * ED, tag, h[RX - 1][r][1], h[RX - 1][r][2]);
    }
    if (is(WAVE_YHI)) {
#pragma unroll
      for (int i = 0; i < RX; ++i)
        put_edge(slot(hr + sy + TX * ED), i, h[i][RY - 1][0], h[i][RY - 1][2]);
    } else if (is(TILE_YHI)) {
#pragma unroll
      for (int i = 0; i < RX; ++i)
        post(oh + oy + i * ED, tag, h[i][RY - 1][0], h[i][RY - 1][2]);
    }
  }
  __device__ __forceinline__ bool late() const {
    return __builtin_amdgcn_readfirstlane(*waits()) == (int)kLate;
  }
  // Polls until load() returns 0 (the lanes whose words have not come) or the
  // wave's waits end.  The first polls are a loop of their own with one exit,
  // whose count is kept while the loads are on their way: with the clock in the
  // same loop, what follows the last load cost 0.1 us an exchange (64^3: 2.85 us
  // a step instead of 2.62).
  template <class F>
  __device__ __forceinline__ void poll(F&& load) const {
    int left = kWaitPolls;
    unsigned long long missing;
    do {
      --left;
      const unsigned more = ~opaque_s(left >> 31);  // all ones, or 0 at the last
      missing = load() & ((unsigned long long)more << 32 | more);
    } while (missing != 0);
    if (__builtin_expect(left < 0, 0)) {
      while (load() != 0)
        if (wait_over(waits())) break;
    }
  }
  // The words p[0], p[64], .. p[64 (NW - 1)] once all carry `tag`, or what is
  // there when the wave's waits end.
  template <int NW>
  __device__ __forceinline__ void wait_edges(float (&v)[NW], const rword_t* p,
                                             unsigned tag) const {
    rword_t w[NW];
    poll([&]() __attribute__((always_inline)) {
      unsigned other = 0;
#pragma unroll
      for (int k = 0; k < NW; ++k)
        w[k] = __hip_atomic_load(p + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int k = 0; k < NW; ++k) other |= (unsigned)(w[k] >> 32) ^ tag;
      return __ballot(other != 0);
    });
#pragma unroll
    for (int k = 0; k < NW; ++k) v[k] = __uint_as_float((unsigned)w[k]);
  }
  // The same for K columns; columns with no such neighbour are zeros.
  template <int K>
  __device__ __forceinline__ void wait(const int (&at)[K], const int (&dst)[K],
                                       const bool (&there)[K], unsigned tag) const {
    constexpr int NW = 2 * CPL;
    rword_t v[K * NW];
    poll([&]() __attribute__((always_inline)) {
      unsigned other = 0;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const rword_t* const p = edge_word(mine, there[k] ? at[k] : 0, lane);
#pragma unroll
        for (int c = 0; c < NW; ++c)
          v[k * NW + c] =
              __hip_atomic_load(p + 64 * c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < NW; ++c)
          other |= there[k] ? (unsigned)(v[k * NW + c] >> 32) ^ tag : 0;
      return __ballot(other != 0);
    });
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float t[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c)
          t[c] = there[k] ? __uint_as_float((unsigned)v[k * NW + q * CPL + c]) : 0.0f;
        lds_put<CPL>(slot(dst[k]) + q * (ED / 2), t);
      }
  }
  // n columns of a border wave's outer slot: the neighbour's edge, or zeros
  // past the domain.  K columns at a time (the registers of the words).
  template <int n>
  __device__ __forceinline__ void take_own(float* dst, int off, bool there, unsigned tag) const {
    constexpr int K = kCols, NW = 2 * CPL;
#pragma unroll
    for (int k0 = 0; k0 < n; k0 += K) {
      float v[K * NW];
      if (!there) {
#pragma unroll
        for (int q = 0; q < K * NW; ++q) v[q] = 0.0f;
      } else if (k0 + K <= n) {
        wait_edges<K * NW>(v, edge_word(mine, off + k0 * ED, lane), tag);
      } else {
        constexpr int rest = n % K ? n % K : K;
        float u[rest * NW];
        wait_edges<rest * NW>(u, edge_word(mine, off + k0 * ED, lane), tag);
#pragma unroll
        for (int q = 0; q < rest * NW; ++q) v[q] = u[q];
      }
#pragma unroll
      for (int k = 0; k < K && k0 + k < n; ++k)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float t[CPL];
#pragma unroll
          for (int c = 0; c < CPL; ++c) t[c] = v[k * NW + q * CPL + c];
          lds_put<CPL>(dst + (k0 + k) * ED + q * (ED / 2), t);
        }
    }
  }
  // The tile's TY + TX columns shared out over its waves.
  __device__ __forceinline__ void take_shared(int lds_x, int lds_y, int word_x, int word_y,
                                              bool there_x, bool there_y, unsigned tag) const {
    for (int k0 = 0; w + kResWaves * k0 < TX + TY; k0 += kCols) {
      int at[kCols], dst[kCols];
      bool there[kCols];
#pragma unroll
      for (int k = 0; k < kCols; ++k) {
        int q = w + kResWaves * (k0 + k);
        if (q >= TX + TY) q = w + kResWaves * k0;  // (again)
        const bool x = q < TY;
        at[k] = x ? word_x + q * ED : word_y + (q - TY) * ED;
        dst[k] = x ? lds_x + q * ED : lds_y + (q - TY) * ED;
        there[k] = x ? there_x : there_y;
      }
      wait<kCols>(at, dst, there, tag);
    }
  }
  // The neighbouring workgroups' edges into the outer slots (zeros past the
  // domain); after these every edge that the wave's columns need is in LDS.
  // Every poll is a trip to memory in the step's critical path (0.8 us).  Up to
  // 20 cells a lane the border waves wait for their own columns, in one or two
  // polls an edge; beyond, all waves share the tile's columns (150x140x96: 14.3
  // -> 12.6 us a step; 64^3, where one poll is enough, 2.9 with its own
  // columns, 3.6 shared).
  static constexpr int kCols = CPL == 1 ? 4 : 2;  // columns a poll: 16 registers
  static constexpr bool kShared = C * CPL > 20;
  __device__ __forceinline__ void take_low(unsigned tag) const {
    if constexpr (kShared) {
      take_shared(er + (WX - 1) * TY * ED, er + (WX * TY + (WY - 1) * TX) * ED, fx, fy + TY * ED,
                  is(TILE_XHI), is(TILE_YHI), tag);
      lds_barrier();
    } else {
      lds_barrier();
      if (!is(WAVE_XHI)) take_own<RY>(low_x(), fx + ox, is(TILE_XHI), tag);
      if (!is(WAVE_YHI)) take_own<RX>(low_y(), fy + oy, is(TILE_YHI), tag);
    }
  }
  __device__ __forceinline__ void take_high(unsigned tag) const {
    if constexpr (kShared) {
      take_shared(hr, hr + WX * TY * ED, oh - fx, oh - fy + TY * ED, is(TILE_XLO),
                  is(TILE_YLO), tag);
      lds_barrier();
    } else {
      lds_barrier();
      if (!is(WAVE_XLO)) take_own<RY>(high_x(), oh + ox - fx, is(TILE_XLO), tag);
      if (!is(WAVE_YLO)) take_own<RX>(high_y(), oh + oy - fy, is(TILE_YLO), tag);
    }
  }
  // With one set of edge buffers: before it is written again.
  __device__ __forceinline__ void edges_read() const {
    if (is(ALIAS)) lds_barrier();
  }
};

// The waits of a launch of `steps` steps (at most about 20 us each): 60 s, far
// more than other streams' kernels hold a workgroup back, and 1 ms a step.
inline WaitArgs wait_args(const WaitWords& w, int steps) {
  const double ms = w.no_time ? 0.0 : 60e3 + steps;
  return {(unsigned)std::min(ms * (100e3 / kWaitTick), 1e9), w.stalled, w.report};
}

// Workgroups to launch: without the last, a run whose waits have no time (tests)
// waits for words that nobody posts.
inline unsigned launched_tiles(const ResTileArgs& a) {
  const int n = a.ntx * a.nty;
  return a.waits.ticks == 0 && n > 1 ? n - 1 : n;
}

inline ResTileArgs tile_args(const Geom& g, const ResPlan& p, rword_t* words, const WaitArgs& w) {
  ResTileArgs a;
  a.waits = w;
  a.xs = a.own0 = 0;
  a.xe = a.own1 = g.X;
  a.X = g.X; a.Y = g.Y; a.Z = g.Z; a.lo = g.lo; a.hi = g.hi; a.NP = g.NP;
  a.N = (int)g.N;
  a.P = g.X * g.Y * g.NP;
  a.wx = p.wx; a.wy = p.wy; a.ntx = p.ntx; a.nty = p.nty;
  a.alias = p.alias;
  a.words = words;
  return a;
}

// A state in memory: E and H (3N floats each) and the four psi components.
struct ResState {
  float *E, *H, *psi;
};

// Steps [begin, end) in one launch, on columns [xs, xe) of x, of which [own0,
// own1) are written (xe = 0: the whole domain).
struct ResRun {
  int begin, end;
  ResState in, out;   // out.E = null: the last state is not stored
  float* capture;     // E^n - E^(n+1) of each step (or null)
  float* ckpt;        // states before steps begin, begin + every, ... (or null)
  int every;
  unsigned tag0;      // exchange numbers used before (the words start from 0)
  rword_t* words = nullptr;  // null: at L.E1
  int xs = 0, xe = 0, own0 = 0, own1 = 0;
};
// Exchange numbers a run of n steps uses.
inline unsigned resident_tags(int n) { return (unsigned)n + 1; }

// The tiling for a domain on `cus` compute units (rx = 0: it does not fit).
ResPlan resident_plan(const Geom& g, int saxis, int cus);
// What a step of a tiling takes, about, us.
double resident_step_us(const ResPlan& p);

// A domain that does not fit as a whole, in `n` slabs of x run one after the
// other, `steps` at a time: each with that many columns more on its inner
// sides, whose outermost is wrong after one step, the next after two, ...
// (n = 0: none worth it; tile: of the widest slab).
struct SlabPlan {
  ResPlan tile;
  int n, steps;
};
SlabPlan slab_plan(const Geom& g, int saxis, int cus);
// Steps r of a domain in slabs, from buffer set *r.cur to the one it is set
// to; words: slab_words() of them.  After an error the set holds the state
// before step *done (r.begin if untouched).
inline size_t slab_words(const SlabPlan& p) { return p.n > 0 ? p.tile.words() : 0; }
hipError_t run_slabs(const Geom& g, const pjz_fdtd_problem& p, const float* mask, const Src& src,
                     const OutWin& win, char* ws, const Layout& L, const SlabPlan& plan,
                     rword_t* words, const StepRange& r, int* done, hipStream_t s);

// Whether a tiling's kernel that also writes each step's change of E is worth
// its while: past 25 cells a lane, two a column, it spills (the one-step
// change takes 6 more registers a column).
constexpr bool tiling_captures(int cpl, int rx, int ry) {
  return rx > 0 && (cpl == 1 || cpl * rx * ry <= 25);
}
inline bool resident_captures(const ResPlan& p) { return tiling_captures(p.cpl, p.rx, p.ry); }

// The words (at L.E1, cleared before a call's first run) and the state it is
// given in memory are the caller's to prepare.
hipError_t run_resident(const Geom& g, const pjz_fdtd_problem& p, const float* mask,
                        const Src& src, const OutWin& win, char* ws, const Layout& L,
                        const ResPlan& plan, const ResRun& r, hipStream_t s);

// Reversed steps end - 1 down to begin in one launch, from and to adjoint set
// 0: D = E^n - E^(n+1) of the steps from `begin` on, gout the snapshots'
// cotangents.  Uses resident_tags(end - begin) exchange numbers.
bool adjoint_resident_supported(const ResPlan& p);
hipError_t run_adjoint_resident(const Geom& g, const pjz_fdtd_problem& p, const float* mask,
                                char* ws, const Layout& L, const ResPlan& plan, const float* D,
                                const float* gout, int begin, int end, unsigned tag0,
                                hipStream_t s);

}  // namespace pjz
