// Parts of the resident steppers (kernels_resident.hip, forward, and
// kernels_adjoint_resident.hip, reverse): the tiling of a domain over the
// compute units and the exchange of edge columns between workgroups.
#pragma once

#include <type_traits>
#include <utility>

#include "stream_common.h"

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
// Pins a result where it is computed: the compiler would otherwise move the
// updates of all columns past the next branch, with their inputs live.
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }

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

// The words p[0], p[64], .. p[64 (NW - 1)] once all carry `tag`.  A peer posts
// within microseconds, so a wait of seconds means that the words were
// overwritten (two calls that share one workspace): the wave then sets `dead`,
// waits no more and its fields become NaN.
constexpr int kMaxPolls = 1 << 22;

template <int NW>
__device__ __forceinline__ void wait_edges(float (&v)[NW], const rword_t* p, unsigned tag,
                                           bool& dead) {
  rword_t w[NW];
  for (int polls = 0;; ++polls) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < NW; ++k)
      w[k] = __hip_atomic_load(p + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int k = 0; k < NW; ++k) ok &= (unsigned)(w[k] >> 32) == tag;
    if (__all(ok) || dead) break;
    dead = polls >= kMaxPolls;
  }
#pragma unroll
  for (int k = 0; k < NW; ++k) v[k] = __uint_as_float((unsigned)w[k]);
}

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

// A state in memory: E and H (3N floats each) and the four psi components.
struct ResState {
  float *E, *H, *psi;
};

// Steps [begin, end) in one launch.
struct ResRun {
  int begin, end;
  ResState in, out;   // out.E = null: the last state is not stored
  float* capture;     // E^n - E^(n+1) of each step (or null)
  float* ckpt;        // states before steps begin, begin + every, ... (or null)
  int every;
  unsigned tag0;      // exchange numbers used before (the words start from 0)
};
// Exchange numbers a run of n steps uses.
inline unsigned resident_tags(int n) { return (unsigned)n + 1; }

// The tiling for a domain on `cus` compute units (rx = 0: it does not fit).
ResPlan resident_plan(const Geom& g, int saxis, int cus);

// The words (at L.E1, cleared before a call's first run) and the state it is
// given in memory are the caller's to prepare.
hipError_t run_resident(const Geom& g, const pjz_fdtd_problem& p, const float* mask,
                        const Src& src, const OutWin& win, char* ws, const Layout& L,
                        const ResPlan& plan, const ResRun& r, hipStream_t s);

}  // namespace pjz
