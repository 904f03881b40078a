// Device and host pieces shared by the temporally blocked 2D tile kernels
// (forward: tiled2d.hip; reverse: reverse2d.hip): the tile's LDS region and
// thread mapping, the checked quotients by dx, tile enumeration and row
// profiles.
#pragma once
#include <algorithm>

#include "common.h"
#include "tiled2d.h"

namespace mt {
namespace {

template <typename T>
__device__ __forceinline__ T dget(const T* p, long long idx, bool ok) {
  return ok ? p[idx] : T(0);
}

// LDS region of a TX x TY x NS tile and its thread mapping for at most MAXB
// threads: PER rows per thread, ROWS rows per pass, BLK threads.
template <int TX, int TY, int NS, int MAXB>
struct Shape {
  static constexpr int RX = TX + 2 * NS + 1, RY = TY + 2 * NS + 1, RC = RX * RY;
  static constexpr int PASSES = (RX + MAXB / RY - 1) / (MAXB / RY);
  static constexpr int ROWS = (RX + PASSES - 1) / PASSES;
  static constexpr int PER = (RX + ROWS - 1) / ROWS;
  static constexpr int STR = ROWS * RY;
  static constexpr int BLK = (STR + 63) / 64 * 64;
  static_assert(MAXB >= RY && BLK <= 1024, "tile rows must fit a workgroup");
};

// Quotients ax(u) / dx and ay(u) / dx of one half-step, checked together:
// each takes div_c's fast sequence and records its dividend's exponent; a
// lane for which some dividend falls outside the verified range (or a
// divisor without a verified reciprocal, rdx = 0) redoes its quotients with
// IEEE division, from dividends formed again (the LDS values they read do not
// change within a half-step).  FP64 always divides.
template <typename T, int PER, typename FX, typename FY>
__device__ __forceinline__ void step_quots(T dx, T rdx, FX ax, FY ay, T (&qx)[PER], T (&qy)[PER]) {
  if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int u = 0; u < PER; ++u) qx[u] = ax(u) / dx, qy[u] = ay(u) / dx;
  } else {
    unsigned worst = rdx == T(0) ? ~0u : 0u;
    auto q = [&](T a) -> T {
      const T q0 = a * rdx;
      const T r = fma(-q0, dx, a);
      worst = max(worst, (unsigned)(__builtin_amdgcn_frexp_expf(a) + 99));
      return copysign(fma(r, rdx, q0), a);
    };
#pragma unroll
    for (int u = 0; u < PER; ++u) qx[u] = q(ax(u)), qy[u] = q(ay(u));
    if (worst > 200u) {
      __asm__ volatile("");  // a real branch: keeps the divisions off the common path
#pragma unroll
      for (int u = 0; u < PER; ++u) qx[u] = ax(u) / dx, qy[u] = ay(u) / dx;
    }
  }
}

// Tile (tr, tc) for linear index b of the interior rectangle or of the ring.
__device__ __forceinline__ void tile_linear(bool pml, const TileMap& m, int b, int* tr, int* tc) {
  if (!pml) {
    int w = m.c1 - m.c0;
    *tr = m.r0 + b / w;
    *tc = m.c0 + b % w;
    return;
  }
  if (b < m.r0 * m.C) {
    *tr = b / m.C;
    *tc = b % m.C;
    return;
  }
  b -= m.r0 * m.C;
  if (b < (m.R - m.r1) * m.C) {
    *tr = m.r1 + b / m.C;
    *tc = b % m.C;
    return;
  }
  b -= (m.R - m.r1) * m.C;
  int per = m.c0 + (m.C - m.c1);
  *tr = m.r0 + b / per;
  int k = b % per;
  *tc = k < m.c0 ? k : m.c1 + (k - m.c0);
}

// Row profiles of the region in LDS: (b, a) of the two x-axis profiles, for
// rows inside the shells (other entries are never read).
template <typename T, int RX>
__device__ __forceinline__ void load_rows(const Pml<T>& h, const Pml<T>& e, int a0, int nh, int ne, T* prof) {
  for (int li = threadIdx.x; li < RX; li += blockDim.x) {
    const int i = a0 + li;
    if (i >= 0 && i < nh && h.in(i)) {
      prof[li] = h.b[i];
      prof[RX + li] = h.a[i];
    }
    if (i >= 1 && i - 1 < ne && e.in(i - 1)) {
      prof[2 * RX + li] = e.b[i - 1];
      prof[3 * RX + li] = e.a[i - 1];
    }
  }
}

// Which tiles a launch covers: the interior rectangle, the ring around it,
// or (one launch) all of them, each workgroup taking its tile's path.
enum { kInterior, kRing, kAll };

template <int MODE>
__device__ __forceinline__ bool pick_tile(const TileMap& m, int* tr, int* tc) {
  if constexpr (MODE == kAll) {
    *tr = blockIdx.x / m.C;
    *tc = blockIdx.x % m.C;
    return !(*tr >= m.r0 && *tr < m.r1 && *tc >= m.c0 && *tc < m.c1);
  }
  tile_linear(MODE == kRing, m, blockIdx.x, tr, tc);
  return MODE == kRing;
}

// Interior tiles: the rectangle of tiles whose whole LDS region avoids every
// CPML shell; PML tiles: the ring around it.
template <int TX, int TY, int NS>
TileMap make_map(int nx, int ny, int in_i0, int in_i1, int in_j0, int in_j1) {
  TileMap m;
  m.R = (nx + TX - 1) / TX;
  m.C = (ny + TY - 1) / TY;
  auto lo = [](int edge, int t, int ns) { return (edge + ns + 1 + t - 1) / t; };
  auto hi = [](int edge, int t, int ns) { int v = edge - t - ns; return v < 0 ? 0 : v / t + 1; };
  m.r0 = std::min(m.R, lo(in_i0, TX, NS));
  m.r1 = std::max(m.r0, std::min(m.R, hi(in_i1, TX, NS)));
  m.c0 = std::min(m.C, lo(in_j0, TY, NS));
  m.c1 = std::max(m.c0, std::min(m.C, hi(in_j1, TY, NS)));
  if (m.r1 == m.r0 || m.c1 == m.c0) m.r0 = m.r1 = m.c0 = m.c1 = 0;
  return m;
}

}  // namespace
}  // namespace mt
