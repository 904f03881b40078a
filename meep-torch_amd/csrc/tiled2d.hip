// Temporally blocked 2D TM / TE steppers: NS Yee steps per launch on
// overlapped LDS tiles.
//
// A workgroup owns a TX x TY block of the (i, j) cell lattice.  It loads the
// block plus a halo (NS+1 cells on the low sides, NS on the high sides) of
// the evolving fields, advances NS steps on chip, and writes back only the
// cells it owns.  Per half-step the stencil reaches one cell (D/E halves
// towards lower indices, H/B halves towards higher ones), so after NS steps
// every owned cell, and the one row/column below it that averaged H monitor
// samples need, is exact.  Halo cells are recomputed redundantly; cells whose
// neighbours fall outside the tile compute throw-away values that never reach
// an owned cell.  Reads come from one set of global buffers and writes go to
// the other (ping-pong), so tiles never see each other's partial results.
//
// Thread mapping: a thread owns one column lj of the region and every
// ROWS-th row of it (rows l0, l0 + ROWS, ...), the same cells in every
// sub-step.  All of a cell's values live in its thread's registers (fields,
// D, eps, CPML memory); the LDS holds only the copies that neighbours and
// monitor taps read.  The column's CPML profile values are per-thread
// constants in registers, the rows' come from a small LDS table, so the
// sub-step loop touches no global memory.  (Before, a thread's cells were a
// flat stride through the region: every half-step recomputed each cell's
// row, column and bounds and read the CPML profiles from global memory.
// TE 2048^2, 16x64x4: 25.7 -> 23.4 us per step; the CPML ring of a 256^2 TM
// grid, where that latency was the whole launch, 7.9 -> 3.9 us per step.)
//
// Arithmetic per cell is the per-half-step kernels' (yee2d.hip), op for op,
// so results are bit-identical to them and to the reference's FP32 stepper.
// Tiles whose region touches a CPML shell also run the four psi recursions
// (template PML = true); interior tiles carry none.  Monitor samples are
// taken inside the tile after each step by the tile that owns the sampled
// cell and written to the staging ring consumed by the DFT flush (dft.hip).
#include <hip/hip_runtime.h>

#include "common.h"
#include "tile2d_dev.h"
#include "tiled2d.h"

namespace mt {
namespace {

// ---------------------------------------------------------------- taps
// Whether any monitor term has cells in the owned block [I0, I0+TXo) x
// [J0, J0+TYo) (the cells write_taps writes).  Uniform over the workgroup:
// a tile without taps skips write_taps and the barrier after it.
__device__ __forceinline__ bool taps_touch(const TapSet& taps, int I0, int J0, int TXo, int TYo) {
  for (int q = 0; q < taps.n; ++q) {
    const Tap& t = taps.t[q];
    if (t.line == 1) {
      if (t.fix >= I0 && t.fix < I0 + TXo && t.lo < J0 + TYo && t.lo + t.n > J0) return true;
    } else if (t.line == 2) {
      if (t.fix >= J0 && t.fix < J0 + TYo && t.lo < I0 + TXo && t.lo + t.n > I0) return true;
    } else if (t.line == 3) {
      if (I0 < t.n0 && J0 < t.n1) return true;
    } else if (t.line == 4) {
      if (t.fix >= I0 && t.fix < I0 + TXo && t.lo >= J0 && t.lo < J0 + TYo) return true;
    } else {
      return true;
    }
  }
  return false;
}

// Write this tile's share of every monitor term after sub-step `s`.
// FIELD(id, li, lj) returns the LDS value of field `id` at local cell, for the
// terms of fields F0 to F1 - 1.  D (ids from 3 up) lives in the owning thread's
// registers: its terms are left to write_taps_own, or D visits the LDS where
// some term averages it (AVGD).
template <typename T, int RX, int RY, int F0, int F1, typename F>
__device__ void write_taps(const TapSet& taps, int s, int I0, int J0, int TXo, int TYo, int a0, int b0,
                           F field, int slot_base) {
  const int tid = threadIdx.x;
  for (int q = 0; q < taps.n; ++q) {
    const Tap& t = taps.t[q];
    if ((F0 > 0 && t.field < F0) || t.field >= F1) continue;
    T* out = static_cast<T*>(t.out) + (long long)(t.slot0 + slot_base + s) * t.slot_stride;
    if (t.line == 1) {  // row: fixed i = fix, j = lo + e
      if (t.fix < I0 || t.fix >= I0 + TXo) continue;
      int jlo = max(t.lo, J0), jhi = min(t.lo + t.n, J0 + TYo);
      for (int j = jlo + tid; j < jhi; j += blockDim.x) {
        int li = t.fix - a0, lj = j - b0;
        T v = field(t.field, li, lj);
        if (t.avg) v = T(0.5) * (field(t.field, li - 1, lj) + v);
        out[j - t.lo] = v;
      }
    } else if (t.line == 2) {  // column: fixed j = fix, i = lo + e
      if (t.fix < J0 || t.fix >= J0 + TYo) continue;
      int ilo = max(t.lo, I0), ihi = min(t.lo + t.n, I0 + TXo);
      for (int i = ilo + tid; i < ihi; i += blockDim.x) {
        int li = i - a0, lj = t.fix - b0;
        T v = field(t.field, li, lj);
        if (t.avg) v = T(0.5) * (field(t.field, li, lj - 1) + v);
        out[i - t.lo] = v;
      }
    } else if (t.line == 3) {  // whole field, row-major with row length t.n1
      int ihi = min(I0 + TXo, t.n0), jhi = min(J0 + TYo, t.n1);
      int w = jhi - J0;
      if (I0 >= ihi || w <= 0) continue;
      int cnt = (ihi - I0) * w;
      for (int c = tid; c < cnt; c += blockDim.x) {
        int i = I0 + c / w, j = J0 + c % w;
        out[(long long)i * t.n1 + j] = field(t.field, i - a0, j - b0);
      }
    } else if (t.line == 4) {  // single cell (fix, lo); stacked per step
      if (tid == 0 && t.fix >= I0 && t.fix < I0 + TXo && t.lo >= J0 && t.lo < J0 + TYo)
        out[0] = field(t.field, t.fix - a0, t.lo - b0);
    }
  }
}

// The terms of one D field (id `field`): an owned cell (i, j) with value v
// writes itself (no term averages D; else the AVGD form runs).
template <typename T>
__device__ __forceinline__ void write_taps_own(const TapSet& taps, int s, int field, int i, int j, T v,
                                               int slot_base) {
  for (int q = 0; q < taps.n; ++q) {
    const Tap& t = taps.t[q];
    if (t.field != field) continue;
    T* out = static_cast<T*>(t.out) + (long long)(t.slot0 + slot_base + s) * t.slot_stride;
    if (t.line == 1) {
      if (i == t.fix && j >= t.lo && j < t.lo + t.n) out[j - t.lo] = v;
    } else if (t.line == 2) {
      if (j == t.fix && i >= t.lo && i < t.lo + t.n) out[i - t.lo] = v;
    } else if (t.line == 3) {
      if (i < t.n0 && j < t.n1) out[(long long)i * t.n1 + j] = v;
    } else if (t.line == 4) {
      if (i == t.fix && j == t.lo) out[0] = v;
    }
  }
}

__device__ __forceinline__ bool taps_have(const TapSet& taps, int field0) {
  for (int q = 0; q < taps.n; ++q)
    if (taps.t[q].field >= field0) return true;
  return false;
}

// Does box s reach the region [a0, a0 + RX) x [b0, b0 + RY)?
__device__ __forceinline__ bool box_touches(const mt_source2d& s, int a0, int b0, int RX, int RY) {
  return s.present && s.i0 < a0 + RX && s.i1 > a0 && s.j0 < b0 + RY && s.j1 > b0;
}
__device__ __forceinline__ bool box_has(const mt_source2d& s, int i, int j) {
  return i >= s.i0 && i < s.i1 && j >= s.j0 && j < s.j1;
}
template <typename T>
__device__ __forceinline__ T box_w(const mt_source2d& s, int i, int j) {
  return static_cast<const T*>(s.w)[(long long)(i - s.i0) * (s.j1 - s.j0) + (j - s.j0)];
}

// ------------------------------------------------------------------- TE
template <typename T, int TX, int TY, int NS, int MAXB, bool PML, bool AVGD>
__device__ __forceinline__ void te_tile(const TeTiled<T>& p, const TapSet& taps, int nsub, int write_e, int tr,
                                        int tc, T* sm) {
  using S = Shape<TX, TY, NS, MAXB>;
  constexpr int RX = S::RX, RY = S::RY, RC = S::RC, ROWS = S::ROWS, STR = S::STR, PER = S::PER;
  T *sHz = sm, *sEx = sm + RC, *sEy = sm + 2 * RC, *prof = sm + 3 * RC;
  constexpr int PP = PML ? PER : 1;
  T vPzy[PP], vPzx[PP], vPyx[PP], vPxy[PP];  // psi_Hzy (Dx, y shell, (i, j-1)), psi_Hzx (Dy, x shell,
                                             // (i-1, j)), psi_Eyx / psi_Exy (Hz, x / y shell, (i, j))
  T vHz[PER], vDx[PER], vDy[PER], vKx[PER], vKy[PER], vEx[PER], vEy[PER];
  const int nx = p.nx, ny = p.ny;
  const int I0 = tr * TX, J0 = tc * TY;
  const int a0 = I0 - NS - 1, b0 = J0 - NS - 1;
  const int tid = threadIdx.x, l0 = tid / RY, lj = tid - l0 * RY;
  const int i0 = a0 + l0, j = b0 + lj;
  const T dt = p.dt, dx = p.dx, rdx = p.rdx;
  // shell rows, by value: read through p in the sub-step loop, a batched
  // launch (p in device memory) would load them again after every store
  const int hx_lo = p.hx.lo_end, hx_hi = p.hx.hi_begin, ex_lo = p.ex.lo_end + 1, ex_hi = p.ex.hi_begin + 1;
  auto in_hx = [&](int i) { return i < hx_lo || i >= hx_hi; };
  auto in_ex = [&](int i) { return i < ex_lo || i >= ex_hi; };
  auto ok = [&](int u) { return tid < STR && (u < PER - 1 || l0 + u * ROWS < RX); };
  const bool jhz = j >= 0 && j < ny - 1, jex = j >= 0 && j < ny;   // columns of Hz / Ey and of Ex
  const bool jin = j >= 1 && j < ny - 1;
  const bool in_hy = PML && jhz && p.hy.in(j), in_ey = PML && jin && p.ey.in(j - 1);
  T bhy = T(0), ahy = T(0), bey = T(0), aey = T(0);
  if constexpr (PML) {
    if (in_hy) bhy = p.hy.b[j], ahy = p.hy.a[j];
    if (in_ey) bey = p.ey.b[j - 1], aey = p.ey.a[j - 1];
    load_rows<T, RX>(p.hx, p.ex, a0, nx - 1, nx - 2, prof);
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    const bool rx = !PML || (i >= 0 && i < nx - 1), ry = !PML || (i >= 0 && i < nx);
    const bool hz = ok(u) && rx && (!PML || jhz), ex = ok(u) && rx && (!PML || jex);
    const bool ey = ok(u) && ry && (!PML || jhz);
    vHz[u] = dget(p.Hz, (long long)i * (ny - 1) + j, hz);
    vDx[u] = dget(p.Dx, (long long)i * ny + j, ex);
    vDy[u] = dget(p.Dy, (long long)i * (ny - 1) + j, ey);
    vKx[u] = ex ? p.eps_x[(long long)i * ny + j] : T(1);
    vKy[u] = ey ? p.eps_y[(long long)i * (ny - 1) + j] : T(1);
    if constexpr (PML) {
      vPzy[u] = dget(p.pHzy, (long long)i * (ny - 2) + (j - 1), ex && in_ey);
      vPzx[u] = dget(p.pHzx, (long long)(i - 1) * (ny - 1) + j, ey && i >= 1 && i < nx - 1 && in_ex(i));
      vPyx[u] = dget(p.pEyx, (long long)i * (ny - 1) + j, hz && in_hx(i));
      vPxy[u] = dget(p.pExy, (long long)i * (ny - 1) + j, hz && in_hy);
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (ok(u)) sHz[tid + u * STR] = vHz[u];
  __syncthreads();
  // uniform per tile: does the source reach the LDS region, do taps reach the owned block
  const bool src_tile = box_touches(p.src, a0, b0, RX, RY);
  const bool tap_tile = taps.n && taps_touch(taps, I0, J0, TX, TY);
  const bool tap_d = tap_tile && taps_have(taps, 3);
  const bool jown = lj > NS && lj <= NS + TY && tid < STR;
  auto own = [&](int u) { return jown && l0 + u * ROWS > NS && l0 + u * ROWS <= NS + TX; };
  for (int s = 0; s < nsub; ++s) {
    const T coef = p.coef[s];
    // D half (stepper_te.py:80-103,131-134,160-168)
    {
      T qx[PER], qy[PER];
      auto ax = [&](int u) -> T {
        const int c = tid + u * STR, i = i0 + u * ROWS;
        const bool l = ok(u) && lj >= 1 && (!PML || (jin && i >= 0 && i < nx - 1));
        return l ? vHz[u] - sHz[c - 1] : T(0);
      };
      auto ay = [&](int u) -> T {
        const int c = tid + u * STR, i = i0 + u * ROWS;
        const bool l = ok(u) && (u > 0 || l0 >= 1) && (!PML || (jhz && i >= 1 && i < nx - 1));
        return l ? vHz[u] - sHz[c - RY] : T(0);
      };
      step_quots<T, PER>(dx, rdx, ax, ay, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
        if (!ok(u)) break;
        T cx = qx[u], cy = qy[u];
        if constexpr (PML) {
          if (in_ey && lj >= 1 && i >= 0 && i < nx - 1) {
            const T ps = bey * vPzy[u] + aey * cx;
            vPzy[u] = ps;
            cx = cx + ps;
          }
          if (jhz && (u > 0 || l0 >= 1) && i >= 1 && i < nx - 1 && in_ex(i)) {
            const T ps = prof[2 * RX + li] * vPzx[u] + prof[3 * RX + li] * cy;
            vPzx[u] = ps;
            cy = cy + ps;
          }
        }
        T dyv = vDy[u] - dt * cy;
        vDx[u] = vDx[u] + dt * cx;
        if (src_tile && box_has(p.src, i, j))
          dyv = dyv - coef * static_cast<const T*>(p.src.w)[(long long)s * p.src.wstep +
                                                             (long long)(i - p.src.i0) * (p.src.j1 - p.src.j0) +
                                                             (j - p.src.j0)];
        vDy[u] = dyv;
        vEx[u] = vDx[u] / vKx[u];
        vEy[u] = dyv / vKy[u];
        sEx[c] = vEx[u];
        sEy[c] = vEy[u];
      }
    }
    __syncthreads();
    // B half (stepper_te.py:106-117)
    {
      T qx[PER], qy[PER];
      auto hz = [&](int u) {
        const int i = i0 + u * ROWS;
        return ok(u) && lj < RY - 1 && (u < PER - 1 || l0 + u * ROWS < RX - 1) &&
               (!PML || (jhz && i >= 0 && i < nx - 1));
      };
      auto ax = [&](int u) -> T { return hz(u) ? sEx[tid + u * STR + 1] - vEx[u] : T(0); };
      auto ay = [&](int u) -> T { return hz(u) ? sEy[tid + u * STR + RY] - vEy[u] : T(0); };
      step_quots<T, PER>(dx, rdx, ax, ay, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
        if (!ok(u)) break;
        T a1 = qy[u];
        if constexpr (PML) {
          const bool h = lj < RY - 1 && li < RX - 1 && jhz && i >= 0 && i < nx - 1;
          if (h && in_hx(i)) {
            const T ps = prof[li] * vPyx[u] + prof[RX + li] * qy[u];
            vPyx[u] = ps;
            a1 = a1 + ps;
          }
          a1 = a1 - qx[u];
          if (h && in_hy) {
            const T ps = bhy * vPxy[u] + ahy * qx[u];
            vPxy[u] = ps;
            a1 = a1 - ps;
          }
        } else {
          a1 = a1 - qx[u];
        }
        vHz[u] = vHz[u] - dt * a1;
        sHz[c] = vHz[u];
      }
    }
    __syncthreads();
    if (tap_tile) {
      auto field = [&](int f, int li, int lj) -> T {
        int c = li * RY + lj;
        return f == 0 ? sHz[c] : f == 1 || (AVGD && f == 3) ? sEx[c] : sEy[c];
      };
      write_taps<T, RX, RY, 0, 3>(taps, s, I0, J0, TX, TY, a0, b0, field, 0);
      if (AVGD && tap_d) {   // D takes the place of E, which the next D half writes before it is read
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; ++u)
          if (ok(u)) sEx[tid + u * STR] = vDx[u], sEy[tid + u * STR] = vDy[u];
        __syncthreads();
        write_taps<T, RX, RY, 3, 5>(taps, s, I0, J0, TX, TY, a0, b0, field, 0);
      } else if (tap_d) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          const int i = i0 + u * ROWS;
          if (!own(u)) continue;
          if (i < nx - 1 && j < ny) write_taps_own<T>(taps, s, 3, i, j, vDx[u], 0);
          if (i < nx && j < ny - 1) write_taps_own<T>(taps, s, 4, i, j, vDy[u], 0);
        }
      }
      __syncthreads();
    }
  }
  // write back the owned cells from the registers of the threads that updated them
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    if (!own(u)) continue;
    const long long h = (long long)i * (ny - 1) + j, e = (long long)i * ny + j;
    if (i < nx - 1 && j < ny - 1) {
      p.oHz[h] = vHz[u];
      if constexpr (PML) {
        if (in_hx(i)) p.oEyx[h] = vPyx[u];
        if (in_hy) p.oExy[h] = vPxy[u];
      }
    }
    if (i < nx - 1 && j < ny) {
      p.oDx[e] = vDx[u];
      if (write_e) p.Ex[e] = vEx[u];
      if constexpr (PML)
        if (in_ey) p.oHzy[(long long)i * (ny - 2) + (j - 1)] = vPzy[u];
    }
    if (i < nx && j < ny - 1) {
      p.oDy[h] = vDy[u];
      if (write_e) p.Ey[h] = vEy[u];
      if constexpr (PML)
        if (i >= 1 && i < nx - 1 && in_ex(i)) p.oHzx[(long long)(i - 1) * (ny - 1) + j] = vPzx[u];
    }
  }
}

// ------------------------------------------------------------------- TM
template <typename T, int TX, int TY, int NS, int MAXB, bool PML, bool AVGD = false>
__device__ __forceinline__ void tm_tile(const TmTiled<T>& p, const TapSet& taps, int nsub, int tape_s0, int tr,
                                        int tc, int slot_base, int coef_t0, T* sm) {
  using S = Shape<TX, TY, NS, MAXB>;
  constexpr int RX = S::RX, RY = S::RY, RC = S::RC, ROWS = S::ROWS, STR = S::STR, PER = S::PER;
  T *sEz = sm, *sHx = sm + RC, *sHy = sm + 2 * RC, *prof = sm + 3 * RC;
  constexpr int PP = PML ? PER : 1;
  T vPzy[PP], vPzx[PP], vPyx[PP], vPxy[PP];  // psi_Ezy (Hx, y shell, (i, j)), psi_Ezx (Hy, x shell, (i, j)),
                                             // psi_Hyx / psi_Hxy (Dz, x / y shell, (i-1, jj))
  T vEz[PER], vDz[PER], vHx[PER], vHy[PER], vK[PER];
  const int nx = p.nx, ny = p.ny, ny_e = p.ny_e;
  const int I0 = tr * TX, J0 = tc * TY;
  const int a0 = I0 - NS - 1, b0 = J0 - NS - 1;
  const int tid = threadIdx.x, l0 = tid / RY, lj = tid - l0 * RY;
  const int i0 = a0 + l0, j = b0 + lj, jj = j - (p.y_pmc ? 0 : 1);
  const T dt = p.dt, dx = p.dx, rdx = p.rdx;
  // shell rows, by value: read through p in the sub-step loop, a batched
  // launch (p in device memory) would load them again after every store
  const int hx_lo = p.hx.lo_end, hx_hi = p.hx.hi_begin, ex_lo = p.ex.lo_end + 1, ex_hi = p.ex.hi_begin + 1;
  auto in_hx = [&](int i) { return i < hx_lo || i >= hx_hi; };
  auto in_ex = [&](int i) { return i < ex_lo || i >= ex_hi; };
  auto ok = [&](int u) { return tid < STR && (u < PER - 1 || l0 + u * ROWS < RX); };
  const bool jez = j >= 0 && j < ny, jhx = j >= 0 && j < ny - 1;
  const bool jlive = jez && jj >= 0 && jj < ny_e;   // columns the D half updates
  const bool in_hy = PML && jhx && p.hy.in(j), in_ey = PML && jlive && p.ey.in(jj);
  T bhy = T(0), ahy = T(0), bey = T(0), aey = T(0);
  if constexpr (PML) {
    if (in_hy) bhy = p.hy.b[j], ahy = p.hy.a[j];
    if (in_ey) bey = p.ey.b[jj], aey = p.ey.a[jj];
    load_rows<T, RX>(p.hx, p.ex, a0, nx - 1, nx - 2, prof);
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    const bool ez = ok(u) && (!PML || (i >= 0 && i < nx && jez));
    const bool hx = ez && (!PML || jhx), hy = ez && (!PML || i < nx - 1);
    const long long e = (long long)i * ny + j;
    vEz[u] = dget(p.Ez, e, ez);
    vHx[u] = dget(p.Hx, (long long)i * (ny - 1) + j, hx);
    vHy[u] = dget(p.Hy, e, hy);
    vDz[u] = dget(p.Dz, e, ez);
    vK[u] = ez ? p.eps[e] : T(1);
    if constexpr (PML) {
      const bool live = ez && i >= 1 && i < nx - 1 && jlive;
      const long long q = (long long)(i - 1) * ny_e + jj;
      vPzy[u] = dget(p.pEzy, (long long)i * (ny - 1) + j, hx && in_hy);
      vPzx[u] = dget(p.pEzx, e, hy && in_hx(i));
      vPyx[u] = dget(p.pHyx, q, live && in_ex(i));
      vPxy[u] = dget(p.pHxy, q, live && in_ey);
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int c = tid + u * STR;
    if (ok(u)) {
      sEz[c] = vEz[u];
      sHx[c] = vHx[u];
      sHy[c] = vHy[u];
    }
  }
  __syncthreads();
  // uniform per tile: do the sources reach the LDS region, do taps reach the owned block
  const bool src_tile = box_touches(p.src, a0, b0, RX, RY);
  const bool hx_tile = box_touches(p.hsrc[0], a0, b0, RX, RY), hy_tile = box_touches(p.hsrc[1], a0, b0, RX, RY);
  const bool tap_tile = taps.n && taps_touch(taps, I0, J0, TX, TY);
  const bool tap_d = tap_tile && taps_have(taps, 3);
  const T *coef_tab = p.coef_tab, *hcoef_tab = p.hcoef_tab;
  T* tape = p.tape;
  const bool jown = lj > NS && lj <= NS + TY && tid < STR && j < ny;
  auto own = [&](int u) {
    return jown && l0 + u * ROWS > NS && l0 + u * ROWS <= NS + TX && i0 + u * ROWS < nx;
  };
  for (int s = 0; s < nsub; ++s) {
    const T coef = coef_tab ? coef_tab[coef_t0 + s] : p.coef[s];
    const T hc = hcoef_tab ? hcoef_tab[coef_t0 + s] : p.hcoef[s];
    // B half (stepper_tm.py:85-92,126-128)
    {
      T qx[PER], qy[PER];
      auto ay = [&](int u) -> T {
        const int i = i0 + u * ROWS;
        const bool l = ok(u) && lj < RY - 1 && (!PML || (i >= 0 && i < nx && jhx));
        return l ? sEz[tid + u * STR + 1] - vEz[u] : T(0);
      };
      auto ax = [&](int u) -> T {
        const int i = i0 + u * ROWS;
        const bool l = ok(u) && (u < PER - 1 || l0 + u * ROWS < RX - 1) &&
                       (!PML || (i >= 0 && i < nx - 1 && jez));
        return l ? sEz[tid + u * STR + RY] - vEz[u] : T(0);
      };
      step_quots<T, PER>(dx, rdx, ax, ay, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
        if (!ok(u)) break;
        T cy = qy[u], cx = qx[u];
        if constexpr (PML) {
          if (in_hy && lj < RY - 1 && i >= 0 && i < nx) {
            const T ps = bhy * vPzy[u] + ahy * cy;
            vPzy[u] = ps;
            cy = cy + ps;
          }
          if (jez && li < RX - 1 && i >= 0 && i < nx - 1 && in_hx(i)) {
            const T ps = prof[li] * vPzx[u] + prof[RX + li] * cx;
            vPzx[u] = ps;
            cx = cx + ps;
          }
        }
        T hxv = vHx[u] - dt * cy, hyv = vHy[u] + dt * cx;
        if (hx_tile && box_has(p.hsrc[0], i, j)) hxv = hxv - hc * box_w<T>(p.hsrc[0], i, j);  // stepper_tm.py:190-191
        if (hy_tile && box_has(p.hsrc[1], i, j)) hyv = hyv - hc * box_w<T>(p.hsrc[1], i, j);  // stepper_tm.py:188-189
        vHx[u] = hxv;
        vHy[u] = hyv;
        sHx[c] = hxv;
        sHy[c] = hyv;
      }
    }
    __syncthreads();
    // D half (stepper_tm.py:130-166,197-200,226-227).  Under y_pmc the H
    // beyond a wall is zero: those LDS cells were loaded as zero and no B
    // half updates them.
    {
      T qx[PER], qy[PER];
      auto lv = [&](int u) {
        const int i = i0 + u * ROWS;
        return ok(u) && lj >= 1 && (u > 0 || l0 >= 1) && (!PML || (jlive && i >= 1 && i < nx - 1));
      };
      auto ax = [&](int u) -> T { return lv(u) ? vHx[u] - sHx[tid + u * STR - 1] : T(0); };
      auto ay = [&](int u) -> T { return lv(u) ? vHy[u] - sHy[tid + u * STR - RY] : T(0); };
      step_quots<T, PER>(dx, rdx, ax, ay, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
        if (!ok(u)) break;
        T curl = qy[u];
        if constexpr (PML) {
          const bool live = lj >= 1 && (u > 0 || l0 >= 1) && jlive && i >= 1 && i < nx - 1;
          if (live && in_ex(i)) {
            const T ps = prof[2 * RX + li] * vPyx[u] + prof[3 * RX + li] * qy[u];
            vPyx[u] = ps;
            curl = curl + ps;
          }
          curl = curl - qx[u];
          if (live && in_ey) {
            const T ps = bey * vPxy[u] + aey * qx[u];
            vPxy[u] = ps;
            curl = curl - ps;
          }
        } else {
          curl = curl - qx[u];
        }
        T dz = vDz[u] + dt * curl;
        if (src_tile && box_has(p.src, i, j))
          dz = dz - coef * static_cast<const T*>(p.src.w)[(long long)s * p.src.wstep +
                                                          (long long)(i - p.src.i0) * (p.src.j1 - p.src.j0) +
                                                          (j - p.src.j0)];
        vDz[u] = dz;
        vEz[u] = dz / vK[u];
        sEz[c] = vEz[u];
      }
    }
    __syncthreads();
    if (tape) {
#pragma unroll
      for (int u = 0; u < PER; ++u)
        if (own(u)) tape[(long long)(tape_s0 + s) * nx * ny + (long long)(i0 + u * ROWS) * ny + j] = vEz[u];
    }
    if (tap_tile) {
      auto field = [&](int f, int li, int lj) -> T {
        int c = li * RY + lj;
        return f == 0 ? sEz[c] : f == 1 || (AVGD && f == 3) ? sHx[c] : sHy[c];
      };
      write_taps<T, RX, RY, 0, 3>(taps, s, I0, J0, TX, TY, a0, b0, field, slot_base);
      if (AVGD && tap_d) {   // Dz takes the place of Hx, which the next B half writes before it is read
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; ++u)
          if (ok(u)) sHx[tid + u * STR] = vDz[u];
        __syncthreads();
        write_taps<T, RX, RY, 3, 4>(taps, s, I0, J0, TX, TY, a0, b0, field, slot_base);
      } else if (tap_d) {
#pragma unroll
        for (int u = 0; u < PER; ++u)
          if (own(u)) write_taps_own<T>(taps, s, 3, i0 + u * ROWS, j, vDz[u], slot_base);
      }
      __syncthreads();
    }
  }
  // write back the owned cells from the registers of the threads that updated them
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    if (!own(u)) continue;
    const long long e = (long long)i * ny + j;
    p.oEz[e] = vEz[u];
    p.oDz[e] = vDz[u];
    if (j < ny - 1) p.oHx[(long long)i * (ny - 1) + j] = vHx[u];
    if (i < nx - 1) p.oHy[e] = vHy[u];
    if constexpr (PML) {
      if (in_hy) p.oEzy[(long long)i * (ny - 1) + j] = vPzy[u];
      if (i < nx - 1 && in_hx(i)) p.oEzx[e] = vPzx[u];
      if (i >= 1 && i < nx - 1 && jlive) {
        const long long q = (long long)(i - 1) * ny_e + jj;
        if (in_ex(i)) p.oHyx[q] = vPyx[u];
        if (in_ey) p.oHxy[q] = vPxy[u];
      }
    }
  }
}

// ---------------------------------------------------------------- kernels
// Threads per workgroup, at most.  TM tiles and CPML tiles take up to 1024
// (few cells per thread: their launches are latency chains); TE interior
// tiles of the large shapes take 512 (on 2048^2 that launch is
// arithmetic-bound and 1024-thread tiles measured slower, 98 -> 123 us).  FP64
// TE interior tiles take two cells per thread: with one, two blocks fill a CU
// (8 x 64 x 2 tiles on 2048^2, per two steps: 175 -> 113 us), with three, 101
// registers do (16 x 64 x 2: 101 -> 98 us, 8 x 64 x 4 no faster).
constexpr int kMaxTm = 1024;
template <typename T, int TX, int TY, int NS>
constexpr int te_max(bool pml) {
  if (pml) return 1024;
  const int cells = (TX + 2 * NS + 1) * (TY + 2 * NS + 1);
  return sizeof(T) == 8 ? (cells <= 1024 ? 512 : 1024) : (cells <= 1100 ? 1024 : 512);
}
template <typename T, int TX, int TY, int NS, int MAXB, bool PML>
constexpr int lds_elems() {
  using S = Shape<TX, TY, NS, MAXB>;
  return 3 * S::RC + (PML ? 4 * S::RX : 0);
}

template <typename T, int TX, int TY, int NS, int MAXB, int MODE, bool AVGD>
__global__ __launch_bounds__((Shape<TX, TY, NS, MAXB>::BLK)) void te_tiled(TeTiled<T> p, TapSet taps, int nsub,
                                                                          int write_e) {
  __shared__ T sm[lds_elems<T, TX, TY, NS, MAXB, MODE != kInterior>()];
  int tr, tc;
  const bool pml = pick_tile<MODE>(p.map, &tr, &tc);
  if (MODE == kRing || (MODE == kAll && pml))
    te_tile<T, TX, TY, NS, MAXB, true, AVGD>(p, taps, nsub, write_e, tr, tc, sm);
  else
    te_tile<T, TX, TY, NS, MAXB, false, AVGD>(p, taps, nsub, write_e, tr, tc, sm);
}

template <typename T, int TX, int TY, int NS, int MODE, bool AVGD>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxTm>::BLK)) void tm_tiled(TmTiled<T> p, TapSet taps, int nsub,
                                                                           int tape_s0) {
  __shared__ T sm[lds_elems<T, TX, TY, NS, kMaxTm, MODE != kInterior>()];
  int tr, tc;
  const bool pml = pick_tile<MODE>(p.map, &tr, &tc);
  if (MODE == kRing || (MODE == kAll && pml))
    tm_tile<T, TX, TY, NS, kMaxTm, true, AVGD>(p, taps, nsub, tape_s0, tr, tc, 0, 0, sm);
  else
    tm_tile<T, TX, TY, NS, kMaxTm, false, AVGD>(p, taps, nsub, tape_s0, tr, tc, 0, 0, sm);
}

// FP32 interior tiles held to 64 VGPRs (eight waves per SIMD): two
// 1024-thread workgroups fit a CU (their LDS allows it), so one hides the
// other's barrier and load latency (the 32 x 64 shapes spill 9 VGPRs, 40 B of
// scratch, for it).  Ring tiles (CPML psi) and FP64 keep the plain bound.
template <typename T, int TX, int TY, int NS>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxTm>::BLK)) __attribute__((amdgpu_waves_per_eu(8, 8))) void
tm_tiled_in2(TmTiled<T> p, TapSet taps, int nsub, int tape_s0) {
  __shared__ T sm[lds_elems<T, TX, TY, NS, kMaxTm, false>()];
  int tr, tc;
  tile_linear(false, p.map, blockIdx.x, &tr, &tc);
  tm_tile<T, TX, TY, NS, kMaxTm, false>(p, taps, nsub, tape_s0, tr, tc, 0, 0, sm);
}

// Persistent batched form: every workgroup walks the flattened (variant,
// tile) work list of all variants: the interior tiles, the ring tiles, or
// (kAll) the ring tiles and then the interior ones.  Per-variant problems
// (both ping-pong orientations), taps and tile maps live in device memory, so
// the launch depends only on scalars and can be captured in a graph and
// replayed.
template <typename T, int TX, int TY, int NS, int MODE, bool AVGD>
__device__ __forceinline__ void tm_batch_body(const TmBatchVar<T>* vars, const int* pre_in, const int* pre_ring,
                                              int nvar, int nsub, int parity, int t0, int slot_base, int tape_s0,
                                              T* sm) {
  const int n_ring = MODE == kInterior ? 0 : pre_ring[nvar];
  const int total = n_ring + (MODE == kRing ? 0 : pre_in[nvar]);
  const XcdItems deal = xcd_items(blockIdx.x, gridDim.x, total);
  for (int item = deal.first; item < deal.end; item += deal.stride) {
    const bool ring = MODE == kRing || (MODE == kAll && item < n_ring);
    const int* prefix = ring ? pre_ring : pre_in;
    const int it = ring ? item : item - n_ring;
    int lo = 0, hi = nvar;
    while (hi - lo > 1) {
      int mid = (lo + hi) >> 1;
      if (prefix[mid] <= it) lo = mid;
      else hi = mid;
    }
    const TmBatchVar<T>& V = vars[lo];
    const TmTiled<T>& p = parity ? V.pB : V.pA;
    int tr, tc;
    tile_linear(ring, p.map, it - prefix[lo], &tr, &tc);
    if (MODE == kRing || (MODE == kAll && ring))
      tm_tile<T, TX, TY, NS, kMaxTm, true, AVGD>(p, V.taps, nsub, tape_s0, tr, tc, slot_base, t0, sm);
    else
      tm_tile<T, TX, TY, NS, kMaxTm, false, AVGD>(p, V.taps, nsub, tape_s0, tr, tc, slot_base, t0, sm);
    __syncthreads();
  }
}

template <typename T, int TX, int TY, int NS, int MODE, bool AVGD>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxTm>::BLK)) void tm_batch(const TmBatchVar<T>* vars,
                                                                           const int* pre_in, const int* pre_ring,
                                                                           int nvar, int nsub, int parity, int t0,
                                                                           int slot_base, int tape_s0) {
  __shared__ T sm[lds_elems<T, TX, TY, NS, kMaxTm, MODE != kInterior>()];
  tm_batch_body<T, TX, TY, NS, MODE, AVGD>(vars, pre_in, pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0, sm);
}

// the interior form held to 64 VGPRs, as tm_tiled_in2
template <typename T, int TX, int TY, int NS>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxTm>::BLK)) __attribute__((amdgpu_waves_per_eu(8, 8))) void
tm_batch_in2(const TmBatchVar<T>* vars, const int* pre_in, const int* pre_ring, int nvar, int nsub, int parity,
             int t0, int slot_base, int tape_s0) {
  __shared__ T sm[lds_elems<T, TX, TY, NS, kMaxTm, false>()];
  tm_batch_body<T, TX, TY, NS, kInterior, false>(vars, pre_in, pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0, sm);
}

}  // namespace

// ------------------------------------------------------------- launchers
// A launch whose tiles all find a CU of their own (at most kOneRound) covers
// interior and ring together: their latency chains then run side by side
// instead of one after the other (TM 256^2, 16x64x4 tiles: 31.8 us per 4
// steps in two launches, 15.6 us in one).  Larger grids take two launches,
// which lets the interior kernel keep its smaller register footprint (and two
// workgroups per CU).  The interior (or common) launch is the one the kernel
// timing hook measures, its cell-steps the cells of its tiles times the
// substeps.
template <typename KA, typename K1, typename K2>
void launch_tiles(const TileMap& m, KA kall, K1 kin, K2 kpml, hipStream_t s, long long tile_cells, int nsub) {
  const int n_in = (m.r1 - m.r0) * (m.c1 - m.c0), n = m.R * m.C, n_ring = n - n_in;
  if (n <= kOneRound && n_in && n_ring) {
    timing_begin(s);
    kall(dim3(n));
    timing_end(s, (long long)n * tile_cells * nsub);
    return;
  }
  if (n_in) {
    timing_begin(s);
    kin(dim3(n_in));
    timing_end(s, (long long)n_in * tile_cells * nsub);
  }
  if (n_ring) kpml(dim3(n_ring));
}

template <typename T, int TX, int TY, int NS, bool AVGD = false>
int launch_te_tiled(TeTiled<T> p, const TapSet& taps, int nsub, int write_e, hipStream_t s) {
  constexpr int MI = te_max<T, TX, TY, NS>(false), MR = te_max<T, TX, TY, NS>(true);
  p.map = make_map<TX, TY, NS>(p.nx, p.ny, p.in_i0, p.in_i1, p.in_j0, p.in_j1);
  launch_tiles(
      p.map,
      [&](dim3 g) {
        hipLaunchKernelGGL((te_tiled<T, TX, TY, NS, MR, kAll, AVGD>), g, dim3(Shape<TX, TY, NS, MR>::BLK), 0, s, p, taps, nsub, write_e);
      },
      [&](dim3 g) {
        hipLaunchKernelGGL((te_tiled<T, TX, TY, NS, MI, kInterior, AVGD>), g, dim3(Shape<TX, TY, NS, MI>::BLK), 0, s, p, taps, nsub, write_e);
      },
      [&](dim3 g) {
        hipLaunchKernelGGL((te_tiled<T, TX, TY, NS, MR, kRing, AVGD>), g, dim3(Shape<TX, TY, NS, MR>::BLK), 0, s, p, taps, nsub, write_e);
      },
      s, (long long)TX * TY, nsub);
  return check_launch("te2d tiled step");
}

template <typename T, int TX, int TY, int NS, bool AVGD = false>
int launch_tm_tiled(TmTiled<T> p, const TapSet& taps, int nsub, int tape_s0, hipStream_t s) {
  constexpr int BLK = Shape<TX, TY, NS, kMaxTm>::BLK;
  p.map = make_map<TX, TY, NS>(p.nx, p.ny, p.in_i0, p.in_i1, p.in_j0, p.in_j1);
  launch_tiles(
      p.map,
      [&](dim3 g) { hipLaunchKernelGGL((tm_tiled<T, TX, TY, NS, kAll, AVGD>), g, dim3(BLK), 0, s, p, taps, nsub, tape_s0); },
      [&](dim3 g) {
        if constexpr (sizeof(T) == 4 && !AVGD)
          hipLaunchKernelGGL((tm_tiled_in2<T, TX, TY, NS>), g, dim3(BLK), 0, s, p, taps, nsub, tape_s0);
        else
          hipLaunchKernelGGL((tm_tiled<T, TX, TY, NS, kInterior, AVGD>), g, dim3(BLK), 0, s, p, taps, nsub, tape_s0);
      },
      [&](dim3 g) { hipLaunchKernelGGL((tm_tiled<T, TX, TY, NS, kRing, AVGD>), g, dim3(BLK), 0, s, p, taps, nsub, tape_s0); },
      s, (long long)TX * TY, nsub);
  return check_launch("tm2d tiled step");
}

template <typename T, int TX, int TY, int NS, bool AVGD = false>
int launch_tm_batch(const TmBatchVar<T>* vars, const int* pre_in, const int* pre_ring, int nvar, int n_in,
                    int n_ring, int grid_in, int grid_ring, int nsub, int parity, int t0, int slot_base,
                    int tape_s0, hipStream_t s) {
  constexpr int BLK = Shape<TX, TY, NS, kMaxTm>::BLK;
  const int n = n_in + n_ring;
  if (n <= kOneRound && n_in && n_ring) {
    timing_begin(s);
    hipLaunchKernelGGL((tm_batch<T, TX, TY, NS, kAll, AVGD>), dim3(one_round_grid(n)), dim3(BLK), 0, s, vars, pre_in,
                       pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0);
    timing_end(s, (long long)n * TX * TY * nsub);
    return check_launch("tm2d batched step");
  }
  if (n_in) {
    timing_begin(s);
    if constexpr (sizeof(T) == 4 && !AVGD)
      hipLaunchKernelGGL((tm_batch_in2<T, TX, TY, NS>), dim3(std::min(one_round_grid(n_in), grid_in)), dim3(BLK), 0, s, vars,
                         pre_in, pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0);
    else
      hipLaunchKernelGGL((tm_batch<T, TX, TY, NS, kInterior, AVGD>), dim3(std::min(one_round_grid(n_in), grid_in)), dim3(BLK), 0, s, vars,
                         pre_in, pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0);
    timing_end(s, (long long)n_in * TX * TY * nsub);
  }
  if (n_ring)
    hipLaunchKernelGGL((tm_batch<T, TX, TY, NS, kRing, AVGD>), dim3(std::min(one_round_grid(n_ring), grid_ring)), dim3(BLK), 0, s, vars,
                       pre_in, pre_ring, nvar, nsub, parity, t0, slot_base, tape_s0);
  return check_launch("tm2d batched step");
}

template <int TX, int TY, int NS>
TileMap map_for(int nx, int ny, int in_i0, int in_i1, int in_j0, int in_j1) {
  return make_map<TX, TY, NS>(nx, ny, in_i0, in_i1, in_j0, in_j1);
}

// Tile-shape variants (index = variant id), (TX, TY, NS): owned rows, owned
// columns, Yee steps per launch.  FP64 tiles are smaller so that registers
// and LDS fit one workgroup.  Variants 0-6 are for grids that fill the chip
// (tune.py chooses 2 and 5 in FP32, 2 and 4 in FP64, 1 for a few steps on large
// grids; 0, 3 and 6, and 1 and 5 of FP64, only callers that name them: variant
// arguments, MEEP_TORCH_AMD_VARIANT, tune());
// 7 on are for grids that do not: there a launch lasts as long as one tile
// (VALU issue of the tile's cells on one CU, about 0.3 us per half-step and
// 1000 cells, over about 6 us of launch, load and store latency), so the
// smallest tile that still gives every tile its own CU wins, with as many
// steps per launch as one cell per thread allows.  Measured per Yee step, TM
// FP32: 256^2 16x16x7 2.2 us, 16x64x4 3.9 us; 100x60 8x8x8 2.0 us, 16x16x7
// 2.2 us; 300^2 16x32x4 3.7 us, 16x64x4 3.9 us, 16x16x7 (361 tiles) 3.8 us.
#define MT_VARIANTS_F32(X, T) \
  X(T, 16, 64, 1) X(T, 16, 64, 2) X(T, 16, 64, 4) X(T, 32, 64, 1) X(T, 32, 64, 2) X(T, 32, 64, 4) X(T, 8, 128, 2) \
  X(T, 16, 16, 7) X(T, 8, 8, 8) X(T, 16, 32, 4)
#define MT_VARIANTS_F64(X, T) \
  X(T, 8, 64, 1) X(T, 8, 64, 2) X(T, 8, 64, 4) X(T, 16, 64, 1) X(T, 16, 64, 2) X(T, 16, 32, 2) X(T, 8, 128, 1) \
  X(T, 16, 16, 6) X(T, 8, 8, 8) X(T, 16, 32, 4)
constexpr int kVariants = 10;
// Runs with a term that averages D take this shape (kAvgVariant in the
// dispatches) whatever variant was asked for: D visits the LDS for such terms,
// and as a branch in every kernel that cost 2% of the TM cases and 6% of a batch of
// ten variants.
constexpr int kAvgShape = 1;
static const int kVarF32[kVariants][3] = {{16, 64, 1}, {16, 64, 2}, {16, 64, 4}, {32, 64, 1}, {32, 64, 2},
                                          {32, 64, 4}, {8, 128, 2}, {16, 16, 7}, {8, 8, 8}, {16, 32, 4}};
static const int kVarF64[kVariants][3] = {{8, 64, 1}, {8, 64, 2}, {8, 64, 4}, {16, 64, 1}, {16, 64, 2},
                                          {16, 32, 2}, {8, 128, 1}, {16, 16, 6}, {8, 8, 8}, {16, 32, 4}};

int te_tiled_dispatch_f32(int variant, const TeTiled<float>& p, const TapSet& taps, int nsub, int write_e,
                          hipStream_t s) {
  int v = 0;
#define X(T, A, B, C) \
  if (variant == v++) return launch_te_tiled<T, A, B, C>(p, taps, nsub, write_e, s);
  MT_VARIANTS_F32(X, float)
#undef X
  if (variant == kAvgVariant) return launch_te_tiled<float, 16, 64, 2, true>(p, taps, nsub, write_e, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

int te_tiled_dispatch_f64(int variant, const TeTiled<double>& p, const TapSet& taps, int nsub, int write_e,
                          hipStream_t s) {
  int v = 0;
#define X(T, A, B, C) \
  if (variant == v++) return launch_te_tiled<T, A, B, C>(p, taps, nsub, write_e, s);
  MT_VARIANTS_F64(X, double)
#undef X
  if (variant == kAvgVariant) return launch_te_tiled<double, 8, 64, 2, true>(p, taps, nsub, write_e, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

int tm_tiled_dispatch_f32(int variant, const TmTiled<float>& p, const TapSet& taps, int nsub, int tape_s0,
                          hipStream_t s) {
  int v = 0;
#define X(T, A, B, C) \
  if (variant == v++) return launch_tm_tiled<T, A, B, C>(p, taps, nsub, tape_s0, s);
  MT_VARIANTS_F32(X, float)
#undef X
  if (variant == kAvgVariant) return launch_tm_tiled<float, 16, 64, 2, true>(p, taps, nsub, tape_s0, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

int tm_tiled_dispatch_f64(int variant, const TmTiled<double>& p, const TapSet& taps, int nsub, int tape_s0,
                          hipStream_t s) {
  int v = 0;
#define X(T, A, B, C) \
  if (variant == v++) return launch_tm_tiled<T, A, B, C>(p, taps, nsub, tape_s0, s);
  MT_VARIANTS_F64(X, double)
#undef X
  if (variant == kAvgVariant) return launch_tm_tiled<double, 8, 64, 2, true>(p, taps, nsub, tape_s0, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

int tm_batch_dispatch_f32(int variant, const TmBatchVar<float>* vars, const int* pre_in, const int* pre_ring,
                          int nvar, int n_in, int n_ring, int grid_in, int grid_ring, int nsub, int parity,
                          int t0, int slot_base, int tape_s0, hipStream_t s) {
  int v = 0;
#define X(T, A, B, C)                                                                                  \
  if (variant == v++)                                                                                  \
    return launch_tm_batch<T, A, B, C>(vars, pre_in, pre_ring, nvar, n_in, n_ring, grid_in, grid_ring, \
                                       nsub, parity, t0, slot_base, tape_s0, s);
  MT_VARIANTS_F32(X, float)
#undef X
  if (variant == kAvgVariant)
    return launch_tm_batch<float, 16, 64, 2, true>(vars, pre_in, pre_ring, nvar, n_in, n_ring, grid_in, grid_ring, nsub,
                                                parity, t0, slot_base, tape_s0, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

int tm_batch_dispatch_f64(int variant, const TmBatchVar<double>* vars, const int* pre_in, const int* pre_ring,
                          int nvar, int n_in, int n_ring, int grid_in, int grid_ring, int nsub, int parity,
                          int t0, int slot_base, int tape_s0, hipStream_t s) {
  int v = 0;
#define X(T, A, B, C)                                                                                  \
  if (variant == v++)                                                                                  \
    return launch_tm_batch<T, A, B, C>(vars, pre_in, pre_ring, nvar, n_in, n_ring, grid_in, grid_ring, \
                                       nsub, parity, t0, slot_base, tape_s0, s);
  MT_VARIANTS_F64(X, double)
#undef X
  if (variant == kAvgVariant)
    return launch_tm_batch<double, 8, 64, 2, true>(vars, pre_in, pre_ring, nvar, n_in, n_ring, grid_in, grid_ring, nsub,
                                                parity, t0, slot_base, tape_s0, s);
  return fail(MT_EINVAL, "unknown tiled variant");
}

TileMap tiled_map(int variant, int dtype, int nx, int ny, int in_i0, int in_i1, int in_j0, int in_j1) {
  if (variant == kAvgVariant) variant = kAvgShape;
  int v = 0;
#define X(T, A, B, C) \
  if (variant == v++) return map_for<A, B, C>(nx, ny, in_i0, in_i1, in_j0, in_j1);
  if (dtype == MT_F64) {
    MT_VARIANTS_F64(X, double)
  } else {
    MT_VARIANTS_F32(X, float)
  }
#undef X
  return TileMap{};
}

int tiled_variant_count() { return kVariants; }

int tiled_variant_steps(int variant, int dtype) {
  if (variant == kAvgVariant) variant = kAvgShape;
  if (variant < 0 || variant >= kVariants) return 0;
  return dtype == MT_F64 ? kVarF64[variant][2] : kVarF32[variant][2];
}

}  // namespace mt

extern "C" int mt_tiled_variants(int dtype, int* steps, int* tx, int* ty) {
  const int(*tab)[3] = dtype == MT_F64 ? mt::kVarF64 : mt::kVarF32;
  for (int v = 0; v < mt::kVariants; ++v) {
    if (steps) steps[v] = tab[v][2];
    if (tx) tx[v] = tab[v][0];
    if (ty) ty[v] = tab[v][1];
  }
  return mt::kVariants;
}
