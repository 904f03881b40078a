// Reverse-time discrete adjoint of the 3D functional Yee step (CPML shells,
// material conductivity, soft sources, DFT monitors), for dL/deps.
//
// Forward step t (yee3d.hip) maps x_t -> x_{t+1}:
//   H half  for each H component, two differences of the old E (÷ dx), each
//           through its CPML recursion psi' = b psi + a g inside a shell:
//           Hx' = Hx - dt (cy - cz), Hy' = Hy - dt (cz - cx), Hz' = Hz - dt (cx - cy)
//   E half  for each E component, two differences of the new H through the
//           E-side psi; curl = 0 on the PEC faces; eps_c = the two-point
//           average of the cell eps along the component's axis;
//           E' = E + (dt curl + source) / eps_c  (in exact arithmetic)
//   then the monitors sample (E', H').
// One reverse step transposes this in
//   inject  monitor cotangents added to the adjoint arrays
//   E pass  per E cell, first the transposed E differences of the H pass of
//           the step after (C), then (A) the eps_c cotangent
//           -(dL/dE') (E' - E) / eps_c (E, E' from the tape), the curl
//           cotangent dt/eps_c dL/dE', the E-side psi cotangents and the
//           cotangents of the H differences (g[0..5])
//   H pass  per H cell: dL/dH' += transposed H differences of g[0..5];
//           H-side psi cotangents and the E-difference cotangents (g[6..11])
// The steps of one call run inject, E, H per step; the first E pass has no C,
// and a last one only does C.  C and A touch the same E cell, so joining them
// (with the injection before both) saves a pass over dL/dE.  The eps_c
// cotangents add up per component (geps, started by the call's first E pass)
// and are averaged onto the cells once, by the last one.
// Of the two difference cotangents of a cell, the second is the negative of
// the first where neither lies in a shell; only shell cells store it and
// readers take the first one's negative elsewhere.
//
// Bound by the bytes moved through L2 and by latency at the sizes of a design
// (its arrays fit the caches): three passes with every cotangent stored and
// the averaging in each step moved 54 words per cell and step, this 37, and
// every load of a cell is issued before its first store (the arrays do not
// alias, which the compiler cannot know).
// FP32, 96 x 88 x 80 (2.7 MB per array), per step: 63.9 us in three passes
// (23.8 + 19.0 + 21.1) -> 33.1 (E 20.8, H 12.3); the whole gradient of 240
// steps 29.3 -> 21.7 ms.
// Identity parts (dE'/dE = 1, dH'/dH = 1) leave the adjoint arrays in place.
// With poles, A also transposes the pole recurrence (pole3_adj).
// With conductivity the step is E' = d1 E + (d2 curl + source) / eps_c and
// H' = h1 H - h2 curl: A scales dL/dE' by d1 in place, uses d2 for dt and
// -(dL/dE') (E' - d1 E) / eps_c for the eps_c cotangent; B scales dL/dH' by
// h1 and uses h2 for dt.
#include <hip/hip_runtime.h>

#include "adjoint2d.h"
#include "common.h"

namespace mt {
namespace {

enum { P_EZ_Y, P_EY_Z, P_EX_Z, P_EZ_X, P_EY_X, P_EX_Y, P_HZ_Y, P_HY_Z, P_HX_Z, P_HZ_X, P_HY_X, P_HX_Y };
// difference-cotangent scratch slots
enum { G_HZ_Y, G_HY_Z, G_HX_Z, G_HZ_X, G_HY_X, G_HX_Y, G_EZ_Y, G_EY_Z, G_EX_Z, G_EZ_X, G_EY_X, G_EX_Y };

template <typename T>
struct A3 {
  int nx, ny, nz;
  T dt, dx;
  const T* eps;
  Pml<T> h[3], e[3];
  T *aEx, *aEy, *aEz, *aHx, *aHy, *aHz;
  T* apsi[12];
  T* g[12];
  T* geps[3];
  T* eps_grad;
  // conductivity pairs (d1, d2) of ex ey ez hx hy hz, or all NULL
  const T* dmp[12];
  // np ADE poles: scalars c1[n], c2[n]; per E component the c3 stack and the
  // cotangents of the P / P_prev stacks (np component grids each)
  int np;
  const T *c1, *c2;
  const T* c3[3];
  T *aPc[3], *aPp[3];
};

// Transpose of one E cell's poles: P' = (c1 P + c2 P_prev) + c3 E and
// E' = (d1 (E eps_c + sum P) + d2 curl - sum P') / eps_c, with r = E'b / eps_c.
// P' gains -r, P gains d1 r + c1 P'b + P_prev'b (P_prev' = P), P_prev gains
// c2 P'b; returns the old E's cotangent from the poles, sum c3 P'b.
template <typename T>
__device__ __forceinline__ T pole3_adj(const A3<T>& p, int a, long long q, long long nq, T d1, T r) {
  T e_old = T(0);
  for (int n = 0; n < p.np; ++n) {
    const long long o = (long long)n * nq + q;
    const T apn = p.aPc[a][o] - r, prev = p.aPp[a][o];
    p.aPc[a][o] = d1 * r + p.c1[n] * apn + prev;
    p.aPp[a][o] = p.c2[n] * apn;
    e_old = e_old + p.c3[a][o] * apn;
  }
  return e_old;
}

// Transpose of c = d + psi', psi' = b psi + a d (psi' only inside a shell):
// given the cotangent cb of c, returns the cotangent of d and updates the
// psi cotangent in place (psi' cotangent from later steps + cb -> b * that).
// Split into loads and arithmetic + store.
template <typename T>
struct CeT {
  bool in;
  T psi, b, a;
};
template <typename T>
__device__ __forceinline__ CeT<T> ce_t_load(const Pml<T>& pr, int idx, bool ok, const T* apsi, long long q) {
  CeT<T> c{ok && pr.in(idx), T(0), T(0), T(0)};
  if (c.in) c.psi = apsi[q], c.b = pr.b[idx], c.a = pr.a[idx];
  return c;
}
template <typename T>
__device__ __forceinline__ T ce_t_apply(const CeT<T>& c, T* apsi, long long q, T cb) {
  if (!c.in) return cb;
  const T tot = c.psi + cb;
  apsi[q] = c.b * tot;
  return cb + c.a * tot;
}

// Second difference cotangent of a cell: stored inside a shell of either
// axis, the first one's negative elsewhere.
template <typename T>
__device__ __forceinline__ T second(const T* g1, const T* g2, long long q, bool shell) {
  const T v = (shell ? g2 : g1)[q];
  return shell ? v : -v;
}

// One E component's reverse update (A) from its loaded values.
template <typename T>
struct ECell {
  T ab, de, epsc, d1, d2, acc;
};

// M: conductivity and poles may be present (their pointers alone cost 64
// spilled scalar registers).
template <typename T, bool C, bool A, bool M>
__global__ __launch_bounds__(kBlock3) void adj3_e(A3<T> p, const T* e0, const T* e1) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, i = blockIdx.z;
  const int nx = p.nx, ny = p.ny, nz = p.nz;
  if (j >= ny || k >= nz) return;
  const T dt = p.dt, rdx = T(1) / p.dx;
  const long long nEx = (long long)(nx - 1) * ny * nz, nEy = (long long)nx * (ny - 1) * nz;
  const long long nEz = (long long)nx * ny * (nz - 1);
  const long long x = ((long long)i * ny + j) * nz + k;                // eps, Ex
  const long long y = ((long long)i * (ny - 1) + j) * nz + k;          // Ey, Hz
  const long long z = ((long long)i * ny + j) * (nz - 1) + k;          // Ez, Hy
  const long long h = ((long long)i * (ny - 1) + j) * (nz - 1) + k;    // Hx
  const bool fx = i < nx - 1, fy = j < ny - 1, fz = k < nz - 1;        // Ex, Ey, Ez exist at this cell
  const bool ix = i >= 1 && fx, jy = j >= 1 && fy, kz = k >= 1 && fz;
  // ---- loads (every one before the first store)
  T ax = T(0), ay = T(0), az = T(0);
  if (fx) ax = p.aEx[x];
  if (fy) ay = p.aEy[y];
  if (fz) az = p.aEz[z];
  T g[12];
  if constexpr (C) {
#pragma unroll
    for (int q = 0; q < 12; ++q) g[q] = T(0);
    const bool hi = p.h[0].in(i), hj = p.h[1].in(j), hk = p.h[2].in(k);
    if (fx) {  // in Hy (z-diff) and Hz (y-diff)
      if (k >= 1) g[0] = p.g[G_EX_Z][z - 1];
      if (fz) g[1] = p.g[G_EX_Z][z];
      if (j >= 1) g[2] = second(p.g[G_EY_X], p.g[G_EX_Y], y - nz, hi || p.h[1].in(j - 1));
      if (fy) g[3] = second(p.g[G_EY_X], p.g[G_EX_Y], y, hi || hj);
    }
    if (fy) {  // in Hx (z-diff) and Hz (x-diff)
      if (k >= 1) g[4] = second(p.g[G_EZ_Y], p.g[G_EY_Z], h - 1, hj || p.h[2].in(k - 1));
      if (fz) g[5] = second(p.g[G_EZ_Y], p.g[G_EY_Z], h, hj || hk);
      if (i >= 1) g[6] = p.g[G_EY_X][y - (long long)(ny - 1) * nz];
      if (fx) g[7] = p.g[G_EY_X][y];
    }
    if (fz) {  // in Hx (y-diff) and Hy (x-diff)
      if (j >= 1) g[8] = p.g[G_EZ_Y][h - (nz - 1)];
      if (fy) g[9] = p.g[G_EZ_Y][h];
      if (i >= 1) g[10] = second(p.g[G_EX_Z], p.g[G_EZ_X], z - (long long)ny * (nz - 1), hk || p.h[0].in(i - 1));
      if (fx) g[11] = second(p.g[G_EX_Z], p.g[G_EZ_X], z, hk || hi);
    }
  }
  if constexpr (!A) {
    T ge = T(0);
    if (fx) ge += p.geps[0][x];
    if (i >= 1) ge += p.geps[0][x - (long long)ny * nz];
    if (fy) ge += p.geps[1][y];
    if (j >= 1) ge += p.geps[1][y - nz];
    if (fz) ge += p.geps[2][z];
    if (k >= 1) ge += p.geps[2][z - 1];
    p.eps_grad[x] += T(0.5) * ge;
    if (fx) p.aEx[x] = (((ax + g[0]) - g[1]) + g[2]) - g[3];
    if (fy) p.aEy[y] = (((ay + g[4]) - g[5]) + g[6]) - g[7];
    if (fz) p.aEz[z] = (((az + g[8]) - g[9]) + g[10]) - g[11];
    return;
  } else {
    const bool m = M && p.dmp[0] != nullptr;
    const T eps0 = p.eps[x];
    ECell<T> cx, cy, cz;
    auto load = [&](ECell<T>& c, int a, long long q, long long base, long long up) {
      c.epsc = T(0.5) * (eps0 + p.eps[x + up]);
      c.d1 = m ? p.dmp[2 * a][q] : T(1);
      c.d2 = m ? p.dmp[2 * a + 1][q] : dt;
      const T old = e0[base + q];
      c.de = e1[base + q] - (m ? c.d1 * old : old);
      c.acc = C ? p.geps[a][q] : T(0);
    };
    if (fx) load(cx, 0, x, 0, (long long)ny * nz);
    if (fy) load(cy, 1, y, nEx, nz);
    if (fz) load(cz, 2, z, nEx + nEy, 1);
    const bool ei = p.e[0].in(i - 1), ej = p.e[1].in(j - 1), ek = p.e[2].in(k - 1);
    const long long qxy = ((long long)i * (ny - 2) + (j - 1)) * nz + k, qxz = ((long long)i * ny + j) * (nz - 2) + (k - 1);
    const long long qyz = ((long long)i * (ny - 1) + j) * (nz - 2) + (k - 1);
    const long long qyx = ((long long)(i - 1) * (ny - 1) + j) * nz + k;
    const long long qzx = ((long long)(i - 1) * ny + j) * (nz - 1) + k;
    const long long qzy = ((long long)i * (ny - 2) + (j - 1)) * (nz - 1) + k;
    const CeT<T> sxy = ce_t_load(p.e[1], j - 1, fx && jy, p.apsi[P_HZ_Y], qxy);
    const CeT<T> sxz = ce_t_load(p.e[2], k - 1, fx && kz, p.apsi[P_HY_Z], qxz);
    const CeT<T> syz = ce_t_load(p.e[2], k - 1, fy && kz, p.apsi[P_HX_Z], qyz);
    const CeT<T> syx = ce_t_load(p.e[0], i - 1, fy && ix, p.apsi[P_HZ_X], qyx);
    const CeT<T> szx = ce_t_load(p.e[0], i - 1, fz && ix, p.apsi[P_HY_X], qzx);
    const CeT<T> szy = ce_t_load(p.e[1], j - 1, fz && jy, p.apsi[P_HX_Y], qzy);
    // ---- arithmetic and stores
    if constexpr (C) {
      ax = (((ax + g[0]) - g[1]) + g[2]) - g[3];
      ay = (((ay + g[4]) - g[5]) + g[6]) - g[7];
      az = (((az + g[8]) - g[9]) + g[10]) - g[11];
    }
    auto stay = [&](int a, T* arr, long long q, long long nq, T ab, const ECell<T>& c) {
      p.geps[a][q] = c.acc - ab * c.de / c.epsc;
      if (M && p.np) arr[q] = c.d1 * ab + pole3_adj(p, a, q, nq, c.d1, ab / c.epsc);
      else if (C || m) arr[q] = m ? c.d1 * ab : ab;
    };
    if (fx) {  // Ex: curl = chy (Hz y-diff) - chz (Hy z-diff)
      stay(0, p.aEx, x, nEx, ax, cx);
      const T cb = (jy && kz) ? ax * cx.d2 / cx.epsc : T(0);
      p.g[G_HZ_Y][x] = ce_t_apply(sxy, p.apsi[P_HZ_Y], qxy, cb) * rdx;
      if (ej || ek) p.g[G_HY_Z][x] = (kz ? ce_t_apply(sxz, p.apsi[P_HY_Z], qxz, -cb) : T(0)) * rdx;
    }
    if (fy) {  // Ey: curl = chz (Hx z-diff) - chx (Hz x-diff)
      stay(1, p.aEy, y, nEy, ay, cy);
      const T cb = (kz && ix) ? ay * cy.d2 / cy.epsc : T(0);
      p.g[G_HX_Z][y] = ce_t_apply(syz, p.apsi[P_HX_Z], qyz, cb) * rdx;
      if (ek || ei) p.g[G_HZ_X][y] = (ix ? ce_t_apply(syx, p.apsi[P_HZ_X], qyx, -cb) : T(0)) * rdx;
    }
    if (fz) {  // Ez: curl = chx (Hy x-diff) - chy (Hx y-diff)
      stay(2, p.aEz, z, nEz, az, cz);
      const T cb = (ix && jy) ? az * cz.d2 / cz.epsc : T(0);
      p.g[G_HY_X][z] = ce_t_apply(szx, p.apsi[P_HY_X], qzx, cb) * rdx;
      if (ei || ej) p.g[G_HX_Y][z] = (jy ? ce_t_apply(szy, p.apsi[P_HX_Y], qzy, -cb) : T(0)) * rdx;
    }
  }
}

template <typename T, bool M>
__global__ __launch_bounds__(kBlock3) void adj3_h(A3<T> p) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, i = blockIdx.z;
  const int nx = p.nx, ny = p.ny, nz = p.nz;
  if (j >= ny || k >= nz) return;
  const T dt = p.dt, rdx = T(1) / p.dx;
  const long long x = ((long long)i * ny + j) * nz + k;                // Ex
  const long long y = ((long long)i * (ny - 1) + j) * nz + k;          // Ey, Hz
  const long long z = ((long long)i * ny + j) * (nz - 1) + k;          // Ez, Hy
  const long long h = ((long long)i * (ny - 1) + j) * (nz - 1) + k;    // Hx
  const bool fx = j < ny - 1 && k < nz - 1, fy = i < nx - 1 && k < nz - 1, fz = i < nx - 1 && j < ny - 1;
  const bool ei = p.e[0].in(i - 1), ej = p.e[1].in(j - 1), ek = p.e[2].in(k - 1);
  const bool hi = p.h[0].in(i), hj = p.h[1].in(j), hk = p.h[2].in(k);
  const bool m = M && p.dmp[0] != nullptr;
  // ---- loads (every one before the first store)
  T hx = T(0), hy = T(0), hz = T(0), g[12], d1x = T(1), d2x = dt, d1y = T(1), d2y = dt, d1z = T(1), d2z = dt;
#pragma unroll
  for (int q = 0; q < 12; ++q) g[q] = T(0);
  if (fx) {
    hx = p.aHx[h];
    g[0] = p.g[G_HX_Z][y];
    g[1] = p.g[G_HX_Z][y + 1];
    g[2] = second(p.g[G_HY_X], p.g[G_HX_Y], z, ei || ej);
    g[3] = second(p.g[G_HY_X], p.g[G_HX_Y], z + (nz - 1), ei || p.e[1].in(j));
    if (m) d1x = p.dmp[6][h], d2x = p.dmp[7][h];
  }
  if (fy) {
    hy = p.aHy[z];
    g[4] = second(p.g[G_HZ_Y], p.g[G_HY_Z], x, ej || ek);
    g[5] = second(p.g[G_HZ_Y], p.g[G_HY_Z], x + 1, ej || p.e[2].in(k));
    g[6] = p.g[G_HY_X][z];
    g[7] = p.g[G_HY_X][z + (long long)ny * (nz - 1)];
    if (m) d1y = p.dmp[8][z], d2y = p.dmp[9][z];
  }
  if (fz) {
    hz = p.aHz[y];
    g[8] = p.g[G_HZ_Y][x];
    g[9] = p.g[G_HZ_Y][x + nz];
    g[10] = second(p.g[G_HX_Z], p.g[G_HZ_X], y, ek || ei);
    g[11] = second(p.g[G_HX_Z], p.g[G_HZ_X], y + (long long)(ny - 1) * nz, ek || p.e[0].in(i));
    if (m) d1z = p.dmp[10][y], d2z = p.dmp[11][y];
  }
  const CeT<T> sxy = ce_t_load(p.h[1], j, fx, p.apsi[P_EZ_Y], h), sxz = ce_t_load(p.h[2], k, fx, p.apsi[P_EY_Z], h);
  const CeT<T> syz = ce_t_load(p.h[2], k, fy, p.apsi[P_EX_Z], z), syx = ce_t_load(p.h[0], i, fy, p.apsi[P_EZ_X], z);
  const CeT<T> szx = ce_t_load(p.h[0], i, fz, p.apsi[P_EY_X], y), szy = ce_t_load(p.h[1], j, fz, p.apsi[P_EX_Y], y);
  // ---- arithmetic and stores
  if (fx) {  // Hx' = h1 Hx - h2 (cy - cz): cy from Ez y-diff, cz from Ey z-diff
    const T a = hx + (g[0] - g[1]) + (g[2] - g[3]);
    p.aHx[h] = m ? d1x * a : a;
    p.g[G_EZ_Y][h] = ce_t_apply(sxy, p.apsi[P_EZ_Y], h, -d2x * a) * rdx;
    if (hj || hk) p.g[G_EY_Z][h] = ce_t_apply(sxz, p.apsi[P_EY_Z], h, d2x * a) * rdx;
  }
  if (fy) {  // Hy' = h1 Hy - h2 (cz - cx): cz from Ex z-diff, cx from Ez x-diff
    const T a = hy + (g[4] - g[5]) + (g[6] - g[7]);
    p.aHy[z] = m ? d1y * a : a;
    p.g[G_EX_Z][z] = ce_t_apply(syz, p.apsi[P_EX_Z], z, -d2y * a) * rdx;
    if (hk || hi) p.g[G_EZ_X][z] = ce_t_apply(syx, p.apsi[P_EZ_X], z, d2y * a) * rdx;
  }
  if (fz) {  // Hz' = h1 Hz - h2 (cx - cy): cx from Ey x-diff, cy from Ex y-diff
    const T a = hz + (g[8] - g[9]) + (g[10] - g[11]);
    p.aHz[y] = m ? d1z * a : a;
    p.g[G_EY_X][y] = ce_t_apply(szx, p.apsi[P_EY_X], y, -d2z * a) * rdx;
    if (hi || hj) p.g[G_EX_Y][y] = ce_t_apply(szy, p.apsi[P_EX_Y], y, d2z * a) * rdx;
  }
}

template <typename T>
__global__ __launch_bounds__(kInjE* kInjS) void adj3_inject(mt_monitor m, int t, double dt_d) {
  adj_inject_block<T>(m, blockIdx.x * kInjE, t, dt_d, 0);
}

template <typename T, bool M>
int adj3_t(const mt_yee3d* d, const mt_yee3d_adj* a, const void* tape, const mt_monitor* mons, int n_mons,
           int step0, int k, hipStream_t s) {
  A3<T> p;
  p.nx = d->nx;
  p.ny = d->ny;
  p.nz = d->nz;
  p.dt = static_cast<T>(d->dt);
  p.dx = static_cast<T>(d->dx);
  p.eps = static_cast<const T*>(d->eps);
  for (int q = 0; q < 3; ++q) {
    p.h[q] = pml_of<T>(d->h[q]);
    p.e[q] = pml_of<T>(d->e[q]);
  }
  p.aEx = static_cast<T*>(a->aEx);
  p.aEy = static_cast<T*>(a->aEy);
  p.aEz = static_cast<T*>(a->aEz);
  p.aHx = static_cast<T*>(a->aHx);
  p.aHy = static_cast<T*>(a->aHy);
  p.aHz = static_cast<T*>(a->aHz);
  for (int q = 0; q < 12; ++q) {
    p.apsi[q] = static_cast<T*>(a->apsi[q]);
    p.g[q] = static_cast<T*>(a->g[q]);
  }
  for (int q = 0; q < 3; ++q) p.geps[q] = static_cast<T*>(a->geps[q]);
  p.eps_grad = static_cast<T*>(a->eps_grad);
  for (int q = 0; q < 12; ++q) p.dmp[q] = static_cast<const T*>(d->damp[q]);
  p.np = (d->n_poles > 0 && a->aP_cur[0]) ? d->n_poles : 0;
  p.c1 = static_cast<const T*>(d->c1);
  p.c2 = static_cast<const T*>(d->c2);
  for (int q = 0; q < 3; ++q) {
    p.c3[q] = static_cast<const T*>(d->c3[q]);
    p.aPc[q] = static_cast<T*>(a->aP_cur[q]);
    p.aPp[q] = static_cast<T*>(a->aP_prev[q]);
  }
  const long long slot = (long long)(p.nx - 1) * p.ny * p.nz + (long long)p.nx * (p.ny - 1) * p.nz +
                         (long long)p.nx * p.ny * (p.nz - 1);
  const T* tp = static_cast<const T*>(tape);
  const dim3 blk = block3(p.ny, p.nz, sizeof(T)), grd = grid3(blk, p.nx, p.ny, p.nz);
  for (int s_ = k - 1; s_ >= 0; --s_) {
    const int t = step0 + s_;
    for (int m = 0; m < n_mons; ++m) {
      const mt_monitor& mm = mons[m];
      const int n = mm.n0 * mm.n1;
      if (n == 0) continue;
      hipLaunchKernelGGL(adj3_inject<T>, dim3((n + kInjE - 1) / kInjE), dim3(kInjE * kInjS), 0, s, mm, t, d->dt);
    }
    const T *e0 = tp + (long long)s_ * slot, *e1 = e0 + slot;
    if (s_ == k - 1) hipLaunchKernelGGL((adj3_e<T, false, true, M>), grd, blk, 0, s, p, e0, e1);
    else hipLaunchKernelGGL((adj3_e<T, true, true, M>), grd, blk, 0, s, p, e0, e1);
    hipLaunchKernelGGL((adj3_h<T, M>), grd, blk, 0, s, p);
    int rc = check_launch("yee3d adjoint step");
    if (rc) return rc;
  }
  if (k > 0) hipLaunchKernelGGL((adj3_e<T, true, false, M>), grd, blk, 0, s, p, (const T*)nullptr, (const T*)nullptr);
  if (int rc = check_launch("yee3d adjoint step")) return rc;
  return MT_OK;
}

}  // namespace
}  // namespace mt

using namespace mt;

extern "C" int mt_yee3d_adjoint(const mt_yee3d* p, const mt_yee3d_adj* a, const void* tape,
                                const mt_monitor* mons, int n_mons, int step0, int k, void* stream) {
  if (!p || !a) return fail(MT_EINVAL, "null problem or adjoint state");
  if (p->nx < 3 || p->ny < 3 || p->nz < 3) return fail(MT_EINVAL, "grid must be at least 3x3x3");
  if ((long long)p->ny * p->nz > (1LL << 31) || p->nx > 65535)
    return fail(MT_EINVAL, "grid too large for the launch shape");
  if (p->lean) return fail(MT_EINVAL, "the 3D adjoint transposes the functional stepper (lean = 0)");
  if (p->absorber) return fail(MT_EINVAL, "the 3D adjoint transposes the CPML path (absorber = 0)");
  if (p->n_poles < 0) return fail(MT_EINVAL, "negative pole count");
  if (p->n_poles) {
    if (!p->damp[0] || !p->c1 || !p->c2) return fail(MT_EINVAL, "3D adjoint with poles needs damp, c1 and c2");
    for (int q = 0; q < 3; ++q)
      if (!p->c3[q] || !a->aP_cur[q] || !a->aP_prev[q])
        return fail(MT_EINVAL, "3D adjoint with poles needs c3 and the pole-stack cotangents");
  }
  for (int q = 1; q < 12; ++q)
    if (!p->damp[q] != !p->damp[0]) return fail(MT_EINVAL, "3D conductivity needs all 12 damping arrays");
  if (k < 0) return fail(MT_EINVAL, "negative step count");
  if (k > 0 && !tape) return fail(MT_EINVAL, "adjoint needs the forward E tape");
  if (p->dtype != MT_F32 && p->dtype != MT_F64) return fail(MT_EINVAL, "dtype must be f32 or f64");
  if (!p->eps || !a->aEx || !a->aEy || !a->aEz || !a->aHx || !a->aHy || !a->aHz || !a->eps_grad)
    return fail(MT_EINVAL, "null adjoint pointer");
  for (int q = 0; q < 12; ++q)
    if (!a->apsi[q] || !a->g[q]) return fail(MT_EINVAL, "null adjoint psi or scratch pointer");
  for (int q = 0; q < 3; ++q)
    if (!a->geps[q]) return fail(MT_EINVAL, "null eps_c cotangent pointer");
  int n[3] = {p->nx, p->ny, p->nz};
  int rc;
  for (int q = 0; q < 3; ++q) {
    if ((rc = check_axis(p->h[q], n[q] - 1, "h"))) return rc;
    if ((rc = check_axis(p->e[q], n[q] - 2, "e"))) return rc;
  }
  for (int i = 0; i < n_mons; ++i) {
    const mt_monitor& m = mons[i];
    if (m.n_terms < 1 || m.n_terms > MT_MAX_TERMS || !m.acc) return fail(MT_EINVAL, "bad monitor");
    if (m.kind == 0 && (m.nfreq < 1 || !m.omega)) return fail(MT_EINVAL, "monitor: no frequencies");
    if (m.kind != 0) return fail(MT_EINVAL, "3D adjoint: DFT monitors only");
    for (int q = 0; q < m.n_terms; ++q)
      if (!m.term[q].a) return fail(MT_EINVAL, "monitor: null adjoint view");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool media = p->damp[0] != nullptr;
  if (p->dtype == MT_F64)
    return media ? adj3_t<double, true>(p, a, tape, mons, n_mons, step0, k, s)
                 : adj3_t<double, false>(p, a, tape, mons, n_mons, step0, k, s);
  return media ? adj3_t<float, true>(p, a, tape, mons, n_mons, step0, k, s)
               : adj3_t<float, false>(p, a, tape, mons, n_mons, step0, k, s);
}
