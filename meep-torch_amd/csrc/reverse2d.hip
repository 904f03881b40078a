// Temporally blocked reverse sweep of the 2D TM step: NS exact transposes of
// the Yee step per launch on overlapped LDS tiles, for problems without media
// or symmetry cuts.
//
// One reverse step is adj_a_cell, adj_b_cell, adj_c_cell (adjoint2d.h), op for
// op, preceded by the monitor cotangents: A needs only its own cell, B reads
// A's results one cell up in i and j, C reads B's one cell down, so the tile
// of the forward stepper (tile2d_dev.h: NS + 1 halo cells low, NS high) keeps
// every owned cell exact for NS steps.  A cell's cotangents, eps and CPML
// cotangents stay in its thread's registers; the four difference cotangents
// pass through LDS; the owned cells' tape values are loaded one step ahead.
// Cotangents are read from one set and written to the other.
//
// Why: the per-step sweep took four launches per step (injection, A, B, C),
// each at launch latency on the small grids of a design loop (256^2: 15.1 us
// per step), and in the batched form read and wrote every cotangent from
// memory once per step.
//
// Monitor cotangents dL/dsample(t) = sum_f dt (cos(w t) dacc_re - sin(w t)
// dacc_im) do not depend on the fields, so they are evaluated for a whole
// block of steps by one launch (stage_cotangents) into a staging ring laid
// out like the forward's (slot, term, element), from which the tiles add them
// step by step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "adjoint2d.h"
#include "common.h"
#include "reverse2d.h"
#include "tile2d_dev.h"
#include "tiled2d.h"

namespace mt {
namespace {

constexpr int kMaxRev = 1024;
constexpr int kLineTaps = 4;   // line terms a tile keeps in LDS for the whole launch

template <typename T, int TX, int TY, int NS, bool PML>
constexpr int rev_lds() {
  using S = Shape<TX, TY, NS, kMaxRev>;
  return 4 * S::RC + (PML ? 4 * S::RX : 0) + kLineTaps * NS * std::max(S::RX, S::RY);
}

// Does term t change cotangents inside [a0, a0 + RX) x [b0, b0 + RY)?
__device__ __forceinline__ bool tap_reaches(const Tap& t, int a0, int b0, int RX, int RY) {
  const int a1 = a0 + RX, b1 = b0 + RY;
  if (t.line == 1) return t.fix >= a0 && t.fix - (t.avg ? 1 : 0) < a1 && t.lo < b1 && t.lo + t.n > b0;
  if (t.line == 2) return t.fix >= b0 && t.fix - (t.avg ? 1 : 0) < b1 && t.lo < a1 && t.lo + t.n > a0;
  if (t.line == 3) return a0 < t.n0 && b0 < t.n1;
  return t.fix >= a0 && t.fix < a1 && t.lo >= b0 && t.lo < b1;
}

template <typename T, int TX, int TY, int NS, bool PML>
__device__ __forceinline__ void rev_tile(const TmRev<T>& p, const TapSet& taps, int nsub, int s_hi, int slot_hi,
                                         int tr, int tc, T* sm) {
  using S = Shape<TX, TY, NS, kMaxRev>;
  constexpr int RX = S::RX, RY = S::RY, RC = S::RC, ROWS = S::ROWS, STR = S::STR, PER = S::PER;
  constexpr int RM = RX > RY ? RX : RY;
  T *sA = sm, *sB = sm + RC, *sC = sm + 2 * RC, *sD = sm + 3 * RC;   // gHy, gHx, gEx, gEy
  T *prof = sm + 4 * RC, *inj = prof + (PML ? 4 * RX : 0);
  constexpr int PP = PML ? PER : 1;
  T vPzy[PP], vPzx[PP], vPyx[PP], vPxy[PP];
  T vE[PER], vD[PER], vHx[PER], vHy[PER], vK[PER], vG[PER], vT[PER];
  const int nx = p.nx, ny = p.ny, ny_e = p.ny_e;
  const int I0 = tr * TX, J0 = tc * TY;
  const int a0 = I0 - NS - 1, b0 = J0 - NS - 1;
  const int tid = threadIdx.x, l0 = tid / RY, lj = tid - l0 * RY;
  const int i0 = a0 + l0, j = b0 + lj, jj = j - (p.y_pmc ? 0 : 1);
  const T dt = p.dt, dx = p.dx, rdx = p.rdx;
  const bool jez = j >= 0 && j < ny, jhx = j >= 0 && j < ny - 1;
  const bool jlive = jez && jj >= 0 && jj < ny_e;
  const bool in_hy = PML && jhx && p.hy.in(j), in_ey = PML && jlive && p.ey.in(jj);
  T bhy = T(0), ahy = T(0), bey = T(0), aey = T(0);
  if constexpr (PML) {
    if (in_hy) bhy = p.hy.b[j], ahy = p.hy.a[j];
    if (in_ey) bey = p.ey.b[jj], aey = p.ey.a[jj];
    load_rows<T, RX>(p.hx, p.ex, a0, nx - 1, nx - 2, prof);
  }
  const int hx_lo = p.hx.lo_end, hx_hi = p.hx.hi_begin, ex_lo = p.ex.lo_end + 1, ex_hi = p.ex.hi_begin + 1;
  auto in_hx = [&](int i) { return i < hx_lo || i >= hx_hi; };
  auto in_ex = [&](int i) { return i < ex_lo || i >= ex_hi; };
  auto ok = [&](int u) { return tid < STR && (u < PER - 1 || l0 + u * ROWS < RX); };
  const bool jown = lj > NS && lj <= NS + TY && tid < STR && j < ny;
  auto own = [&](int u) {
    return jown && l0 + u * ROWS > NS && l0 + u * ROWS <= NS + TX && i0 + u * ROWS < nx;
  };
  const long long cells = (long long)nx * ny;
  const T* tape = p.tape + (long long)s_hi * cells;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    const bool ez = ok(u) && (!PML || (i >= 0 && i < nx && jez));
    const bool hx = ez && (!PML || jhx), hy = ez && (!PML || i < nx - 1);
    const long long e = (long long)i * ny + j;
    vE[u] = dget(p.Ez, e, ez);
    vD[u] = dget(p.Dz, e, ez);
    vHx[u] = dget(p.Hx, (long long)i * (ny - 1) + j, hx);
    vHy[u] = dget(p.Hy, e, hy);
    vK[u] = ez ? p.eps[e] : T(1);
    vG[u] = dget((const T*)p.eps_grad, e, own(u));
    vT[u] = dget(tape, e, own(u));
    if constexpr (PML) {
      const bool live = ez && i >= 1 && i < nx - 1 && jlive;
      const long long q = (long long)(i - 1) * ny_e + jj;
      vPzy[u] = dget(p.pEzy, (long long)i * (ny - 1) + j, hx && in_hy);
      vPzx[u] = dget(p.pEzx, e, hy && in_hx(i));
      vPyx[u] = dget(p.pHyx, q, live && in_ex(i));
      vPxy[u] = dget(p.pHxy, q, live && in_ey);
    }
  }
  // monitor terms that reach the region; the first few line terms' staged
  // values of every step of the launch go to LDS, where a step finds them
  // without a memory round trip
  unsigned reach = 0;
  for (int q = 0; q < taps.n; ++q)
    if (tap_reaches(taps.t[q], a0, b0, RX, RY)) reach |= 1u << q;
  {
    int slot = 0;
    for (unsigned r = reach; r; r &= r - 1) {
      const Tap& t = taps.t[__builtin_ctz(r)];
      if (t.line > 2) continue;
      if (slot == kLineTaps) break;
      const int base = t.line == 1 ? b0 : a0, len = t.line == 1 ? RY : RX;
      for (int x = tid; x < nsub * len; x += S::BLK) {
        const int s = x / len, c = x - s * len, e = base + c - t.lo;
        T v = T(0);
        if (e >= 0 && e < t.n) v = static_cast<const T*>(t.out)[(long long)(t.slot0 + slot_hi - s) * t.slot_stride + e];
        inj[(slot * NS + s) * RM + c] = v;
      }
      ++slot;
    }
  }
  __syncthreads();
  for (int s = 0; s < nsub; ++s) {
    if (reach) {   // monitor cotangents of this step, in term order
      int slot = 0;
      for (unsigned r = reach; r; r &= r - 1) {
        const Tap& t = taps.t[__builtin_ctz(r)];
        const T* st = static_cast<const T*>(t.out) + (long long)(t.slot0 + slot_hi - s) * t.slot_stride;
        const bool lds = t.line <= 2 && slot < kLineTaps;
        const int f = t.field;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          const int i = i0 + u * ROWS, li = l0 + u * ROWS;
          if (!ok(u)) continue;
          bool hit;
          int c, e;
          if (t.line == 1) {
            c = lj, e = j - t.lo;
            hit = (i == t.fix || (t.avg && i == t.fix - 1)) && e >= 0 && e < t.n;
          } else if (t.line == 2) {
            c = li, e = i - t.lo;
            hit = (j == t.fix || (t.avg && j == t.fix - 1)) && e >= 0 && e < t.n;
          } else if (t.line == 3) {
            c = 0, e = i * t.n1 + j;
            hit = i >= 0 && i < t.n0 && j >= 0 && j < t.n1;
          } else {
            c = 0, e = 0;
            hit = i == t.fix && j == t.lo;
          }
          if (!hit) continue;
          const T vb = lds ? inj[(slot * NS + s) * RM + c] : st[e];
          const T v = t.avg ? T(0.5) * vb : vb;
          if (f == 0) vE[u] = vE[u] + v;
          else if (f == 1) vHx[u] = vHx[u] + v;
          else if (f == 2) vHy[u] = vHy[u] + v;
          else vD[u] = vD[u] + v;
        }
        if (t.line <= 2) ++slot;
      }
    }
    // A: eps gradient (owned cells), Dz cotangent, H-difference cotangents
    T gy[PER], gx[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
      gy[u] = gx[u] = T(0);
      if (!ok(u)) break;
      vG[u] = vG[u] + (-vE[u] * vT[u]) / vK[u];   // stored by the owner only
      const T dzb = vD[u] + vE[u] / vK[u];
      vD[u] = dzb;
      if (!PML || (jlive && i >= 1 && i < nx - 1)) {
        const T cb = dt * dzb;
        gy[u] = cb;
        gx[u] = -cb;
        if constexpr (PML) {
          if (in_ex(i)) {
            const T pt = vPyx[u] + cb;
            gy[u] = cb + prof[3 * RX + li] * pt;
            vPyx[u] = prof[2 * RX + li] * pt;
          }
          if (in_ey) {
            const T pt = vPxy[u] - cb;
            gx[u] = -cb + aey * pt;
            vPxy[u] = bey * pt;
          }
        }
      }
      sA[c] = gy[u];
      sB[c] = gx[u];
    }
    if (s + 1 < nsub) {   // the next step's tape values, while B and C run
      tape -= cells;
#pragma unroll
      for (int u = 0; u < PER; ++u) vT[u] = dget(tape, (long long)(i0 + u * ROWS) * ny + j, own(u));
    }
    __syncthreads();
    // B: H cotangents, E-difference cotangents
    {
      T qx[PER], qy[PER];
      auto dy = [&](int u) -> T {   // Hy part
        const int i = i0 + u * ROWS;
        const bool l = ok(u) && (u < PER - 1 || l0 + u * ROWS < RX - 1) && (!PML || (jez && i >= 0 && i < nx - 1));
        return l ? gy[u] - sA[tid + u * STR + RY] : T(0);
      };
      auto dxx = [&](int u) -> T {  // Hx part
        const int i = i0 + u * ROWS;
        const bool l = ok(u) && lj < RY - 1 && (!PML || (jhx && i >= 0 && i < nx));
        return l ? gx[u] - sB[tid + u * STR + 1] : T(0);
      };
      step_quots<T, PER>(dx, rdx, dxx, dy, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int c = tid + u * STR, i = i0 + u * ROWS, li = l0 + u * ROWS;
        gy[u] = gx[u] = T(0);   // from here gEx and gEy
        if (!ok(u)) break;
        if (!PML || (jez && i >= 0 && i < nx - 1)) {
          const T hb = vHy[u] + qy[u];
          vHy[u] = hb;
          T gb = dt * hb;
          if constexpr (PML) {
            if (in_hx(i)) {
              const T pt = vPzx[u] + dt * hb;
              gb = gb + prof[RX + li] * pt;
              vPzx[u] = prof[li] * pt;
            }
          }
          gy[u] = gb;
        }
        if (!PML || (jhx && i >= 0 && i < nx)) {
          const T hb = vHx[u] + qx[u];
          vHx[u] = hb;
          T gb = -dt * hb;
          if constexpr (PML) {
            if (in_hy) {
              const T pt = vPzy[u] - dt * hb;
              gb = gb + ahy * pt;
              vPzy[u] = bhy * pt;
            }
          }
          gx[u] = gb;
        }
        sC[c] = gy[u];
        sD[c] = gx[u];
      }
    }
    __syncthreads();
    // C: Ez cotangent (gEx and gEy of cells beyond a wall are zero)
    {
      T qx[PER], qy[PER];
      auto cx = [&](int u) -> T { return ok(u) && (u > 0 || l0 >= 1) ? sC[tid + u * STR - RY] - gy[u] : T(0); };
      auto cy = [&](int u) -> T { return ok(u) && lj >= 1 ? sD[tid + u * STR - 1] - gx[u] : T(0); };
      step_quots<T, PER>(dx, rdx, cx, cy, qx, qy);
#pragma unroll
      for (int u = 0; u < PER; ++u)
        if (!PML || (i0 + u * ROWS >= 0 && i0 + u * ROWS < nx && jez)) vE[u] = qx[u] + qy[u];
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = i0 + u * ROWS;
    if (!own(u)) continue;
    const long long e = (long long)i * ny + j;
    p.eps_grad[e] = vG[u];
    p.oEz[e] = vE[u];
    p.oDz[e] = vD[u];
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

template <typename T, int TX, int TY, int NS, int MODE>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxRev>::BLK)) void tm_reverse(TmRev<T> p, TapSet taps, int nsub,
                                                                              int s_hi, int slot_hi) {
  __shared__ T sm[rev_lds<T, TX, TY, NS, MODE != kInterior>()];
  int tr, tc;
  const bool pml = pick_tile<MODE>(p.map, &tr, &tc);
  if (MODE == kRing || (MODE == kAll && pml))
    rev_tile<T, TX, TY, NS, true>(p, taps, nsub, s_hi, slot_hi, tr, tc, sm);
  else
    rev_tile<T, TX, TY, NS, false>(p, taps, nsub, s_hi, slot_hi, tr, tc, sm);
}

// Batched form: the (variant, tile) work list in XCD order, as tm_batch.
// The interior form keeps its 72 VGPRs: held to 64 (two 1024-thread
// workgroups per CU, as tm_batch_in2) it spilled and measured slower, 80 ->
// 95 us per launch of 4 steps over 10 variants of 200^2 - 900^2.
template <typename T, int TX, int TY, int NS, int MODE>
__global__ __launch_bounds__((Shape<TX, TY, NS, kMaxRev>::BLK)) void tm_reverse_batch(
    const TmRevVar<T>* vars, const int* pre_in, const int* pre_ring, int nvar, int nsub, int parity, int s_hi,
    int slot_hi) {
  __shared__ T sm[rev_lds<T, TX, TY, NS, MODE != kInterior>()];
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
    const TmRevVar<T>& V = vars[lo];
    const TmRev<T>& p = parity ? V.pB : V.pA;
    int tr, tc;
    tile_linear(ring, p.map, it - prefix[lo], &tr, &tc);
    if (MODE == kRing || (MODE == kAll && ring))
      rev_tile<T, TX, TY, NS, true>(p, V.taps, nsub, s_hi, slot_hi, tr, tc, sm);
    else
      rev_tile<T, TX, TY, NS, false>(p, V.taps, nsub, s_hi, slot_hi, tr, tc, sm);
    __syncthreads();
  }
}

// Staged cotangents of one monitor: block (elements e0.., slot) evaluates the
// phase factors of its step once per (term, frequency) into LDS and sums the
// frequencies in adj_inject_block's order, term by term.
template <typename T>
__device__ void stage_block(const mt_monitor& m, T* out, int e0, int slot, int t, double dt_d) {
  __shared__ T cs[2 * kInjTab];
  __shared__ T part[kInjS][kInjE];
  const int n = m.n0 * m.n1, nq = m.n_terms, nf = m.nfreq;
  const int el = threadIdx.x % kInjE, sl = threadIdx.x / kInjE, e = e0 + el;
  const T dt = static_cast<T>(dt_d);
  const T* om = static_cast<const T*>(m.omega);
  const T* ac = static_cast<const T*>(m.acc);
  out += (long long)slot * nq * n;
  if (nq * nf > kInjTab) {   // uniform over the block: one thread sums every frequency
    if (sl == 0 && e < n)
      for (int q = 0; q < nq; ++q) {
        const T tq = static_cast<T>(((double)t + (m.term[q].t_half ? 0.5 : 1.0)) * dt_d);
        T vb = T(0);
        for (int f = 0; f < nf; ++f) {
          const T ph = om[f] * tq;
          const T re = ac[((long long)f * 2 * nq + 2 * q) * n + e], im = ac[((long long)f * 2 * nq + 2 * q + 1) * n + e];
          vb = vb + (dt * cos(ph)) * re + (-(dt * sin(ph))) * im;
        }
        out[(long long)q * n + e] = vb;
      }
    return;
  }
  for (int x = threadIdx.x; x < nq * nf; x += kInjE * kInjS) {
    const int q = x / nf, f = x - q * nf;
    const double tt = ((double)t + (m.term[q].t_half ? 0.5 : 1.0)) * dt_d;
    const T ph = om[f] * static_cast<T>(tt);
    cs[2 * x] = dt * cos(ph);
    cs[2 * x + 1] = -(dt * sin(ph));
  }
  __syncthreads();
  for (int q = 0; q < nq; ++q) {
    T v = T(0);
    if (e < n)
      for (int f = sl; f < nf; f += kInjS) {
        const T* c = cs + 2 * (q * nf + f);
        const T re = ac[((long long)f * 2 * nq + 2 * q) * n + e], im = ac[((long long)f * 2 * nq + 2 * q + 1) * n + e];
        v = v + c[0] * re + c[1] * im;
      }
    part[sl][el] = v;
    __syncthreads();
    if (sl == 0 && e < n) {
      T vb = part[0][el];
      for (int g = 1; g < kInjS; ++g) vb = vb + part[g][el];
      out[(long long)q * n + e] = vb;
    }
    __syncthreads();
  }
}

template <typename T>
__global__ __launch_bounds__(kInjE* kInjS) void stage_cotangents(mt_monitor m, T* out, int t0, double dt) {
  stage_block<T>(m, out, blockIdx.x * kInjE, blockIdx.y, t0 + blockIdx.y, dt);
}

template <typename T>
__global__ __launch_bounds__(kInjE* kInjS) void stage_cotangents_batch(const mt_monitor* mons, void* const* stage,
                                                                      const int* pre, int nvar, int t0,
                                                                      const double* dts) {
  const int b = blockIdx.x;
  int lo = 0, hi = nvar;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (pre[mid] <= b) lo = mid;
    else hi = mid;
  }
  if (mons[lo].n_terms == 0) return;
  stage_block<T>(mons[lo], static_cast<T*>(stage[lo]), (b - pre[lo]) * kInjE, blockIdx.y, t0 + blockIdx.y, dts[lo]);
}

// Shapes of the reverse sweep: the forward's variant ids (tiled2d.hip) that
// it builds; other ids map to one of them.
template <typename T, typename F>
int with_shape(int variant, F f) {
  if constexpr (sizeof(T) == 8) {
    switch (variant) {
      case 7: return f.template go<16, 16, 6>();
      case 8: return f.template go<8, 8, 8>();
      case 9: return f.template go<16, 32, 4>();
      default: return f.template go<8, 64, 4>();
    }
  } else {
    switch (variant) {
      case 7: return f.template go<16, 16, 7>();
      case 8: return f.template go<8, 8, 8>();
      case 9: return f.template go<16, 32, 4>();
      case 5: return f.template go<32, 64, 4>();
      default: return f.template go<16, 64, 4>();
    }
  }
}

template <typename T>
struct RevLaunch {
  TmRev<T> p;
  const TapSet& taps;
  int nsub, s_hi, slot_hi;
  hipStream_t s;
  template <int TX, int TY, int NS>
  int go() {
    constexpr int BLK = Shape<TX, TY, NS, kMaxRev>::BLK;
    p.map = make_map<TX, TY, NS>(p.nx, p.ny, p.in_i0, p.in_i1, p.in_j0, p.in_j1);
    const TileMap& m = p.map;
    const int n_in = (m.r1 - m.r0) * (m.c1 - m.c0), n = m.R * m.C, n_ring = n - n_in;
    if (n <= kOneRound && n_in && n_ring) {
      hipLaunchKernelGGL((tm_reverse<T, TX, TY, NS, kAll>), dim3(n), dim3(BLK), 0, s, p, taps, nsub, s_hi, slot_hi);
      return MT_OK;
    }
    if (n_in)
      hipLaunchKernelGGL((tm_reverse<T, TX, TY, NS, kInterior>), dim3(n_in), dim3(BLK), 0, s, p, taps, nsub, s_hi,
                         slot_hi);
    if (n_ring)
      hipLaunchKernelGGL((tm_reverse<T, TX, TY, NS, kRing>), dim3(n_ring), dim3(BLK), 0, s, p, taps, nsub, s_hi,
                         slot_hi);
    return MT_OK;
  }
};

struct StepsOf {
  template <int TX, int TY, int NS>
  int go() { return NS; }
};

struct MapOf {
  int nx, ny, i0, i1, j0, j1;
  TileMap* m;
  template <int TX, int TY, int NS>
  int go() {
    *m = make_map<TX, TY, NS>(nx, ny, i0, i1, j0, j1);
    return 0;
  }
};

template <typename T>
struct RevBatchLaunch {
  const TmRevVar<T>* vars;
  const int *pre_in, *pre_ring;
  int nvar, n_in, n_ring, grid, nsub, parity, s_hi, slot_hi;
  hipStream_t s;
  template <int TX, int TY, int NS>
  int go() {
    constexpr int BLK = Shape<TX, TY, NS, kMaxRev>::BLK;
    const int n = n_in + n_ring;
    if (n <= kOneRound && n_in && n_ring) {
      hipLaunchKernelGGL((tm_reverse_batch<T, TX, TY, NS, kAll>), dim3(one_round_grid(n)), dim3(BLK), 0, s, vars, pre_in,
                         pre_ring, nvar, nsub, parity, s_hi, slot_hi);
      return MT_OK;
    }
    if (n_in)
      hipLaunchKernelGGL((tm_reverse_batch<T, TX, TY, NS, kInterior>), dim3(std::min(one_round_grid(n_in), grid)), dim3(BLK), 0, s,
                         vars, pre_in, pre_ring, nvar, nsub, parity, s_hi, slot_hi);
    if (n_ring)
      hipLaunchKernelGGL((tm_reverse_batch<T, TX, TY, NS, kRing>), dim3(std::min(one_round_grid(n_ring), grid)), dim3(BLK), 0, s,
                         vars, pre_in, pre_ring, nvar, nsub, parity, s_hi, slot_hi);
    return MT_OK;
  }
};

}  // namespace

bool rev_terms_ok(const mt_monitor* mons, int n) {
  int taps = 0;
  for (int i = 0; i < n; ++i)
    for (int q = 0; q < mons[i].n_terms; ++q) {
      if (++taps > kMaxTaps) return false;
      const mt_dft_term& t = mons[i].term[q];
      if (t.line < 1 || t.line > 4 || t.field < 0 || t.field > 3 || (t.b && t.line > 2)) return false;
    }
  return true;
}

int rev_steps(int dtype, int variant) {
  return dtype == MT_F64 ? with_shape<double>(variant, StepsOf{}) : with_shape<float>(variant, StepsOf{});
}

TileMap rev_map(int dtype, int variant, int nx, int ny, int i0, int i1, int j0, int j1) {
  TileMap m{};
  const MapOf f{nx, ny, i0, i1, j0, j1, &m};
  dtype == MT_F64 ? with_shape<double>(variant, f) : with_shape<float>(variant, f);
  return m;
}

template <typename T>
TmRev<T> make_rev(const mt_tm2d* d, const mt_tm2d_adj* r, const mt_tm2d_adj* w, const void* tape) {
  TmRev<T> p{};
  p.nx = d->nx;
  p.ny = d->ny;
  p.y_pmc = d->y_pmc;
  p.ny_e = d->y_pmc ? d->ny : d->ny - 2;
  p.dt = static_cast<T>(d->dt);
  p.dx = static_cast<T>(d->dx);
  p.rdx = const_div_recip<T>(p.dx);
  p.eps = static_cast<const T*>(d->eps);
  p.hy = pml_of<T>(d->hy);
  p.hx = pml_of<T>(d->hx);
  p.ex = pml_of<T>(d->ex);
  p.ey = pml_of<T>(d->ey);
  tm_interior(d, &p.in_i0, &p.in_i1, &p.in_j0, &p.in_j1);
  p.Ez = static_cast<const T*>(r->aEz), p.Dz = static_cast<const T*>(r->aDz);
  p.Hx = static_cast<const T*>(r->aHx), p.Hy = static_cast<const T*>(r->aHy);
  p.pEzy = static_cast<const T*>(r->apsi_Ezy), p.pEzx = static_cast<const T*>(r->apsi_Ezx);
  p.pHyx = static_cast<const T*>(r->apsi_Hyx), p.pHxy = static_cast<const T*>(r->apsi_Hxy);
  p.oEz = static_cast<T*>(w->aEz), p.oDz = static_cast<T*>(w->aDz);
  p.oHx = static_cast<T*>(w->aHx), p.oHy = static_cast<T*>(w->aHy);
  p.oEzy = static_cast<T*>(w->apsi_Ezy), p.oEzx = static_cast<T*>(w->apsi_Ezx);
  p.oHyx = static_cast<T*>(w->apsi_Hyx), p.oHxy = static_cast<T*>(w->apsi_Hxy);
  p.eps_grad = static_cast<T*>(r->eps_grad);
  p.tape = static_cast<const T*>(tape);
  return p;
}
template TmRev<float> make_rev<float>(const mt_tm2d*, const mt_tm2d_adj*, const mt_tm2d_adj*, const void*);
template TmRev<double> make_rev<double>(const mt_tm2d*, const mt_tm2d_adj*, const mt_tm2d_adj*, const void*);

int copy_cotangents(const mt_tm2d* d, const mt_tm2d_adj* dst, const mt_tm2d_adj* src, size_t es, hipStream_t s) {
  const size_t nx = d->nx, ny = d->ny, nye = d->y_pmc ? d->ny : d->ny - 2;
  const size_t n[8] = {nx * ny, nx * ny, nx * (ny - 1), (nx - 1) * ny, nx * (ny - 1), (nx - 1) * ny, (nx - 2) * nye,
                       (nx - 2) * nye};
  void* D[8] = {dst->aEz, dst->aDz, dst->aHx, dst->aHy, dst->apsi_Ezy, dst->apsi_Ezx, dst->apsi_Hyx, dst->apsi_Hxy};
  void* R[8] = {src->aEz, src->aDz, src->aHx, src->aHy, src->apsi_Ezy, src->apsi_Ezx, src->apsi_Hyx, src->apsi_Hxy};
  for (int q = 0; q < 8; ++q)
    if (hipMemcpyAsync(D[q], R[q], n[q] * es, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return fail(MT_EHIP, "adjoint: copy back failed");
  return MT_OK;
}

template <typename T>
int rev_batch_run(const RevBatchArgs& a, const RevPart& part, int parity, hipStream_t s) {
  return with_shape<T>(a.variant,
                       RevBatchLaunch<T>{static_cast<const TmRevVar<T>*>(a.vars), a.pre_in, a.pre_ring, a.nvar,
                                         a.n_in, a.n_ring, a.grid, part.nsub, parity, part.s_hi,
                                         part.s_hi - part.lo, s});
}
template int rev_batch_run<float>(const RevBatchArgs&, const RevPart&, int, hipStream_t);
template int rev_batch_run<double>(const RevBatchArgs&, const RevPart&, int, hipStream_t);

template <typename T>
void rev_batch_stage(const mt_monitor* mons, void* const* stage, const int* pre, int nblocks, int nvar, int t0,
                     int nslots, const double* dts, hipStream_t s) {
  hipLaunchKernelGGL(stage_cotangents_batch<T>, dim3(nblocks, nslots), dim3(kInjE * kInjS), 0, s, mons, stage, pre,
                     nvar, t0, dts);
}
template void rev_batch_stage<float>(const mt_monitor*, void* const*, const int*, int, int, int, int, const double*,
                                     hipStream_t);
template void rev_batch_stage<double>(const mt_monitor*, void* const*, const int*, int, int, int, int, const double*,
                                      hipStream_t);

namespace {

template <typename T>
int reverse_t(const mt_tm2d* d, const mt_tm2d_adj* a, const mt_tm2d_adj* b, const void* tape, const MonitorPlan& mp,
              int step0, int k, hipStream_t s) {
  TmRev<T> P[2] = {make_rev<T>(d, a, b, tape), make_rev<T>(d, b, a, tape)};
  P[1].eps_grad = P[0].eps_grad;
  const int dtype = sizeof(T) == 8 ? MT_F64 : MT_F32;
  const int S = mp.n_mons ? mp.stage_steps : k;
  int par = 0, rc;
  for (const RevPart& part : rev_schedule(k, S, rev_steps(dtype, d->variant))) {
    if (part.stage) {   // the block's monitor cotangents
      char* base = static_cast<char*>(mp.stage);
      long long off = 0;
      for (int i = 0; i < mp.n_mons; ++i) {
        const mt_monitor& m = mp.mons[i];
        if (m.kind != 0) continue;
        const long long n = (long long)m.n0 * m.n1;
        if (n)
          hipLaunchKernelGGL(stage_cotangents<T>, dim3((unsigned)((n + kInjE - 1) / kInjE), part.stage),
                             dim3(kInjE * kInjS), 0, s, m, reinterpret_cast<T*>(base + off), step0 + part.lo, d->dt);
        off += ((long long)mp.stage_steps * m.n_terms * n + (long long)m.nfreq * mp.stage_steps * 4) * sizeof(T);
      }
    }
    TapSet taps;
    taps.n = 0;
    if (mp.n_mons && !build_taps(mp, 0, part.lo, sizeof(T), &taps))
      return fail(MT_EINVAL, "reverse sweep: monitor terms without a field position");
    with_shape<T>(d->variant, RevLaunch<T>{P[par], taps, part.nsub, part.s_hi, part.s_hi - part.lo, s});
    par ^= 1;
    if ((rc = check_launch("tm2d reverse sweep"))) return rc;
  }
  return par ? copy_cotangents(d, a, b, sizeof(T), s) : MT_OK;
}

bool adj_complete(const mt_tm2d_adj* a) {
  return a->aEz && a->aDz && a->aHx && a->aHy && a->apsi_Ezy && a->apsi_Ezx && a->apsi_Hyx && a->apsi_Hxy;
}

}  // namespace
}  // namespace mt

using namespace mt;

extern "C" int mt_tm2d_adjoint_tiles_ok(const mt_monitor* mons, int n_mons) {
  return n_mons == 0 || (mons && n_mons > 0 && rev_terms_ok(mons, n_mons)) ? 1 : 0;
}

extern "C" int mt_tm2d_adjoint_tiled(const mt_tm2d* p, const mt_tm2d_adj* a, const mt_tm2d_adj* b, const void* tape,
                                     const mt_monitor* mons, int n_mons, void* stage, long long stage_bytes,
                                     int stage_steps, int step0, int k, void* stream) {
  if (!p || !a || !b) return fail(MT_EINVAL, "null problem or adjoint state");
  if (p->nx < 3 || p->ny < 3) return fail(MT_EINVAL, "grid must be at least 3x3");
  if (k < 0) return fail(MT_EINVAL, "negative step count");
  if (k > 0 && !tape) return fail(MT_EINVAL, "adjoint needs the forward Ez tape");
  if (p->dtype != MT_F32 && p->dtype != MT_F64) return fail(MT_EINVAL, "dtype must be f32 or f64");
  if (!p->eps || !adj_complete(a) || !adj_complete(b) || !a->eps_grad) return fail(MT_EINVAL, "null adjoint pointer");
  if (p->n_poles || p->kerr || p->d1 || p->h1x || p->n_mpoles || p->y_mirror || p->x_mirror || p->y_rot2 || p->rot4)
    return fail(MT_EINVAL, "the tiled reverse sweep carries no media and no symmetry cuts");
  int rc;
  if ((rc = check_axis(p->hy, p->ny - 1, "hy")) || (rc = check_axis(p->hx, p->nx - 1, "hx")) ||
      (rc = check_axis(p->ex, p->nx - 2, "ex")) || (rc = check_axis(p->ey, p->y_pmc ? p->ny : p->ny - 2, "ey")))
    return rc;
  if (!rev_terms_ok(mons, n_mons)) return fail(MT_EINVAL, "reverse sweep: monitor terms without a field position");
  MonitorPlan mp{mons, n_mons, stage, stage_bytes, stage_steps > 0 ? stage_steps : 1, p->dtype};
  if ((rc = monitors_validate(mp))) return rc;
  if (k == 0) return MT_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return p->dtype == MT_F64 ? reverse_t<double>(p, a, b, tape, mp, step0, k, s)
                            : reverse_t<float>(p, a, b, tape, mp, step0, k, s);
}
