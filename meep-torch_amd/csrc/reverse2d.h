// Argument blocks and host helpers of the temporally blocked reverse TM sweep
// (reverse2d.hip), shared with the batched runner (batch2d.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "common.h"
#include "tiled2d.h"

namespace mt {

// One orientation of the two cotangent sets: reads Ez.., writes oEz...
template <typename T>
struct TmRev {
  int nx, ny, y_pmc, ny_e;
  int in_i0, in_i1, in_j0, in_j1;
  TileMap map;
  T dt, dx, rdx;
  const T* eps;
  Pml<T> hy, hx, ex, ey;
  const T *Ez, *Dz, *Hx, *Hy, *pEzy, *pEzx, *pHyx, *pHxy;
  T *oEz, *oDz, *oHx, *oHy, *oEzy, *oEzx, *oHyx, *oHxy;
  T* eps_grad;
  const T* tape;   // Ez after every step of the call, slot s = step s
};

template <typename T>
struct TmRevVar {
  TmRev<T> pA, pB;
  TapSet taps;
};

// At most kMaxTaps terms, each with a field position the reverse tiles know (averages of lines only).
bool rev_terms_ok(const mt_monitor* mons, int n);
int rev_steps(int dtype, int variant);
TileMap rev_map(int dtype, int variant, int nx, int ny, int i0, int i1, int j0, int j1);
template <typename T>
TmRev<T> make_rev(const mt_tm2d* d, const mt_tm2d_adj* r, const mt_tm2d_adj* w, const void* tape);
int copy_cotangents(const mt_tm2d* d, const mt_tm2d_adj* dst, const mt_tm2d_adj* src, size_t es, hipStream_t s);

struct RevBatchArgs {
  const void* vars;   // TmRevVar<T>[nvar], device
  const int *pre_in, *pre_ring;
  int nvar, variant, n_in, n_ring, grid;
};
template <typename T>
int rev_batch_run(const RevBatchArgs& a, const RevPart& part, int parity, hipStream_t s);
template <typename T>
void rev_batch_stage(const mt_monitor* mons, void* const* stage, const int* pre, int nblocks, int nvar, int t0,
                     int nslots, const double* dts, hipStream_t s);

}  // namespace mt
