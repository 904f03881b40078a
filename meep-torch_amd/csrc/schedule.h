// How the tiled runners cut a run into launches and deal a launch's items to
// workgroups: plain C++, so that a host program can check every case.
#pragma once
#include <algorithm>
#include <vector>

namespace mt {

// Items of workgroup `block` of a launch of `grid` workgroups over `total`
// items: first, first + stride, ... below end.  Workgroups are dealt to the
// eight XCDs round robin, so the blocks of XCD x (block % 8 == x) share the
// contiguous range [x * chunk, (x + 1) * chunk): neighbouring tiles, whose
// halos overlap, run on the same XCD (same L2) at about the same time.
struct XcdItems {
  int first, end, stride;
};
constexpr XcdItems xcd_items(int block, int grid, int total) {
  const int x = block & 7, chunk = (total + 7) >> 3, end = (x + 1) * chunk;
  return XcdItems{x * chunk + (block >> 3), end < total ? end : total, (grid - x + 7) >> 3};
}
constexpr int kOneRound = 256;   // compute units: tiles that run side by side (tune.py's ROUND)

// Workgroups of a launch over n items in which no workgroup takes two: every
// XCD gets as many as its range has items (with n workgroups some XCDs have
// one fewer than items, and the launch lasts two tiles instead of one); those
// without an item leave at once.  336 x 310 and 392 x 448 in FP32 (146 tiles),
// forward and gradient over 400 steps: 13.14 -> 9.89 ms.
constexpr int one_round_grid(int n) { return (n + 7) / 8 * 8; }

// Rows of a workgroup of the 3D per-cell kernels: bx cells along k (contiguous)
// by as many rows as 256 threads hold; waves run on from one row into the next.
// Wide rows read a row's cache lines in fewer workgroups (no array starts its
// rows on a line) and leave few lanes idle.
//   nz <= 128      one row (rows of 52 to 63 cells as 64, four either way)
//   nz <= 256      two equal rows; 64-cell rows where they fit exactly, and in
//                  FP32 above 224, where they pad by less than an eighth
//   above          128-cell rows; 64-cell rows at odd multiples of 64, above 384
//                  where 128-cell rows pad by an eighth or more, and in FP64 up to 320
// Forward steps over 160 x 150 x nz, 20 steps, us, 64 x 4 rows / this.  FP32: nz
// 40 759 / 677, 72 1357 / 1008, 96 1416 / 1189, 128 1600 / 1466, 144 1936 /
// 1852, 170 2159 / 2050, 200 2396 / 2396, 220 2481 / 2513, 257 2674 / 2587, 300 3387 /
// 3129, 330 3913 / 3513, 384 3927 / 3783, 512 5271 / 5127, 640 6342 / 6099; FP64:
// 72 2028 / 1477, 128 2457 / 2348, 200 5111 / 4590, 240 5493 / 4937, 330 7226 /
// 6926, 512 10940 / 10038.  64-cell
// rows where they stay: FP32 240 2445 (two rows 2572), 256, 448 4527 (four equal
// rows 4876, 128-cell rows 4943), 704 6809 (7064), 576 equal; FP64 257 5476 (128-cell rows
// 5552), 300 6210 (three equal rows 6781, 128-cell rows 6292), 448 8551 (9572,
// 9753); 100 x 90 x 400 1713 (128-cell rows 1788).
// 384^3 in FP32, timed in turn: 46.09 -> 45.88 ms for 40 steps.
constexpr int kBlock3 = 256;
struct Rows3 {
  int bx, by;
};
constexpr Rows3 rows3(int ny, int nz, bool f64) {
  int bx = nz <= 128 ? nz : nz <= 256 ? (nz + 1) / 2 : 128;
  const int pad = (nz + 127) / 128 * 128 - nz;
  if (nz % 128 == 64 || nz == 256 || (!f64 && nz > 224 && nz < 256) || (f64 && nz > 256 && nz <= 320) ||
      (nz > 384 && 8 * pad >= nz + pad))
    bx = nz > 128 ? 64 : bx;
  const int by = kBlock3 / bx;
  if (by == 4 || (ny + by - 1) / by > 65535) return Rows3{64, 4};
  return Rows3{bx, by};
}

// Steps of each launch of a run of k steps: blocks of S steps (the monitors'
// staging ring; S = k without monitors), NS per launch, the first launch of
// several steps cut in two where the number would be odd, so that a run ends
// in the buffers it began in.  The copy back that an odd number needs moves
// eight arrays per grid, about the bytes of a launch, in eight (or, batched,
// eight per variant) dependent copies of 3 us or more; a launch of half the
// steps costs little over half.
// Ten variants of 200 to 900 cells a side, forward and gradient over 400
// steps in segments of 100: 50.4 -> 49.2 ms; 100 x 60 in FP64, 400 steps: 1.58 -> 1.56.
struct LaunchSteps {
  int NS, S, left, slot = 0, rest = 0;
  bool cut;
  LaunchSteps(int k, int S_, int NS_) : NS(NS_), S(S_), left(k) {
    const long long n = S > 0 ? (long long)(k / S) * ((S + NS - 1) / NS) + (k % S + NS - 1) / NS : 0;
    cut = n % 2 != 0;
  }
  int next() {
    int n = rest ? rest : std::min(NS, std::min(left, S - slot));
    rest = 0;
    if (cut && n > 1) {
      rest = n / 2;
      n -= rest;
      cut = false;
    }
    left -= n;
    slot = (slot + n) % S;
    return n;
  }
};

// One launch of a sweep: steps s_hi, s_hi - 1, ... (nsub of them) of the
// staging block that starts at step lo; stage > 0: fill the block's first
// `stage` slots before the launch.
struct RevPart {
  int s_hi, nsub, lo, stage;
};
// Launch lengths of a sweep over k steps in blocks of S staged steps: NS steps
// each, an even number of launches where one of them has several steps to
// give (the sets alternate, so the cotangents then end where they began).
inline std::vector<RevPart> rev_schedule(int k, int S, int NS) {
  std::vector<RevPart> v;
  for (int hi = k - 1; hi >= 0;) {
    const int lo = std::max(0, hi + 1 - S);
    for (int s = hi; s >= lo;) {
      const int n = std::min(NS, s - lo + 1);
      v.push_back(RevPart{s, n, lo, s == hi ? hi - lo + 1 : 0});
      s -= n;
    }
    hi = lo - 1;
  }
  if (v.size() % 2 && k > 1)
    for (size_t q = 0; q < v.size(); ++q)
      if (v[q].nsub > 1) {
        RevPart b = v[q];
        v[q].nsub = b.nsub / 2;
        b.s_hi -= v[q].nsub;
        b.nsub -= v[q].nsub;
        b.stage = 0;
        v.insert(v.begin() + q + 1, b);
        break;
      }
  return v;
}

}  // namespace mt
