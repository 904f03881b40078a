// Checks csrc/schedule.h over all cases of a range; prints the first failure
// and exits 1.
#include <cstdio>
#include <cstdlib>

#include "schedule.h"

using namespace mt;

static void die(const char* what, int a, int b, int c) {
  std::printf("%s: %d %d %d\n", what, a, b, c);
  std::exit(1);
}

// every item dealt once; within one_round_grid no workgroup takes two
static void deal(int grid, int total, bool one) {
  std::vector<int> seen(total, 0);
  for (int b = 0; b < grid; ++b) {
    const XcdItems it = xcd_items(b, grid, total);
    int n = 0;
    for (int i = it.first; i < it.end; i += it.stride, ++n) {
      if (i < 0 || i >= total) die("item out of range", grid, total, i);
      ++seen[i];
    }
    if (one && n > 1) die("workgroup with two items", grid, total, b);
  }
  for (int i = 0; i < total; ++i)
    if (seen[i] != 1) die("item not dealt once", grid, total, i);
}

int main() {
  for (int n = 1; n <= 1100; ++n) deal(one_round_grid(n), n, true);
  for (int n = 1; n <= 256; ++n)
    if (one_round_grid(n) > 256) die("more workgroups than compute units", n, one_round_grid(n), 0);
  for (int grid : {8, 64, 256, 1024})
    for (int n : {1, 7, 9, 255, 257, 1000, 1025, 4099, 33000}) deal(grid, n, false);
  // 3D rows: at most 256 threads, no lane of a whole column of workgroups idle
  for (int f64 = 0; f64 < 2; ++f64)
    for (int ny : {3, 40, 700, 200000, 262140})
      for (int nz = 3; nz <= 1100; ++nz) {
        const Rows3 r = rows3(ny, nz, f64);
        if (r.bx < 1 || r.by < 1 || r.bx * r.by > kBlock3 || (ny + r.by - 1) / r.by > 65535) die("3D rows", ny, nz, f64);
        if (ny < 1000 && (nz + r.bx - 1) / r.bx * r.bx - nz >= std::max(r.bx, 64)) die("3D rows idle", ny, nz, f64);
      }
  const int rows[][3] = {{40, 40, 40},   {56, 64, 64},   {72, 72, 72},    {128, 128, 128}, {144, 72, 72},
                         {192, 64, 64},  {220, 110, 110}, {240, 64, 120}, {256, 64, 64},   {257, 128, 64},
                         {300, 128, 64}, {330, 128, 128}, {384, 128, 128}, {400, 64, 64}, {448, 64, 64}, {500, 128, 128},
                         {512, 128, 128}, {576, 64, 64}};
  for (const auto& r : rows)
    if (rows3(90, r[0], false).bx != r[1] || rows3(90, r[0], true).bx != r[2]) die("3D row rule", r[0], r[1], r[2]);
  for (int NS = 1; NS <= 8; ++NS)
    for (int S : {1, 2, 3, 5, 7, 8, 20, 64})
      for (int k = 1; k <= 210; ++k) {
        // forward: steps add up, no launch longer than NS or across a staging
        // block, an even number of launches if one has more than one step
        LaunchSteps ls(k, S, NS);
        int done = 0, n = 0, longest = 0;
        while (done < k) {
          const int s = ls.next();
          if (s < 1 || s > NS) die("launch length", k, S, NS);
          if (done / S != (done + s - 1) / S) die("launch crosses a staging block", k, S, NS);
          done += s;
          longest = std::max(longest, s);
          ++n;
        }
        if (done != k) die("steps do not add up", k, S, NS);
        if (n % 2 && longest > 1) die("odd number of launches", k, S, NS);
        // reverse: the same, downwards, every block staged by its first launch
        int hi = k - 1, lo = -1, m = 0;
        longest = 0;
        for (const RevPart& p : rev_schedule(k, S, NS)) {
          if (p.s_hi != hi || p.nsub < 1 || p.nsub > NS || p.s_hi - p.nsub + 1 < p.lo) die("reverse launch", k, S, NS);
          if ((p.stage > 0) != (lo != p.lo)) die("block not staged by its first launch", k, S, NS);
          if (p.stage && (p.stage > S || p.lo + p.stage - 1 != p.s_hi)) die("staged slots", k, S, NS);
          lo = p.lo;
          hi -= p.nsub;
          longest = std::max(longest, p.nsub);
          ++m;
        }
        if (hi != -1) die("reverse steps do not add up", k, S, NS);
        if (m % 2 && longest > 1) die("odd number of reverse launches", k, S, NS);
      }
  return 0;
}
