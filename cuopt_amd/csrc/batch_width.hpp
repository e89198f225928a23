// batch_width.hpp -- which LPs of a batch get wide workgroups (batch_solver.hip).
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace cuopt_amd {

// An LP as the choice sees it: the row blocks of its two matrices in a narrow and in a wide
// workgroup, what an iteration walks one after the other.
struct BatchLp {
  int nnz, narrow, wide;
};

// Whether an iteration of an LP takes less time in a wide workgroup: not that of a small
// one, nor one whose matrices are a block each in a narrow workgroup already.  m rows, 2.5 m
// columns, FP64, narrow / wide: 128 LPs of m 101 (a block each) 12.7 / 13.2 ms; 64 LPs of m 120
// (two blocks of A^T) 15.3 / 13.7 ms, of m 140 16.7 / 12.5 ms.
inline bool gains_from_width(int nnz, int narrow_blocks) { return nnz >= 2000 && narrow_blocks > 2; }

// Estimated time of a batch's launch (of no particular unit).  lps: in the order in which they
// start, the first nwide in wide workgroups.  Each takes the first CU, or half a CU when
// narrow, that is free.  An iteration's time goes by the LP's row blocks; how many iterations
// an LP takes is not known, so the LPs are spread over the usual law of them, most near the
// mean and a few at twice it (u in [0, 1) by reversing the bits of the position).
inline double batch_launch_time(const std::vector<BatchLp>& lps, size_t nwide, int cus, bool fp32)
{
  std::vector<double> free_at(cus, 0.0);  // a heap, the first to be free on top
  double end  = 0.0;
  auto run_on = [&](size_t i, double step) {
    uint32_t r = (uint32_t)i + 1;
    r = (r & 0x55555555u) << 1 | (r >> 1 & 0x55555555u);
    r = (r & 0x33333333u) << 2 | (r >> 2 & 0x33333333u);
    r = (r & 0x0f0f0f0fu) << 4 | (r >> 4 & 0x0f0f0f0fu);
    r = r << 24 | (r & 0xff00u) << 8 | (r >> 8 & 0xff00u) | r >> 24;
    const double u = r * 0x1p-32, steps = fp32 ? 0.8 + 1.3 * u * u * u : 0.65 + 1.6 * u * u * u * u * u;
    const double t = free_at[0] + step * steps;
    end            = std::max(end, t);
    size_t at      = 0;
    for (size_t c; (c = 2 * at + 1) < free_at.size(); at = c) {  // t in place of the top, sifted down
      if (c + 1 < free_at.size() && free_at[c + 1] < free_at[c]) ++c;
      if (free_at[c] >= t) break;
      free_at[at] = free_at[c];
    }
    free_at[at] = t;
  };
  size_t i = 0;
  for (; i < nwide; ++i) run_on(i, fp32 ? 2.8 + 2.8 * lps[i].wide : 3.1 + 2.45 * lps[i].wide);
  std::sort(free_at.begin(), free_at.end());  // halves of the CUs, in order: a heap as well
  free_at.resize(2 * cus);
  for (int c = 2 * cus; c-- > 0;) free_at[c] = free_at[c / 2];
  for (; i < lps.size(); ++i) run_on(i, (fp32 ? 1.4 : 2.3) + 2.4 * lps[i].narrow);
  return end;
}

// Whether the LPs that gain get wide workgroups.  A wide workgroup ends sooner and takes
// twice the share of the chip: few LPs wait for the largest of them, many for the sum, and
// a few more than the chip holds at once (256 wide, 512 narrow) need a second turn when wide.
// Launch, ms, narrow / wide, for LPs of one size (8 nonzeros per column, 2.5 columns per row):
//   rows x LPs    FP32-mixed      FP64               rows x LPs     FP32-mixed      FP64
//   140 x 200    13.1 /  10.0   20.3 /  15.2         500 x 300    34.6 /  31.9    64.3 /  47.3
//   140 x 300    14.5 /  15.2   20.3 /  17.5         800 x 300    62.1 /  49.6     138 /  90.2
//   300 x 256    21.6 /  17.9   32.9 /  26.8         800 x 512    64.8 /  60.7     145 /   101
//   300 x 384    22.0 /  26.2   34.1 /  37.7         800 x 800    94.9 /  97.3     176 /   161
//   300 x 900    36.4 /  46.9   54.8 /  61.5        1300 x 512     116 /   101     260 /   221
// The estimate's constants are fitted to 112 batches in each precision, uniform and mixed: the
// choice takes 0.3 % longer than the better one on average and at most 12 % (512 LPs of
// 1 300 rows in FP32-mixed, narrow), and at most 4 % longer than narrow workgroups.
inline bool prefer_wide(std::vector<BatchLp> lps, int cus, bool fp32)
{
  std::sort(lps.begin(), lps.end(), [](const BatchLp& x, const BatchLp& y) { return x.nnz > y.nnz; });
  const std::vector<BatchLp> all_narrow = lps;
  const auto gains = [](const BatchLp& l) { return gains_from_width(l.nnz, l.narrow); };
  const size_t nwide = std::stable_partition(lps.begin(), lps.end(), gains) - lps.begin();
  if (nwide == 0) return false;
  return batch_launch_time(lps, nwide, cus, fp32) < batch_launch_time(all_narrow, 0, cus, fp32);
}

}  // namespace cuopt_amd
