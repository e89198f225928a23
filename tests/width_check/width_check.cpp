// Host check of the batch's choice of workgroup width (cuopt_amd/csrc/batch_width.hpp), built
// by tests/test_batch_width.py: batches whose launch was measured in both widths get the
// faster one.
#include <cstdio>
#include <vector>

#include "batch_width.hpp"

using namespace cuopt_amd;

static int fails = 0;
#define CHECK(c)                                       \
  do {                                                 \
    if (!(c)) {                                        \
      std::printf("FAIL line %d: %s\n", __LINE__, #c); \
      ++fails;                                         \
    }                                                  \
  } while (0)

// Row blocks of one matrix of `rows` rows in a workgroup of `lanes` lanes, 2 lanes to a row of
// A (20 nonzeros) and one to a row of A^T (8), blocks of 2 552 or 5 112 nonzeros.
static int blocks(int m, int lanes)
{
  const int n = 5 * m / 2, most = lanes == 256 ? 2552 : 5112;
  const int a = std::min(lanes / 2, most / 20), t = std::min(lanes, most / 8);
  return (m + a - 1) / a + (n + t - 1) / t;
}

// `count` LPs of m rows, 2.5 m columns and 8 nonzeros a column on 256 CUs.
static BatchLp lp(int m) { return {20 * m, blocks(m, 256), blocks(m, 768)}; }
static bool wide(int m, int count, bool fp32) { return prefer_wide(std::vector<BatchLp>(count, lp(m)), 256, fp32); }

int main()
{
  // a batch just past 256 LPs: wide ones need a second turn of the chip
  CHECK(!wide(120, 300, true) && !wide(300, 300, true) && !wide(300, 384, true));
  CHECK(wide(140, 300, false) && wide(160, 330, false) && wide(500, 300, true) && wide(500, 400, false));
  // one turn of the chip, and large LPs whose longest sets the time
  for (bool fp32 : {false, true}) {
    CHECK(wide(140, 200, fp32) && wide(300, 256, fp32) && wide(800, 300, fp32) && wide(800, 400, fp32));
    // many LPs: the sum over the chip counts
    CHECK(!wide(300, 512, fp32) && !wide(200, 900, fp32) && !wide(300, 4096, fp32));
    // LPs that do not gain (a block of each matrix), and no LPs
    CHECK(!wide(102, 8, fp32) && wide(103, 8, fp32));
    CHECK(!prefer_wide({}, 256, fp32) && !prefer_wide({{0, 2, 2}}, 256, fp32));
    // the order of the LPs does not matter
    std::vector<BatchLp> up, down;
    for (int i = 0; i < 1024; ++i) up.push_back(lp(50 + i));
    down.assign(up.rbegin(), up.rend());
    CHECK(prefer_wide(up, 256, fp32) == prefer_wide(down, 256, fp32));
  }
  std::printf("%s\n", fails ? "failed" : "OK");
  return fails != 0;
}
