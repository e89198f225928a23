// unrolled.hip -- differentiable unrolled PDHG over a batch of objectives (gfx950).
//
// Forward: K steps of the PDHG iteration of the LP path (projections of
// pdhg.cu:431-545, reflection x-bar = 2 x+ - x) for B right-hand sides at once,
// with a ridge term lam/2 ||x||^2 whose proximal step divides by 1 + tau lam:
//
//   x+ = clamp((x - tau (c - A^T y)) / (1 + tau lam), l, u)
//   y+ = sigma (t - clamp(t, -u_c, -l_c)),   t = y / sigma - A (2 x+ - x)
//
// tau = sigma = eta = 0.998 / sigma_max(A) (the power iteration of
// compute_initial_step_size, pdlp.cu:2622-2738, on the unscaled matrix), no
// restarts: x_K is a piecewise-linear function of (c, l_c, u_c).
//
// Backward: the vector-Jacobian product runs the steps in reverse with the
// clamp states of x+ and y+ (transposed SpMV plus projection masks).  States
// are checkpointed every `every` steps during the forward pass; each segment is
// recomputed from its checkpoint before its reverse sweep.  The c and (l_c, u_c)
// gradients are accumulated in FP64 (in FP32 runs per segment in FP32, then
// added into the FP64 totals).
//
// Layout: the caller's vectors are batch-interleaved (v[i * B + b]); the working ones
// are cut into slabs of W batch members, v[(s * rows + i) * W + w] for member
// s * W + w, so that the rows of one slab's operand (64 bytes each for the usual W)
// fit one XCD's L2.  The last slab stores only the members that the batch has (slabs_of),
// with rows of their width.  A launch gives each XCD a contiguous run of (slab, row block)
// items, so an XCD gathers from one slab or two.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "batch_size.hpp"
#include "common.hpp"
#include "pdlp_kernels.hpp"
#include "unrolled.hpp"

namespace cuopt_amd {

namespace {

constexpr int kUB        = 256;  // 4 wavefronts per workgroup
constexpr unsigned kXcds = 8;    // the XCDs, which take the workgroups of a launch in turn

// ---- SpMM over slabs -----------------------------------------------------------
//
// A group of LW lanes owns one matrix row of one slab; a lane carries VW of the
// slab's W = LW * VW members.  The group loads its row's indices and values LW at a
// time, one per lane, and hands them round with DPP moves; each nonzero then gathers
// W contiguous values of the operand, VW per lane.
//
// Gathers of W contiguous values use the lanes that a wavefront per row leaves idle below
// 64 members, and a slab's operand is smaller than the whole: at 20 000 x 50 000 and
// B = 64 in FP32 slabs of 32 cut the dual step's L2 misses from 733 k to 607 k lines.
template <int LW_, int VW_, bool BIG_, int SHORT_>
struct Lanes {
  static constexpr int LW = LW_;             // lanes per row
  static constexpr int VW = VW_;             // members per lane
  static constexpr bool BIG = BIG_;          // 64-bit gather offsets
  static constexpr int SHORT = SHORT_;       // 2 or 4: no row has more nonzeros; 0: any length
  static constexpr int W  = LW_ * VW_;       // members per slab
  static constexpr int rows_per_wg = kUB / LW_;
};

// Lanes and members per lane of a call.
enum class Shape { k4x1, k8x1, k16x1, k8x2, k8x4 };

inline int slab_width(Shape s)
{
  return s == Shape::k4x1 ? 4 : s == Shape::k8x1 ? 8 : s == Shape::k8x4 ? 32 : 16;
}

// The shape of a call.  Up to 4 members: 8 lanes to a row up to kFewRows rows and columns,
// where a row's chain of loads sets the time and eight lanes read it in fewer rounds, and 4
// lanes above.  207 steps with gradients in FP64, ms, by shape 4x1 / 8x1 (and the kernel
// of one row per wavefront): 200 x 500, B 1 4.33 / 4.16 (4.40); 1 104 x 2 760, B 1 4.62 / 4.23 (4.95);
// 2 000 x 5 000, B 2 4.87 / 4.45 (5.57); 5 500 x 13 750, B 4 6.09 / 5.46 (9.84); 8 000 x 20 000, B 1
// 5.31 / 5.11 (12.2); 12 000 x 30 000, B 1 5.57 / 5.91 (16.5); 20 000 x 50 000, B 1 7.19 / 7.67 (24.9).
// More members: the least of the times of both products, estimated as
//   (members computed, those past B included) x (nonzeros) x (time of a product),
// and, beyond that and a launch's 5 us, the longest row's chain of sums, which one lane
// adds up for each of its members in turn.  Shapes of more than one member per lane must
// leave min_waves wavefronts.  8x1 costs less where the whole launch is small, above all where
// the slabs are a multiple of the XCDs.  Measured, 60 steps with gradients, ms, by shape 8x1 /
// 16x1 / 8x2 / 8x4 (the kernel of one row per wavefront in brackets), * the one taken:
//   FP32 20 000 x 50 000, B 64               9.45 / 8.16 / 7.62 / 7.06*  (7.59)
//   FP32  5 000 x 12 500, B 64               3.15 / 3.05 / 3.02* / 3.28  (3.29)
//   FP32  2 000 x  5 000, B 64               1.83* / 2.04 / 2.17 / 2.44  (2.09)
//   FP32  2 000 x  5 000, B 16               1.69 / 1.61* / 1.83 / 2.12  (1.85)
//   FP64 20 000 x 50 000, B 64               13.6 / 13.4 / 11.2*         (13.3)
//   FP64  2 000 x  5 000, B 64               2.02 / 2.42 / 2.10*         (2.51)
//   FP64  5 000 x 12 500, B 24               2.43* / 2.89 / 2.54         (3.32)
//   FP32 skewed 20 000 x 50 000 (a row of 26 155), B 64   269 / 211* / 380 / 608 (470)
//   FP64 skewed  5 000 x 12 500 (a row of  6 856), B 64   63.6 / 48.1* / 73.7    (68.8)
constexpr int kFewRows = 24576;

template <typename V>
Shape pick_shape(int m, int n, long long nnz, int alongest, int tlongest, int B)
{
  if (const char* e = std::getenv("CUOPT_AMD_UNR_SHAPE")) {  // 10 x lanes + members per lane, for tests
    const int v = std::atoi(e);
    for (Shape s : {Shape::k4x1, Shape::k8x1, Shape::k16x1, Shape::k8x2, Shape::k8x4})
      if (v == (s == Shape::k4x1 ? 41 : s == Shape::k8x1 ? 81 : s == Shape::k16x1 ? 161 : s == Shape::k8x2 ? 82 : 84))
        return s == Shape::k8x4 && sizeof(V) == 8 ? Shape::k8x2 : s;
  }
  if (B <= 4) return std::max(m, n) <= kFewRows ? Shape::k8x1 : Shape::k4x1;
  constexpr bool kF32 = sizeof(V) == 4;
  struct Option {
    Shape s;
    int vw, min_waves;
    double product, chain;  // a product's time against 16x1's, a step of a row's chain in us
  };
  const Option options[] = {{Shape::k8x1, 1, 0, kF32 ? 1.15 : 1.1, kF32 ? 0.055 : 0.050},
                            {Shape::k16x1, 1, 0, 1.0, kF32 ? 0.043 : 0.036},
                            {Shape::k8x2, 2, kF32 ? 1200 : 500, kF32 ? 0.95 : 0.85, kF32 ? 0.076 : 0.060},
                            {Shape::k8x4, 4, 1500, 0.9, 0.120}};
  Shape best  = Shape::k4x1;
  double cost = 1e300;
  for (const Option& o : options) {
    const long long W = slab_width(o.s), slabs = (B + W - 1) / W, members = slabs * W;
    if (o.vw * sizeof(V) > 16) continue;
    if (std::min(m, n) * members / (kWave * o.vw) < o.min_waves) continue;
    if ((unsigned long long)std::max(m, n) * W * sizeof(V) >= (1ULL << 32)) continue;  // 32-bit gather offsets
    double product = o.product;
    if (o.s == Shape::k8x1 && members * nnz < 3000000) product = slabs % kXcds == 0 ? 0.95 : 1.02;
    const double us = (kF32 ? 0.8e-6 : 1.2e-6) * product * members * nnz;  // one launch
    double both     = 2.0 * us;
    for (int longest : {alongest, tlongest}) both += std::max(0.0, o.chain * longest - std::max(us, 5.0));
    if (both < cost) {
      cost = both;
      best = o.s;
    }
  }
  return best;
}

// Whether a gather's offset takes 64 bits.  Otherwise it is one 24-bit multiply-add, of the
// row's number and the bytes that a slab stores of a row.
template <typename V>
bool big_offsets(Shape s, int m, int n)
{
  const unsigned long long rows = std::max(m, n);
  return rows >= (1ULL << 24) || rows * slab_width(s) * sizeof(V) >= (1ULL << 32);
}

// Calls f(Lanes<...>{}) for a shape.
template <typename V, bool BIG, int SHORT, class F>
void with_lanes(Shape s, F&& f)
{
  switch (s) {
    case Shape::k8x1: f(Lanes<8, 1, BIG, SHORT>{}); break;
    case Shape::k16x1: f(Lanes<16, 1, BIG, SHORT>{}); break;
    case Shape::k8x2: f(Lanes<8, 2, BIG, SHORT>{}); break;
    case Shape::k8x4:
      if constexpr (sizeof(V) == 4) f(Lanes<8, 4, BIG, SHORT>{});
      break;
    default: f(Lanes<4, 1, BIG, SHORT>{});
  }
}
// longest: the nonzeros of the matrix's longest row.
template <typename V, class F>
void with_shape(Shape s, int m, int n, int longest, F&& f)
{
  if (big_offsets<V>(s, m, n)) with_lanes<V, true, 0>(s, f);
  else if (longest > 4 || longest == 0) with_lanes<V, false, 0>(s, f);
  else if (longest > 2) with_lanes<V, false, 4>(s, f);
  else with_lanes<V, false, 2>(s, f);
}

// One matrix as the SpMM kernels take it.  runs: in the order in which consecutive
// groups take the rows, each row's number and nonzeros [x, y, z) = (row, begin, end),
// so that a group learns all of it from one load.
template <typename V>
struct MatView {
  const int4* runs;
  const int* idx;
  const V* val;
  int rows;
};

// How a batch lies in slabs: `count` of them, and of the last one only the first `last`
// members of each row are stored.
struct Slabs {
  int count, last;
  __host__ __device__ size_t members(int W) const { return (size_t)(count - 1) * W + last; }
};

// The workgroups of a launch lie in rows of at most 2^kGridShift: a row of 2^24 would have 2^32
// lanes, more than a launch can count.
constexpr int kGridShift = 20;

// The slabs of B members.  Up to four are stored as they are (VW of a lane together), more
// in fours: 100 steps with gradients, ms, with the last slab stored whole / exactly / in fours:
//   FP64 20 000 x 50 000, B 1   4.80 / 3.56 / 3.56      B 33  14.9 / 13.5 / 13.5     B 13  6.76 / 7.53 / 6.75
//   FP32  2 000 x  5 000, B 1   2.51 / 2.20 / 2.20      B 9   2.61 / 2.80 / 2.60     B 13  2.60 / 2.83 / 2.60
//   FP32    500 x  1 250, B 5   2.33 / 2.44 / 2.33
// (rows that start anywhere in a 64-byte line take more requests).  exact: no member more than B,
// for a shape of one member per lane.
inline Slabs slabs_of(Shape shape, int B, bool exact = false)
{
  const int W = slab_width(shape), VW = shape == Shape::k8x4 ? 4 : shape == Shape::k8x2 ? 2 : 1;
  const int count = (B + W - 1) / W, last = B - (count - 1) * W;
  const int unit = exact || last <= 4 ? VW : 4;
  return {count, (last + unit - 1) / unit * unit};
}

template <class L>
dim3 slab_grid(int rows, Slabs S)
{
  const long long items = (long long)((std::max(rows, 1) + L::rows_per_wg - 1) / L::rows_per_wg) * S.count;
  const long long all = (items + kXcds - 1) / kXcds * kXcds, row = 1LL << kGridShift;
  return dim3((unsigned)std::min(all, row), (unsigned)((all + row - 1) / row));
}

// This lane's slab, row and first member within the slab; false past the end.  width:
// the slab's stored members of a row (the same in every lane).  Lanes past it compute
// member 0 again, since their group hands the row's entries round, and store nothing.
struct Place {
  int slab, row, w, k0, k1, width;
  bool live;
};
template <class L>
__device__ inline bool my_place(int rows, Slabs S, const int4* __restrict__ runs, Place& p)
{
  const int blocks = (rows + L::rows_per_wg - 1) / L::rows_per_wg;
  const int items = blocks * S.count, per = (items + (int)kXcds - 1) / (int)kXcds;
  const unsigned at = (blockIdx.y << kGridShift) + blockIdx.x;
  const int item    = (int)(at % kXcds) * per + (int)(at / kXcds);
  if ((int)(at / kXcds) >= per || item >= items) return false;
  p.slab        = item / blocks;
  const int pos = (item - p.slab * blocks) * L::rows_per_wg + (int)threadIdx.x / L::LW;
  if (pos >= rows) return false;
  const int4 run = runs[pos];
  p.row = run.x;
  p.k0  = run.y;
  p.k1  = run.z;
  p.width = p.slab + 1 == S.count ? S.last : L::W;
  p.w     = (int)threadIdx.x % L::LW * L::VW;
  p.live  = p.w < p.width;
  if (!p.live) p.w = 0;
  return true;
}
// Offset of the lane's members of row i in a slab array of `rows` rows.
template <class L>
__device__ inline size_t slab_at(const Place& p, int rows, int i)
{
  const size_t slab = (size_t)p.slab * rows * L::W;
  if constexpr (L::BIG) return slab + (size_t)i * p.width + p.w;
  return slab + (__umul24(i, p.width) + p.w);
}
// Slab, row and member within the slab of element o of a slab array of `rows` rows.
struct SlabElement {
  int slab, row, w;
};
__device__ inline SlabElement slab_element(size_t o, int rows, int W, Slabs S)
{
  auto split = [&](auto o, auto per) -> SlabElement {  // in 32 bits where they do: divisions
    const int slab  = (int)min(o / per, (decltype(o))(S.count - 1));
    const auto r    = o - slab * per;
    const int width = slab + 1 == S.count ? S.last : W;
    const auto row  = r / width;
    return {slab, (int)row, (int)(r - row * width)};
  };
  const size_t per = (size_t)rows * W;
  if (per * S.count < (1ULL << 31)) return split((unsigned)o, (unsigned)per);
  return split(o, per);
}

// VW contiguous values, loaded and stored as one vector.
template <typename V, int VW>
struct alignas(sizeof(V) * VW) Pack {
  V v[VW];
};
template <typename V, int VW>
__device__ inline Pack<V, VW> load_pack(const V* p)
{
  return *reinterpret_cast<const Pack<V, VW>*>(p);
}
template <typename V, int VW>
__device__ inline void store_pack(V* p, const Pack<V, VW>& x)
{
  *reinterpret_cast<Pack<V, VW>*>(p) = x;
}

// Lane I's value of v within each group of LW lanes, by DPP: quad_perm for 4; for 8 the
// same, mirrored into the group's other quad; row_newbcast for 16.
template <int LW, int I>
__device__ inline int group_value(int v)
{
  if constexpr (LW == 16) {
    return __builtin_amdgcn_update_dpp(v, v, 0x150 + I, 0xf, 0xf, false);
  } else {
    const int q = __builtin_amdgcn_update_dpp(v, v, (I % 4) * 0x55, 0xf, 0xf, false);
    if constexpr (LW == 4) return q;
    return __builtin_amdgcn_update_dpp(q, q, 0x141, 0xf, I < 4 ? 0xa : 0x5, false);  // row_half_mirror
  }
}
template <int LW, int I>
__device__ inline float group_value(float v)
{
  return __int_as_float(group_value<LW, I>(__float_as_int(v)));
}
template <int LW, int I>
__device__ inline double group_value(double v)
{
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)group_value<LW, I>((int)(unsigned)u);
  const unsigned hi = (unsigned)group_value<LW, I>((int)(unsigned)(u >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// a[i] = dot product of the matrix row with member i of the lane's operand (slab: its
// first row, the same in every lane).  Every member's products are added in
// increasing k, as a row-at-a-time loop would.  A chunk's gathers (eight nonzeros or
// more) are issued before its sums, and the next chunk's indices and values in
// between.
//
// In FP32 the vector ALU is what bounds the forward steps (at 20 000 x 50 000, B = 64 it
// issues in 81-84 % of the CUs' busy cycles; ten operations per product for the compensated
// sum), and most of the adjoint steps' time (58-66 %; they also read and write more).  So the
// rest is kept small: a gather is one 32-bit offset from a scalar base (64 bits only where a
// slab's operand needs them, BIG), and a chunk that is whole in every row of the wavefront
// is summed without looking at the rows' ends.
template <typename V, class L, int... I>
__device__ inline void row_dot_chunks(const MatView<V>& M, const Place& p, const V* __restrict__ slab,
                                      typename AccFor<V>::type (&a)[L::VW], std::integer_sequence<int, I...>)
{
  using Acc       = typename AccFor<V>::type;
  constexpr int C = L::LW, N = L::LW == 4 ? 2 : 1;  // nonzeros per load, loads per chunk
  const int gl    = (int)threadIdx.x % L::LW;
  const int ke    = p.k1;
  const char* base = reinterpret_cast<const char*>(slab);
  const unsigned w = (unsigned)p.w * (unsigned)sizeof(V);
  const unsigned row = (unsigned)p.width * (unsigned)sizeof(V);
#pragma unroll
  for (int i = 0; i < L::VW; ++i) a[i] = Acc::zero();
  int ci[N];
  V vi[N];
  auto load = [&](int k) {
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const int kk = k + q * C + gl;
      ci[q] = 0;  // past the row's end: gathered from row 0 and not used
      vi[q] = V(0);
      if (kk < ke) {
        ci[q] = M.idx[kk];
        vi[q] = M.val[kk];
      }
    }
  };
  auto gather = [&](int col) {
    if constexpr (L::BIG)
      return load_pack<V, L::VW>(reinterpret_cast<const V*>(base + ((size_t)(unsigned)col * row + w)));
    else
      return load_pack<V, L::VW>(reinterpret_cast<const V*>(base + (__umul24((unsigned)col, row) + w)));
  };
  load(p.k0);
  // Matrices of short rows gather no more than the longest row has nonzeros, where a whole
  // chunk is eight or sixteen: transportation 5 000 x 12 000 (two to a column), 60 steps with
  // gradients, B 8 in FP64 3.31 -> 3.00 ms, B 33 in FP32 6.54 -> 5.80.
  if constexpr (L::SHORT > 0) {
    Pack<V, L::VW> x[L::SHORT];
    V v[L::SHORT];
    auto slot = [&](auto U) {
      constexpr int u = decltype(U)::value;
      x[u] = gather(group_value<L::LW, u>(ci[0]));
      v[u] = group_value<L::LW, u>(vi[0]);
    };
    using std::integral_constant;
    slot(integral_constant<int, 0>{}), slot(integral_constant<int, 1>{});
    if constexpr (L::SHORT == 4) slot(integral_constant<int, 2>{}), slot(integral_constant<int, 3>{});
#pragma unroll
    for (int u = 0; u < L::SHORT; ++u)
      if (p.k0 + u < ke)
#pragma unroll
        for (int i = 0; i < L::VW; ++i) a[i].add(Acc::prod(v[u], x[u].v[i]));
    return;
  }
  for (int k = p.k0; k < ke; k += N * C) {
    Pack<V, L::VW> x[N][C];
    V v[N];
#pragma unroll
    for (int q = 0; q < N; ++q) {
      ((x[q][I] = gather(group_value<L::LW, I>(ci[q]))), ...);
      v[q] = vi[q];
    }
    load(k + N * C);
    auto add = [&](int q, int u, V av) {
#pragma unroll
      for (int i = 0; i < L::VW; ++i) a[i].add(Acc::prod(av, x[q][u].v[i]));
    };
    auto add_in_row = [&](int q, int u, V av) {
      if (k + q * C + u < ke) add(q, u, av);
    };
    if (__builtin_amdgcn_ballot_w64(k + N * C > ke) == 0) {
#pragma unroll
      for (int q = 0; q < N; ++q) (add(q, I, group_value<L::LW, I>(v[q])), ...);
    } else {
#pragma unroll
      for (int q = 0; q < N; ++q) (add_in_row(q, I, group_value<L::LW, I>(v[q])), ...);
    }
  }
}
template <typename V, class L>
__device__ inline void row_dot(const MatView<V>& M, const Place& p, const V* __restrict__ slab,
                               typename AccFor<V>::type (&a)[L::VW])
{
  row_dot_chunks<V, L>(M, p, slab, a, std::make_integer_sequence<int, L::LW>{});
}

// The bounds of a row for the lane's members: one per row, or per member (ldb).
template <typename V, class L>
__device__ inline Pack<V, L::VW> row_bound(const V* __restrict__ b, bool per_member, const Place& p, int rows)
{
  if (per_member) return load_pack<V, L::VW>(b + slab_at<L>(p, rows, p.row));
  Pack<V, L::VW> x;
  const V v = b[p.row];
#pragma unroll
  for (int i = 0; i < L::VW; ++i) x.v[i] = v;
  return x;
}

// ---- forward ----------------------------------------------------------------

template <typename V, class L>
__global__ __launch_bounds__(kUB) void unr_primal(MatView<V> T, int m, Slabs slabs, const V* __restrict__ y,
                                                  const V* __restrict__ x, const V* __restrict__ c,
                                                  const V* __restrict__ lb, const V* __restrict__ ub, V tau,
                                                  V inv_prox, V* __restrict__ xn, V* __restrict__ xb)
{
  Place p;
  if (!my_place<L>(T.rows, slabs, T.runs, p)) return;
  // The row's own operands are loaded before its gathers, so their latency
  // overlaps the gathers'.
  const size_t o = slab_at<L>(p, T.rows, p.row);
  const auto xr = load_pack<V, L::VW>(x + o), cr = load_pack<V, L::VW>(c + o);
  const V lo = lb[p.row], hi = ub[p.row];
  typename AccFor<V>::type aty[L::VW];
  row_dot<V, L>(T, p, y + (size_t)p.slab * m * L::W, aty);
  Pack<V, L::VW> xnew, bar;
#pragma unroll
  for (int i = 0; i < L::VW; ++i) {
    const V v = (xr.v[i] - tau * aty[i].rsub(cr.v[i])) * inv_prox;
    xnew.v[i] = mx(mn(v, hi), lo);
    bar.v[i]  = V(2) * xnew.v[i] - xr.v[i];
  }
  if (!p.live) return;
  store_pack<V, L::VW>(xn + o, xnew);
  store_pack<V, L::VW>(xb + o, bar);
}

template <typename V, class L>
__global__ __launch_bounds__(kUB) void unr_dual(MatView<V> A, int n, Slabs slabs, const V* __restrict__ xb,
                                                const V* __restrict__ y, const V* __restrict__ lc,
                                                const V* __restrict__ uc, int ldb, V sigma, V* __restrict__ yn)
{
  Place p;
  if (!my_place<L>(A.rows, slabs, A.runs, p)) return;
  const size_t o = slab_at<L>(p, A.rows, p.row);
  const auto yo  = load_pack<V, L::VW>(y + o);  // loaded before the gathers
  const auto lo = row_bound<V, L>(lc, ldb != 0, p, A.rows), hi = row_bound<V, L>(uc, ldb != 0, p, A.rows);
  typename AccFor<V>::type ax[L::VW];
  row_dot<V, L>(A, p, xb + (size_t)p.slab * n * L::W, ax);
  Pack<V, L::VW> out;
#pragma unroll
  for (int i = 0; i < L::VW; ++i) {
    const V t    = ax[i].rsub(yo.v[i] / sigma);
    const V proj = mx(-hi.v[i], mn(t, -lo.v[i]));
    out.v[i]     = (t - proj) * sigma;
  }
  if (!p.live) return;
  store_pack<V, L::VW>(yn + o, out);
}

// ---- backward ---------------------------------------------------------------

// gt = sigma (1 - inside) ay for the step that produced y+ (its clamp states),
// and the FP64 (l_c, u_c) gradient terms.
template <typename V>
__device__ inline V dual_adjoint(V ay, V yplus, V l, V u, V sigma, double& dl, double& du)
{
  const bool eq = l == u;
  if (yplus == V(0) && !eq) {
    dl = du = 0.0;
    return V(0);
  }
  const double g = (double)sigma * (double)ay;
  if (yplus >= V(0)) {  // also y+ == 0 on an equality row: either side, both are b
    dl = g;
    du = 0.0;
  } else {
    dl = 0.0;
    du = g;
  }
  return sigma * ay;
}

// Per-step accumulators of the c and (l_c, u_c) gradients: FP64 in FP64 runs; in
// FP32 runs an FP32 partial per checkpoint segment (at most `every` terms), which
// unr_flush adds into the FP64 totals at the segment's end.  The adjoint kernels
// read and write their accumulators every step, and in FP64 those were about
// half of their traffic.
template <typename V>
struct GradAcc {
  using type = double;
};
template <>
struct GradAcc<float> {
  using type = float;
};

// acc += part; part = 0 (a kernel, not a memset, so that segment graphs may hold it).
__global__ __launch_bounds__(kUB) void unr_flush(size_t n, float* __restrict__ part, double* __restrict__ acc)
{
  for (size_t i = blockIdx.x * (size_t)kUB + threadIdx.x; i < n; i += (size_t)gridDim.x * kUB) {
    acc[i] += (double)part[i];
    part[i] = 0.f;
  }
}

// Start of the reverse sweep: gt for the last step from the upstream y-gradient
// (tot elements of slab arrays).
template <typename V>
__global__ __launch_bounds__(kUB) void unr_adj_start(size_t tot, int m, int W, Slabs S, const V* ay,  // may alias gt
                                                     const V* __restrict__ yplus, const V* __restrict__ lc,
                                                     const V* __restrict__ uc, int ldb, V sigma, V* gt,
                                                     typename GradAcc<V>::type* __restrict__ glc,
                                                     typename GradAcc<V>::type* __restrict__ guc)
{
  using GA = typename GradAcc<V>::type;
  for (size_t o = blockIdx.x * (size_t)kUB + threadIdx.x; o < tot; o += (size_t)gridDim.x * kUB) {
    const size_t q = ldb ? o : slab_element(o, m, W, S).row;  // per-member bounds, or one per row
    double dl, du;
    gt[o] = dual_adjoint(ay ? ay[o] : V(0), yplus[o], lc[q], uc[q], sigma, dl, du);
    glc[o] += (GA)dl;
    guc[o] += (GA)du;
  }
}

// Rows j of A^T: gxb = -A^T gt; gw = inner(x+) (ax + 2 gxb) / (1 + tau lam);
// ax <- gw - gxb (adjoint of x before the step); gc_acc += gw (FP64).
template <typename V, class L>
__global__ __launch_bounds__(kUB) void unr_adj_primal(MatView<V> T, int m, Slabs slabs, const V* __restrict__ gt,
                                                      const V* __restrict__ xplus, const V* __restrict__ lb,
                                                      const V* __restrict__ ub, V inv_prox, V* __restrict__ ax,
                                                      V* __restrict__ gw,
                                                      typename GradAcc<V>::type* __restrict__ gc_acc)
{
  using GA = typename GradAcc<V>::type;
  Place p;
  if (!my_place<L>(T.rows, slabs, T.runs, p)) return;
  // Element operands first (gt, which the row gathers, is none of them).
  const size_t o = slab_at<L>(p, T.rows, p.row);
  const auto xp = load_pack<V, L::VW>(xplus + o), axo = load_pack<V, L::VW>(ax + o);
  auto gc    = load_pack<GA, L::VW>(gc_acc + o);
  const V lo = lb[p.row], hi = ub[p.row];
  typename AccFor<V>::type s[L::VW];
  row_dot<V, L>(T, p, gt + (size_t)p.slab * m * L::W, s);
  Pack<V, L::VW> w, an;
#pragma unroll
  for (int i = 0; i < L::VW; ++i) {
    const V gxb = -s[i].value();
    w.v[i]      = xp.v[i] > lo && xp.v[i] < hi ? (axo.v[i] + V(2) * gxb) * inv_prox : V(0);
    an.v[i]     = w.v[i] - gxb;
    gc.v[i]     = gc.v[i] + (GA)w.v[i];
  }
  if (!p.live) return;
  store_pack<V, L::VW>(gw + o, w);
  store_pack<V, L::VW>(ax + o, an);
  store_pack<GA, L::VW>(gc_acc + o, gc);
}

// Rows i of A: ay_prev = gt / sigma + tau A gw; then, if there is an earlier
// step, its gt from ay_prev and the clamp states of its y+ (= y before this step).
// gt is read and rewritten in place, element by element.
template <typename V, class L>
__global__ __launch_bounds__(kUB) void unr_adj_dual(MatView<V> A, int n, Slabs slabs, const V* __restrict__ gw, V tau,
                                                    V sigma, const V* __restrict__ yprev, const V* __restrict__ lc,
                                                    const V* __restrict__ uc, int ldb, V* __restrict__ gt,
                                                    typename GradAcc<V>::type* __restrict__ glc,
                                                    typename GradAcc<V>::type* __restrict__ guc)
{
  using GA = typename GradAcc<V>::type;
  Place p;
  if (!my_place<L>(A.rows, slabs, A.runs, p)) return;
  // Element operands first (gw, which the row gathers, is none of them).
  const size_t o = slab_at<L>(p, A.rows, p.row);
  auto gto       = load_pack<V, L::VW>(gt + o);
  const auto yp  = load_pack<V, L::VW>(yprev + o);
  const auto lo = row_bound<V, L>(lc, ldb != 0, p, A.rows), hi = row_bound<V, L>(uc, ldb != 0, p, A.rows);
  auto glo = load_pack<GA, L::VW>(glc + o), guo = load_pack<GA, L::VW>(guc + o);
  typename AccFor<V>::type s[L::VW];
  row_dot<V, L>(A, p, gw + (size_t)p.slab * n * L::W, s);
#pragma unroll
  for (int i = 0; i < L::VW; ++i) {
    const V ay = gto.v[i] / sigma + tau * s[i].value();  // adjoint of y before this step
    double dl, du;
    gto.v[i] = dual_adjoint(ay, yp.v[i], lo.v[i], hi.v[i], sigma, dl, du);
    glo.v[i] = glo.v[i] + (GA)dl;
    guo.v[i] = guo.v[i] + (GA)du;
  }
  if (!p.live) return;
  store_pack<V, L::VW>(gt + o, gto);
  store_pack<GA, L::VW>(glc + o, glo);
  store_pack<GA, L::VW>(guc + o, guo);
}

// Caller's layout (i * B + b) to slabs of W members; stored members past B are zero.
template <typename V>
__global__ __launch_bounds__(kUB) void unr_convert_in(int rows, int B, int W, Slabs S, const double* __restrict__ in,
                                                      V* __restrict__ out)
{
  const size_t tot = rows * S.members(W);
  for (size_t o = blockIdx.x * (size_t)kUB + threadIdx.x; o < tot; o += (size_t)gridDim.x * kUB) {
    const SlabElement e = slab_element(o, rows, W, S);
    const int b         = e.slab * W + e.w;
    out[o] = b < B ? (V)in[(size_t)e.row * B + b] : V(0);
  }
}
template <typename V>
__global__ __launch_bounds__(kUB) void unr_convert_rows(int rows, const double* __restrict__ in, V* __restrict__ out)
{
  for (int i = blockIdx.x * kUB + threadIdx.x; i < rows; i += gridDim.x * kUB) out[i] = (V)in[i];
}
// Slabs to the caller's layout, scaled.
template <typename V>
__global__ __launch_bounds__(kUB) void unr_convert_out(int rows, int B, int W, Slabs S, const V* __restrict__ in, double scale,
                                                       double* __restrict__ out)
{
  const size_t tot = (size_t)rows * B;
  for (size_t o = blockIdx.x * (size_t)kUB + threadIdx.x; o < tot; o += (size_t)gridDim.x * kUB) {
    const size_t i = o / B;
    const int b = (int)(o - i * B), s = b / W;
    out[o] = scale * (double)in[(size_t)s * rows * W + i * (s + 1 == S.count ? S.last : W) + b % W];
  }
}
template <typename V>
__global__ __launch_bounds__(kUB) void unr_init_x(size_t tot, int n, int W, Slabs S, const V* __restrict__ lb,
                                                  const V* __restrict__ ub, V* __restrict__ x)
{
  for (size_t o = blockIdx.x * (size_t)kUB + threadIdx.x; o < tot; o += (size_t)gridDim.x * kUB) {
    const int j = slab_element(o, n, W, S).row;
    x[o]        = mn(mx(V(0), lb[j]), ub[j]);
  }
}
__global__ __launch_bounds__(kUB) void unr_zero64(size_t n, double* __restrict__ v)
{
  for (size_t i = blockIdx.x * (size_t)kUB + threadIdx.x; i < n; i += (size_t)gridDim.x * kUB) v[i] = 0.0;
}
template <typename V>
__global__ __launch_bounds__(kUB) void unr_zero(size_t n, V* __restrict__ v)
{
  for (size_t i = blockIdx.x * (size_t)kUB + threadIdx.x; i < n; i += (size_t)gridDim.x * kUB) v[i] = V(0);
}
// d = c / ||z|| style power step helpers (B = 1): z <- A A^T z, then norms on the host.
__global__ __launch_bounds__(kUB) void unr_sumsq(int n, const double* __restrict__ v, double* __restrict__ out)
{
  __shared__ double lds[kUB];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kUB) s += v[i] * v[i];
  lds[threadIdx.x] = s;
  __syncthreads();
  for (int off = kUB / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) lds[threadIdx.x] += lds[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = lds[0];
}
__global__ __launch_bounds__(kUB) void unr_spmv64(const int* __restrict__ ptr, const int* __restrict__ idx,
                                                  const double* __restrict__ val, int rows, const double* __restrict__ x,
                                                  double scale, double* __restrict__ y)
{
  const int r = blockIdx.x * kUB + threadIdx.x;
  if (r >= rows) return;
  double s = 0.0;
  for (int k = ptr[r]; k < ptr[r + 1]; ++k) s += val[k] * (x[idx[k]] * scale);
  y[r] = s;
}

// Y = A X over slabs (the SpMM timed by the batch-size search).
template <typename V, class L>
__global__ __launch_bounds__(kUB) void unr_spmm(MatView<V> M, int cols, Slabs slabs, const V* __restrict__ x,
                                                V* __restrict__ y)
{
  Place p;
  if (!my_place<L>(M.rows, slabs, M.runs, p)) return;
  typename AccFor<V>::type s[L::VW];
  row_dot<V, L>(M, p, x + (size_t)p.slab * cols * L::W, s);
  Pack<V, L::VW> out;
#pragma unroll
  for (int i = 0; i < L::VW; ++i) out.v[i] = s[i].value();
  if (!p.live) return;
  store_pack<V, L::VW>(y + slab_at<L>(p, M.rows, p.row), out);
}

inline int ew_blocks(size_t n) { return (int)std::max<size_t>(1, std::min<size_t>((n + kUB - 1) / kUB, 4096)); }

// Checkpoint slots addressed by a device-side segment counter, so that one
// captured segment graph serves every segment: store copies src into slot
// *seg of base, load copies slot *seg of base into dst.
template <typename V>
__global__ __launch_bounds__(kUB) void unr_ckpt_store(size_t len, const V* __restrict__ src, V* __restrict__ base,
                                                      const int* __restrict__ seg)
{
  V* dst = base + (size_t)(*seg) * len;
  for (size_t i = blockIdx.x * (size_t)kUB + threadIdx.x; i < len; i += (size_t)gridDim.x * kUB) dst[i] = src[i];
}
template <typename V>
__global__ __launch_bounds__(kUB) void unr_ckpt_load(size_t len, const V* __restrict__ base,
                                                     const int* __restrict__ seg, V* __restrict__ dst)
{
  const V* src = base + (size_t)(*seg) * len;
  for (size_t i = blockIdx.x * (size_t)kUB + threadIdx.x; i < len; i += (size_t)gridDim.x * kUB) dst[i] = src[i];
}
// seg <- set ? value : seg + value (one lane; a vector store)
__global__ void unr_seg_update(int* seg, int value, int set)
{
  if (threadIdx.x == 0 && blockIdx.x == 0) *seg = set ? value : *seg + value;
}

struct UnrolledImpl {
  int m = 0, n = 0, precision = 1;
  long long nnz = 0;
  DevBuf<int4> aruns, truns;  // MatView::runs of A and A^T
  int alongest = 0, tlongest = 0;  // nonzeros of their longest rows
  double lam = 0.0, eta = 1.0;
  // structure (device)
  DevBuf<int> aptr, aidx, tptr, tidx;
  DevBuf<double> aval64, tval64;
  DevBuf<float> aval32, tval32;
  DevBuf<double> lb64, ub64;
  DevBuf<float> lb32, ub32;
  // last forward; ready: it was queued whole, and its checkpoints stand in `work`
  bool ready = false;
  int B = 0, K = 0, every = 1, ldb = 0;
  Shape shape = Shape::k4x1;
  int W = 4;  // members per slab
  Slabs slabs{0, 0};
  DevBuf<unsigned char> work;  // typed views below
  size_t ckpt_off = 0, seg_off = 0;
  DevBuf<int> seg;  // checkpoint segment counter read by the segment graphs
  // Captured segment graphs: a full forward segment starting from either ping-pong
  // buffer, and a full backward segment (checkpoint load, recompute, reverse sweep)
  // with an earlier segment before it.  Valid while graph_key matches.
  hipGraphExec_t fwd_graph[2] = {nullptr, nullptr};
  hipGraphExec_t bwd_graph    = nullptr;
  std::vector<long long> graph_key;
  hipStream_t cap = nullptr;  // private capture stream (default priority)
  void drop_graphs()
  {
    for (hipGraphExec_t* g : {&fwd_graph[0], &fwd_graph[1], &bwd_graph}) {
      if (*g) (void)hipGraphExecDestroy(*g);
      *g = nullptr;
    }
    graph_key.clear();
  }
  ~UnrolledImpl()
  {
    drop_graphs();
    if (cap) (void)hipStreamDestroy(cap);
  }
};

template <typename V>
Shape pick_shape(const UnrolledImpl& U, int B)
{
  return pick_shape<V>(U.m, U.n, U.nnz, U.alongest, U.tlongest, B);
}

// Graph replay of full segments unless CUOPT_AMD_GRAPHS=0 (direct launches of
// the same kernels, for tests).
inline bool unrolled_graphs_enabled()
{
  const char* g = std::getenv("CUOPT_AMD_GRAPHS");
  return !(g && std::atoi(g) == 0);
}

// Records what f launches on the handle's capture stream and instantiates it.
template <class F>
hipGraphExec_t capture_graph(UnrolledImpl& U, F f)
{
  if (!U.cap) CUOPT_HIP_CHECK(hipStreamCreateWithFlags(&U.cap, hipStreamNonBlocking));
  hipGraph_t g;
  CUOPT_HIP_CHECK(hipStreamBeginCapture(U.cap, hipStreamCaptureModeThreadLocal));
  try {
    f(U.cap);
  } catch (...) {
    (void)hipStreamEndCapture(U.cap, &g);
    if (g) (void)hipGraphDestroy(g);
    throw;
  }
  CUOPT_HIP_CHECK(hipStreamEndCapture(U.cap, &g));
  hipGraphExec_t e = nullptr;
  const hipError_t r = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  CUOPT_HIP_CHECK(r);
  return e;
}

template <typename V>
struct Views {
  MatView<V> A, T;
  const V *lb, *ub;
};

template <typename V>
Views<V> views(UnrolledImpl& U)
{
  const MatView<V> none{};
  Views<V> v{none, none, nullptr, nullptr};
  if constexpr (std::is_same<V, double>::value) {
    v.A.val = U.aval64.get(), v.T.val = U.tval64.get();
    v.lb = U.lb64.get(), v.ub = U.ub64.get();
  } else {
    v.A.val = U.aval32.get(), v.T.val = U.tval32.get();
    v.lb = U.lb32.get(), v.ub = U.ub32.get();
  }
  v.A.runs = U.aruns.get(), v.A.idx = U.aidx.get(), v.A.rows = U.m;
  v.T.runs = U.truns.get(), v.T.idx = U.tidx.get(), v.T.rows = U.n;
  return v;
}

// Working storage of one forward/backward pair, carved from U.work:
//   c, lc, uc (working precision), x[2], y[2], xb, checkpoints (x, y) per segment,
//   segment states x+/y+ for every step of one segment, adjoints.
template <typename V>
struct Work {
  V *c, *lc, *uc, *x[2], *y[2], *xb, *ck_x, *ck_y, *sx, *sy, *ax, *gt, *gw;
  double *gc, *glc, *guc;
  // What the adjoint kernels accumulate into: FP32 segment partials in FP32 runs,
  // gc / glc / guc themselves in FP64 runs.
  typename GradAcc<V>::type *pc, *plc, *puc;
};

template <typename V>
Work<V> carve(UnrolledImpl& U, int nseg, bool allocate)
{
  const size_t members = U.slabs.members(U.W);
  const size_t nB = U.n * members, mB = U.m * members, lcn = U.ldb ? mB : (size_t)U.m;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) & ~(size_t)255;
    return o;
  };
  const size_t o_c = take(nB * sizeof(V)), o_lc = take(lcn * sizeof(V)), o_uc = take(lcn * sizeof(V));
  const size_t o_x0 = take(nB * sizeof(V)), o_x1 = take(nB * sizeof(V)), o_y0 = take(mB * sizeof(V)),
               o_y1 = take(mB * sizeof(V)), o_xb = take(nB * sizeof(V));
  const size_t o_ckx = take((size_t)(nseg + 1) * nB * sizeof(V)), o_cky = take((size_t)(nseg + 1) * mB * sizeof(V));
  const size_t o_sx = take((size_t)(U.every + 1) * nB * sizeof(V)), o_sy = take((size_t)(U.every + 1) * mB * sizeof(V));
  const size_t o_ax = take(nB * sizeof(V)), o_gt = take(mB * sizeof(V)), o_gw = take(nB * sizeof(V));
  const size_t o_gc = take(nB * sizeof(double)), o_glc = take(mB * sizeof(double)), o_guc = take(mB * sizeof(double));
  constexpr bool kPart = std::is_same<V, float>::value;
  const size_t o_pc = take(kPart ? nB * sizeof(float) : 0), o_plc = take(kPart ? mB * sizeof(float) : 0),
               o_puc = take(kPart ? mB * sizeof(float) : 0);
  if (allocate && U.work.size() < off) U.work.resize(off);  // kept across calls: no free / malloc per forward
  unsigned char* p = U.work.get();
  auto at = [&](size_t o) { return reinterpret_cast<V*>(p + o); };
  auto atd = [&](size_t o) { return reinterpret_cast<double*>(p + o); };
  using GA  = typename GradAcc<V>::type;
  auto atg = [&](size_t o, size_t whole) { return reinterpret_cast<GA*>(p + (kPart ? o : whole)); };
  return Work<V>{at(o_c),   at(o_lc),  at(o_uc),  {at(o_x0), at(o_x1)},
                 {at(o_y0), at(o_y1)}, at(o_xb), at(o_ckx), at(o_cky),
                 at(o_sx),  at(o_sy),  at(o_ax),  at(o_gt),
                 at(o_gw),  atd(o_gc), atd(o_glc), atd(o_guc),
                 atg(o_pc, o_gc), atg(o_plc, o_glc), atg(o_puc, o_guc)};
}

// One PDHG step (x, y) -> (xn, yn) through the scratch xb.
template <typename V>
void step(const Views<V>& M, UnrolledImpl& U, const Work<V>& W, const V* x, const V* y, V* xn, V* yn, hipStream_t s)
{
  const V tau = (V)U.eta, sigma = (V)U.eta, inv_prox = (V)(1.0 / (1.0 + U.eta * U.lam));
  with_shape<V>(U.shape, U.m, U.n, U.tlongest, [&](auto lanes) {
    using L = decltype(lanes);
    hipLaunchKernelGGL((unr_primal<V, L>), slab_grid<L>(U.n, U.slabs), dim3(kUB), 0, s, M.T, U.m, U.slabs, y, x,
                       (const V*)W.c, M.lb, M.ub, tau, inv_prox, xn, W.xb);
  });
  with_shape<V>(U.shape, U.m, U.n, U.alongest, [&](auto lanes) {
    using L = decltype(lanes);
    hipLaunchKernelGGL((unr_dual<V, L>), slab_grid<L>(U.m, U.slabs), dim3(kUB), 0, s, M.A, U.n, U.slabs,
                       (const V*)W.xb, y, (const V*)W.lc, (const V*)W.uc, U.ldb, sigma, yn);
  });
}

template <typename V>
void forward_impl(UnrolledImpl& U, const double* c, const double* lc, const double* uc, double* x_out, double* y_out,
                  hipStream_t s)
{
  const int nseg = (U.K + U.every - 1) / U.every;
  Work<V> W      = carve<V>(U, nseg, true);
  Views<V> M     = views<V>(U);
  const size_t members = U.slabs.members(U.W), nB = U.n * members, mB = U.m * members;
  if (!U.seg.get()) U.seg.resize(1);
  // The captured graphs hold the work buffer's addresses and the layout.  Where carve()
  // places the checkpoints and all that follows them goes by the number of segments.
  const std::vector<long long> key{(long long)(uintptr_t)U.work.get(), U.B, nseg, U.every, U.ldb,
                                   (long long)sizeof(V), (long long)U.shape, U.slabs.last};
  if (key != U.graph_key) {
    U.drop_graphs();
    U.graph_key = key;
  }
  hipLaunchKernelGGL(unr_convert_in<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, U.n, U.B, U.W, U.slabs, c, W.c);
  for (auto [from, to] : {std::make_pair(lc, W.lc), std::make_pair(uc, W.uc)}) {
    if (U.ldb)
      hipLaunchKernelGGL(unr_convert_in<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, U.m, U.B, U.W, U.slabs, from, to);
    else
      hipLaunchKernelGGL(unr_convert_rows<V>, dim3(ew_blocks(U.m)), dim3(kUB), 0, s, U.m, from, to);
  }
  hipLaunchKernelGGL(unr_init_x<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, nB, U.n, U.W, U.slabs, M.lb, M.ub, W.x[0]);
  hipLaunchKernelGGL(unr_zero<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, W.y[0]);
  hipLaunchKernelGGL(unr_seg_update, dim3(1), dim3(kWave), 0, s, U.seg.get(), 0, 1);
  // One segment from buffer p: checkpoint (x, y) into slot *seg, advance the
  // counter, then L steps.  Full segments replay a captured copy of this.
  auto segment = [&](int p, int L, hipStream_t q) {
    hipLaunchKernelGGL(unr_ckpt_store<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, q, nB, (const V*)W.x[p], W.ck_x,
                       (const int*)U.seg.get());
    hipLaunchKernelGGL(unr_ckpt_store<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, q, mB, (const V*)W.y[p], W.ck_y,
                       (const int*)U.seg.get());
    hipLaunchKernelGGL(unr_seg_update, dim3(1), dim3(kWave), 0, q, U.seg.get(), 1, 0);
    int c = p;
    for (int t = 0; t < L; ++t, c ^= 1) step<V>(M, U, W, W.x[c], W.y[c], W.x[c ^ 1], W.y[c ^ 1], q);
  };
  const bool graphs = unrolled_graphs_enabled() && nseg > 1;
  int cur = 0;
  for (int sg = 0; sg < nseg; ++sg) {
    const int L = std::min(U.K, (sg + 1) * U.every) - sg * U.every;
    if (graphs && L == U.every) {
      if (!U.fwd_graph[cur]) U.fwd_graph[cur] = capture_graph(U, [&](hipStream_t q) { segment(cur, L, q); });
      CUOPT_HIP_CHECK(hipGraphLaunch(U.fwd_graph[cur], s));
    } else {
      segment(cur, L, s);
    }
    cur ^= (L & 1);
  }
  CUOPT_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(unr_convert_out<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, U.n, U.B, U.W, U.slabs, (const V*)W.x[cur], 1.0,
                     x_out);
  if (y_out)
    hipLaunchKernelGGL(unr_convert_out<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, U.m, U.B, U.W, U.slabs,
                       (const V*)W.y[cur], 1.0, y_out);
  // final state kept for the backward pass (segment states are recomputed)
  CUOPT_HIP_CHECK(hipGetLastError());
}

template <typename V>
void backward_impl(UnrolledImpl& U, const double* gx, const double* gy, double* gc, double* glc, double* guc,
                   hipStream_t s)
{
  const int nseg  = (U.K + U.every - 1) / U.every;
  Work<V> W       = carve<V>(U, nseg, false);
  Views<V> M      = views<V>(U);
  const size_t members = U.slabs.members(U.W), nB = U.n * members, mB = U.m * members;
  const V tau = (V)U.eta, sigma = (V)U.eta, inv_prox = (V)(1.0 / (1.0 + U.eta * U.lam));
  hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(nB)), dim3(kUB), 0, s, nB, W.gc);
  hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, W.glc);
  hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, W.guc);
  constexpr bool kPart = std::is_same<V, float>::value;
  if constexpr (kPart) {
    hipLaunchKernelGGL(unr_zero<float>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, nB, W.pc);
    hipLaunchKernelGGL(unr_zero<float>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, W.plc);
    hipLaunchKernelGGL(unr_zero<float>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, W.puc);
  }
  hipLaunchKernelGGL(unr_convert_in<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, U.n, U.B, U.W, U.slabs, gx, W.ax);
  // y-gradient: start value of ay (zero when absent), staged in gw's slot of size m*B? use gt as ay first.
  if (gy)
    hipLaunchKernelGGL(unr_convert_in<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, U.m, U.B, U.W, U.slabs, gy, W.gt);
  // The segments run last to first; the counter names the checkpoint slot.
  hipLaunchKernelGGL(unr_seg_update, dim3(1), dim3(kWave), 0, s, U.seg.get(), nseg - 1, 1);
  // One segment of L steps: load its checkpoint, recompute states x_{k0..k0+L},
  // y_{k0..k0+L} into the segment store (slot t holds step k0 + t), run the
  // reverse sweep, step the counter back.  last: the segment holding the final
  // step (gt starts from the upstream y-gradient); first: segment 0, whose first
  // step starts from the constant y = 0 and propagates into no earlier step.
  auto segment = [&](int L, bool last, bool first, hipStream_t q) {
    hipLaunchKernelGGL(unr_ckpt_load<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, q, nB, (const V*)W.ck_x,
                       (const int*)U.seg.get(), W.sx);
    hipLaunchKernelGGL(unr_ckpt_load<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, q, mB, (const V*)W.ck_y,
                       (const int*)U.seg.get(), W.sy);
    for (int t = 0; t < L; ++t)
      step<V>(M, U, W, W.sx + (size_t)t * nB, W.sy + (size_t)t * mB, W.sx + (size_t)(t + 1) * nB,
              W.sy + (size_t)(t + 1) * mB, q);
    for (int t = L - 1; t >= 0; --t) {
      const V* xplus = W.sx + (size_t)(t + 1) * nB;
      const V* yplus = W.sy + (size_t)(t + 1) * mB;
      if (last && t == L - 1)
        hipLaunchKernelGGL(unr_adj_start<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, q, mB, U.m, U.W, U.slabs,
                           gy ? (const V*)W.gt : (const V*)nullptr, yplus, (const V*)W.lc, (const V*)W.uc, U.ldb,
                           sigma, W.gt, W.plc, W.puc);
      with_shape<V>(U.shape, U.m, U.n, U.tlongest, [&](auto lanes) {
        using L = decltype(lanes);
        hipLaunchKernelGGL((unr_adj_primal<V, L>), slab_grid<L>(U.n, U.slabs), dim3(kUB), 0, q, M.T, U.m, U.slabs,
                           (const V*)W.gt, xplus, M.lb, M.ub, inv_prox, W.ax, W.gw, W.pc);
      });
      if (!first || t > 0)
        with_shape<V>(U.shape, U.m, U.n, U.alongest, [&](auto lanes) {
          using L = decltype(lanes);
          hipLaunchKernelGGL((unr_adj_dual<V, L>), slab_grid<L>(U.m, U.slabs), dim3(kUB), 0, q, M.A, U.n, U.slabs,
                             (const V*)W.gw, tau, sigma, (const V*)(W.sy + (size_t)t * mB), (const V*)W.lc,
                             (const V*)W.uc, U.ldb, W.gt, W.plc, W.puc);
        });
    }
    if constexpr (kPart) {  // the segment's FP32 partials into the FP64 totals
      hipLaunchKernelGGL(unr_flush, dim3(ew_blocks(nB)), dim3(kUB), 0, q, nB, W.pc, W.gc);
      hipLaunchKernelGGL(unr_flush, dim3(ew_blocks(mB)), dim3(kUB), 0, q, mB, W.plc, W.glc);
      hipLaunchKernelGGL(unr_flush, dim3(ew_blocks(mB)), dim3(kUB), 0, q, mB, W.puc, W.guc);
    }
    hipLaunchKernelGGL(unr_seg_update, dim3(1), dim3(kWave), 0, q, U.seg.get(), -1, 0);
  };
  const bool graphs = unrolled_graphs_enabled();
  for (int sg = nseg - 1; sg >= 0; --sg) {
    const int L = std::min(U.K, (sg + 1) * U.every) - sg * U.every;
    const bool last = sg == nseg - 1, first = sg == 0;
    if (graphs && !last && !first) {  // middle segments are always full
      if (!U.bwd_graph) U.bwd_graph = capture_graph(U, [&](hipStream_t q) { segment(L, false, false, q); });
      CUOPT_HIP_CHECK(hipGraphLaunch(U.bwd_graph, s));
    } else {
      segment(L, last, first, s);
    }
  }
  CUOPT_HIP_CHECK(hipGetLastError());
  // gc = -tau / (1 + tau lam) * sum of gw: the kernel accumulated gw, already divided by (1 + tau lam).
  hipLaunchKernelGGL(unr_convert_out<double>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, U.n, U.B, U.W, U.slabs,
                     (const double*)W.gc, -U.eta, gc);
  hipLaunchKernelGGL(unr_convert_out<double>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, U.m, U.B, U.W, U.slabs,
                     (const double*)W.glc, 1.0, glc);
  hipLaunchKernelGGL(unr_convert_out<double>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, U.m, U.B, U.W, U.slabs,
                     (const double*)W.guc, 1.0, guc);
  CUOPT_HIP_CHECK(hipGetLastError());
}

}  // namespace

// MatView::runs.  The rows come by length within windows of 1 024, so that the 16 rows of
// a wavefront end together: on Poisson-like rows of 20 nonzeros the longest of 16 in
// index order has 28.
static std::vector<int4> row_runs(const int* ptr, int rows)
{
  constexpr int kWindow = 1024;
  std::vector<int4> runs(rows);
  for (int i = 0; i < rows; ++i) runs[i] = make_int4(i, ptr[i], ptr[i + 1], 0);
  for (int b = 0; b < rows; b += kWindow)
    std::stable_sort(runs.begin() + b, runs.begin() + std::min(rows, b + kWindow),
                     [](const int4& x, const int4& y) { return x.z - x.y > y.z - y.y; });
  return runs;
}

// ---- C++ entry points used by the C ABI ---------------------------------------------

UnrolledHandle* unrolled_create(int m, int n, const int* rowptr, const int* colidx, const double* vals,
                                const double* lb, const double* ub, double lam, int precision)
{
  auto* U = new UnrolledImpl();
  PoolStore::get().trim();
  try {
    U->m = m;
    U->n = n;
    U->lam = lam;
    U->precision = precision;
    const int nnz = rowptr[m];
    U->nnz        = nnz;
    // A^T by a stable counting sort
    std::vector<int> tp(n + 1, 0), ti(nnz);
    std::vector<double> tv(nnz);
    for (int k = 0; k < nnz; ++k) tp[colidx[k] + 1]++;
    for (int j = 0; j < n; ++j) tp[j + 1] += tp[j];
    {
      std::vector<int> cur(tp.begin(), tp.end() - 1);
      for (int i = 0; i < m; ++i)
        for (int k = rowptr[i]; k < rowptr[i + 1]; ++k) {
          const int d = cur[colidx[k]]++;
          ti[d]       = i;
          tv[d]       = vals[k];
        }
    }
    hipStream_t s = nullptr;
    const std::vector<int4> ar = row_runs(rowptr, m), tr = row_runs(tp.data(), n);
    for (const int4& r : ar) U->alongest = std::max(U->alongest, r.z - r.y);
    for (const int4& r : tr) U->tlongest = std::max(U->tlongest, r.z - r.y);
    U->aruns.resize(std::max(m, 1));
    U->aruns.upload(ar, s);
    U->truns.resize(std::max(n, 1));
    U->truns.upload(tr, s);
    U->aptr.resize(m + 1);
    U->aptr.upload(rowptr, m + 1, s);
    U->aidx.resize(std::max(nnz, 1));
    U->aidx.upload(colidx, nnz, s);
    U->tptr.resize(n + 1);
    U->tptr.upload(tp.data(), n + 1, s);
    U->tidx.resize(std::max(nnz, 1));
    U->tidx.upload(ti.data(), nnz, s);
    U->aval64.resize(std::max(nnz, 1));
    U->aval64.upload(vals, nnz, s);
    U->tval64.resize(std::max(nnz, 1));
    U->tval64.upload(tv.data(), nnz, s);
    U->lb64.resize(std::max(n, 1));
    U->lb64.upload(lb, n, s);
    U->ub64.resize(std::max(n, 1));
    U->ub64.upload(ub, n, s);
    std::vector<float> f, g, l, u;  // host sources of the async uploads, alive until the final sync
    if (precision == CUOPT_AMD_PRECISION_FP32_MIXED) {
      f.assign(vals, vals + nnz);
      g.assign(tv.begin(), tv.end());
      l.assign(lb, lb + n);
      u.assign(ub, ub + n);
      U->aval32.resize(std::max(nnz, 1));
      U->aval32.upload(f, s);
      U->tval32.resize(std::max(nnz, 1));
      U->tval32.upload(g, s);
      U->lb32.resize(std::max(n, 1));
      U->lb32.upload(l, s);
      U->ub32.resize(std::max(n, 1));
      U->ub32.upload(u, s);
    }
    // power iteration on A A^T (FP64): z <- A (A^T z / ||z||), sigma_max^2 = ||z_new|| at convergence
    DevBuf<double> z(std::max(m, 1)), w(std::max(n, 1)), nrm(1);
    std::vector<double> z0(m);
    for (int i = 0; i < m; ++i) z0[i] = 1.0 + 0.5 * std::sin(0.7 * i + 0.3);  // deterministic start
    z.upload(z0, s);
    double norm2 = 0.0, prev = 0.0, s2 = 0.0;
    hipLaunchKernelGGL(unr_sumsq, dim3(1), dim3(kUB), 0, s, m, z.get(), nrm.get());
    nrm.download(&norm2, 1, s);
    CUOPT_HIP_CHECK(hipStreamSynchronize(s));
    for (int it = 0; it < 2000 && m > 0 && n > 0; ++it) {
      const double inv = 1.0 / std::sqrt(norm2);
      hipLaunchKernelGGL(unr_spmv64, dim3((n + kUB - 1) / kUB), dim3(kUB), 0, s, U->tptr.get(), U->tidx.get(),
                         U->tval64.get(), n, z.get(), inv, w.get());
      hipLaunchKernelGGL(unr_spmv64, dim3((m + kUB - 1) / kUB), dim3(kUB), 0, s, U->aptr.get(), U->aidx.get(),
                         U->aval64.get(), m, w.get(), 1.0, z.get());
      hipLaunchKernelGGL(unr_sumsq, dim3(1), dim3(kUB), 0, s, m, z.get(), nrm.get());
      nrm.download(&norm2, 1, s);
      CUOPT_HIP_CHECK(hipStreamSynchronize(s));
      s2 = std::sqrt(norm2);  // ||A A^T q|| -> sigma_max^2
      if (it > 10 && std::fabs(s2 - prev) <= 1e-10 * s2) break;
      prev = s2;
    }
    U->eta = s2 > 0.0 ? 0.998 / std::sqrt(s2) : 1.0;
    CUOPT_HIP_CHECK(hipStreamSynchronize(s));
  } catch (...) {
    delete U;
    throw;
  }
  return reinterpret_cast<UnrolledHandle*>(U);
}

void unrolled_destroy(UnrolledHandle* h) { delete reinterpret_cast<UnrolledImpl*>(h); }

double unrolled_step_size(UnrolledHandle* h) { return reinterpret_cast<UnrolledImpl*>(h)->eta; }

void unrolled_forward(UnrolledHandle* h, int B, int K, int every, const double* c, const double* lc, const double* uc,
                      int bounds_per_batch, double* x, double* y, void* stream)
{
  auto* U = reinterpret_cast<UnrolledImpl*>(h);
  if (B <= 0 || K < 0 || every <= 0) throw validation_error("batch and checkpoint interval must be positive");
  U->ready = false;  // a call that fails (its working storage may not fit) leaves nothing to differentiate
  U->B     = B;
  U->K     = K;
  U->every = every;
  U->ldb   = bounds_per_batch ? B : 0;
  const bool fp32 = U->precision == CUOPT_AMD_PRECISION_FP32_MIXED;
  hipStream_t s   = static_cast<hipStream_t>(stream);
  auto run = [&](Shape shape, bool exact) {
    U->shape = shape;
    U->W     = slab_width(shape);
    U->slabs = slabs_of(shape, B, exact);
    if (fp32) forward_impl<float>(*U, c, lc, uc, x, y, s);
    else forward_impl<double>(*U, c, lc, uc, x, y, s);
  };
  const Shape shape = fp32 ? pick_shape<float>(*U, B) : pick_shape<double>(*U, B);
  try {
    run(shape, false);
  } catch (const hip_error& e) {
    // Where the stored members past B do not fit, B alone may.
    const Shape narrow = shape == Shape::k8x2 || shape == Shape::k8x4 ? Shape::k16x1 : shape;
    if (e.code != hipErrorOutOfMemory || U->slabs.members(U->W) == (size_t)B) throw;
    run(narrow, true);
  }
  U->ready = true;
}

void unrolled_backward(UnrolledHandle* h, const double* gx, const double* gy, double* gc, double* glc, double* guc,
                       void* stream)
{
  auto* U = reinterpret_cast<UnrolledImpl*>(h);
  if (!U->ready) throw validation_error("backward called without a completed forward");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (U->K == 0) {
    const size_t nB = (size_t)U->n * U->B, mB = (size_t)U->m * U->B;
    hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(nB)), dim3(kUB), 0, s, nB, gc);
    hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, glc);
    hipLaunchKernelGGL(unr_zero64, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, guc);
    return;
  }
  if (U->precision == CUOPT_AMD_PRECISION_FP32_MIXED)
    backward_impl<float>(*U, gx, gy, gc, glc, guc, s);
  else
    backward_impl<double>(*U, gx, gy, gc, glc, guc, s);
}

template <typename V>
int optimal_batch_size_impl(UnrolledImpl& U, int max_batch)
{
  const Views<V> M = views<V>(U);
  hipStream_t s;
  CUOPT_HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  DevBuf<V> x, y;
  auto cleanup = [&]() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(s);
  };
  try {
    CUOPT_HIP_CHECK(hipEventCreate(&e0));
    CUOPT_HIP_CHECK(hipEventCreate(&e1));
    auto cost = [&](int B) {
      const Shape shape = pick_shape<V>(U, B);
      const Slabs slabs    = slabs_of(shape, B);
      const size_t members = slabs.members(slab_width(shape)), nB = std::max(U.n, 1) * members,
                   mB = std::max(U.m, 1) * members;
      if (x.size() < nB) x.resize(nB);
      if (y.size() < mB) y.resize(mB);
      hipLaunchKernelGGL(unr_zero<V>, dim3(ew_blocks(nB)), dim3(kUB), 0, s, nB, x.get());
      hipLaunchKernelGGL(unr_zero<V>, dim3(ew_blocks(mB)), dim3(kUB), 0, s, mB, y.get());
      auto run = [&]() {
        if (U.m > 0)
          with_shape<V>(shape, U.m, U.n, U.alongest, [&](auto lanes) {
            using L = decltype(lanes);
            hipLaunchKernelGGL((unr_spmm<V, L>), slab_grid<L>(U.m, slabs), dim3(kUB), 0, s, M.A, U.n, slabs,
                               (const V*)x.get(), y.get());
          });
        if (U.n > 0)
          with_shape<V>(shape, U.m, U.n, U.tlongest, [&](auto lanes) {
            using L = decltype(lanes);
            hipLaunchKernelGGL((unr_spmm<V, L>), slab_grid<L>(U.n, slabs), dim3(kUB), 0, s, M.T, U.m, slabs,
                               (const V*)y.get(), x.get());
          });
      };
      run();
      CUOPT_HIP_CHECK(hipEventRecord(e0, s));
      constexpr int kRuns = 5;
      for (int i = 0; i < kRuns; ++i) run();
      CUOPT_HIP_CHECK(hipEventRecord(e1, s));
      CUOPT_HIP_CHECK(hipGetLastError());
      CUOPT_HIP_CHECK(hipEventSynchronize(e1));
      float ms = 0.f;
      CUOPT_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
      return (double)ms / kRuns / B;
    };
    const int best = search_batch_size(max_batch, cost);
    cleanup();
    return best;
  } catch (...) {
    cleanup();
    throw;
  }
}

int unrolled_optimal_batch_size(UnrolledHandle* h, int max_batch)
{
  auto& U = *reinterpret_cast<UnrolledImpl*>(h);
  if (U.precision == CUOPT_AMD_PRECISION_FP32_MIXED) return optimal_batch_size_impl<float>(U, max_batch);
  return optimal_batch_size_impl<double>(U, max_batch);
}

}  // namespace cuopt_amd
