// small_block.hpp -- PDHG iterations of a small LP in one workgroup (gfx950).
//
// An LP whose A and A^T have a few tiles each (spmv_tiles.hpp) is bound by launches, not
// by arithmetic or bytes: an iteration is two launches of about 2.5 us, and a
// termination check six more, a copy and a wait.  Here one workgroup of 1 024 lanes
// runs the iterations and termination checks up to the next restart test in one
// launch.  Four groups of 256 lanes take the tiles of a matrix in turn, each as a
// workgroup of tiled_spmv_kernel would: the same products, the same lanes per row and
// the same order of every sum, so the iterates, residuals and trace are those of the
// tiled kernels bit for bit.  The vectors live in LDS for the length of the launch,
// the scaled matrices in registers.  What bounds an iteration now is the chain of LDS
// reads and barriers of its two passes, about 1 us each.
//
// Measured (m x 2.5 m, 8 nonzeros per column, whole solves in FP64 to 1e-4 and FP32-mixed to 1e-8):
// m = 50: 6.5 -> 2.7 and 11.4 -> 4.9 ms; m = 200: 12.1 -> 5.4 and 19.6 -> 9.4 ms; m = 400 (two
// tiles per group): 12.6 -> 10.5 and 22.3 -> 18.8 ms.  With four tiles per group
// (m = 450 to 800), read from memory in every pass, it was slower than the launches
// (15.7 -> 47.0 ms), so kSmallRounds ends at two.
#pragma once

#include "pdlp_kernels.hpp"

namespace cuopt_amd {

constexpr int kSmallThreads = 1024;
constexpr int kSmallGroups  = kSmallThreads / kBlock;
constexpr int kSmallTile    = 1024;              // products per tile, at most
constexpr int kSmallPer     = kSmallTile / kBlock;  // nonzeros of a tile per lane
constexpr int kSmallRounds  = 2;                 // tiles per group and matrix, at most
constexpr int kSmallTiles   = kSmallGroups * kSmallRounds;

// Sum of count values v[i * stride] in the order of reduce_partials_kernel (a tree
// over 1 024 slots of which the first kSmallTiles hold values).
__device__ inline double small_tree(const double* v, int count, int stride)
{
  double s[kSmallTiles];
#pragma unroll
  for (int i = 0; i < kSmallTiles; ++i) s[i] = 0.0 + (i < count ? v[i * stride] : 0.0);
#pragma unroll
  for (int off = kSmallTiles / 2; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < off; ++i) s[i] += s[i + off];
  return s[0];
}

// One matrix as the kernel takes it; ptr, tiles and meta point to LDS copies.
struct SmallShape {
  const int* ptr;
  const Tile* tiles;
  const int* meta;
  int ntiles;
};

// A lane's nonzeros of its group's tiles.
template <typename Mat, int R>
struct SmallStream {
  Mat v[R][kSmallPer];
  int c[R][kSmallPer];
  __device__ void load_tile(int j, const SmallShape& M, const int* __restrict__ idx, const Mat* __restrict__ vals)
  {
    const int t = (int)threadIdx.x / kBlock + kSmallGroups * j, lt = (int)threadIdx.x % kBlock;
    if (t >= M.ntiles) return;
    const Tile tl = M.tiles[t];
#pragma unroll
    for (int i = 0; i < kSmallPer; ++i) {
      const int e = tl.z0 + lt + i * kBlock;
      if (e < tl.z1) {
        v[j][i] = vals[e];
        c[j][i] = idx[e];
      }
    }
  }
  __device__ void load(const SmallShape& M, const int* __restrict__ idx, const Mat* __restrict__ vals)
  {
#pragma unroll
    for (int j = 0; j < R; ++j) load_tile(j, M, idx, vals);
  }
};

// All rows of one matrix.  HELD: S holds the stream; otherwise each tile's is loaded
// here, one round ahead.  Reductions go to part[tile * NRED + k], a sum per tile as
// tiled_spmv_kernel leaves them.  Ends with a barrier (a matrix has a tile at least).
template <class Epi, int R, bool HELD>
__device__ inline void small_pass(const SmallShape& M, const int* __restrict__ idx,
                                  const typename Epi::Mat* __restrict__ vals, SmallStream<typename Epi::Mat, R>& S,
                                  typename Epi::Acc::Elem* prod, const Epi& epi, double* part,
                                  double (*red_lds)[kMaxRed])
{
  using Acc     = typename Epi::Acc;
  using Elem    = typename Acc::Elem;
  const int g   = (int)threadIdx.x / kBlock, lt = (int)threadIdx.x % kBlock;
  const int lane = (int)threadIdx.x & (kWave - 1), wave = (int)threadIdx.x / kWave;
  if constexpr (!HELD) S.load_tile(0, M, idx, vals);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int t     = g + kSmallGroups * j;
    const bool live = t < M.ntiles;
    if (kSmallGroups * j >= M.ntiles) break;  // the same in every lane
    Tile tl{0, 0, 0, 0};
    int lg = 0;
    // The lane group's first row: its bounds and operands, loaded beside the products.
    int rb = 0, re = 0;
    typename Epi::Pre pre{};
    if (live) {
      tl = M.tiles[t];
      lg = M.meta[t];
      const int r = tl.r0 + (lt >> lg);
      if (r < tl.r1) {
        rb  = M.ptr[r] - tl.z0;
        re  = M.ptr[r + 1] - tl.z0;
        pre = epi.load(r);
      }
#pragma unroll
      for (int i = 0; i < kSmallPer; ++i) {
        const int e = lt + i * kBlock;
        if (tl.z0 + e < tl.z1) prod[e] = epi.product(S.v[j][i], S.c[j][i], tl.z0 + e);
      }
    }
    __syncthreads();
    if constexpr (!HELD)
      if (j + 1 < R) S.load_tile(j + 1, M, idx, vals);
    double red[kMaxRed];
#pragma unroll
    for (int k = 0; k < kMaxRed; ++k) red[k] = 0.0;
    if (live) {
      const int G = 1 << lg, sub = lt & (G - 1);
      int r = tl.r0 + (lt >> lg);
      while (r < tl.r1) {
        Acc a = Acc::zero();
        int k = rb + sub;
        for (; k + 3 * G < re; k += 4 * G) {  // four LDS reads in flight, added in order
          const Elem p0 = prod[k], p1 = prod[k + G], p2 = prod[k + 2 * G], p3 = prod[k + 3 * G];
          a.add(p0);
          a.add(p1);
          a.add(p2);
          a.add(p3);
        }
        if (k + G < re) {
          const Elem p0 = prod[k], p1 = prod[k + G];
          a.add(p0);
          a.add(p1);
          k += 2 * G;
        }
        if (k < re) a.add(prod[k]);
        for (int off = G >> 1; off > 0; off >>= 1) a.merge(a.shfl(off));
        if (sub == 0) epi.row(r, a, pre, red);
        r += kBlock >> lg;
        if (r < tl.r1) {
          rb  = M.ptr[r] - tl.z0;
          re  = M.ptr[r + 1] - tl.z0;
          pre = epi.load(r);
        }
      }
    }
    if constexpr (Epi::NRED > 0) {
#pragma unroll
      for (int k = 0; k < Epi::NRED; ++k)
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) red[k] += shfl_xor_d(red[k], off);
      if (lane == 0)
#pragma unroll
        for (int k = 0; k < Epi::NRED; ++k) red_lds[wave][k] = red[k];
    }
    __syncthreads();
    if constexpr (Epi::NRED > 0) {
      if (live && lt == 0)
#pragma unroll
        for (int k = 0; k < Epi::NRED; ++k) {
          double s = red_lds[wave][k];
          for (int w = 1; w < kBlock / kWave; ++w) s += red_lds[wave + w][k];
          part[t * Epi::NRED + k] = s;
        }
      __syncthreads();
    }
  }
}

template <typename V>
struct SmallArgs {
  using V2 = typename Vec2<V>::type;
  int m, n;
  // A and A^T: structure, plans, working and unscaled values
  const int *aptr, *aidx, *tptr, *tidx;
  const Tile *atiles, *ttiles;
  const int *ameta, *tmeta;
  int natiles, nttiles;
  const V *aw, *tw;
  const double *aorig, *torig;
  // state and operands of the steps
  V *x, *y, *x_old;  // x_old: scratch of n values
  const V *x0, *y0, *c;
  const V2 *bnd, *cb;
  const V* kink;
  V *xhat, *yhat, *slack, *aty, *ybar;
  StepScalars sc;
  bool refine;
  long long k;   // iterations done
  int count;     // iterations to run; the last one is followed by a check
  int limit;     // stop at the first check past so many of them
  bool restarted;
  // Optimality test at the checks on the way (PdlpSolver::is_optimal).
  double tol_p, tol_d, abs_gap, rel_gap, obj_sf, obj_off;
  // termination check
  KktPointF<V> point;
  KktRowsEpi<V> rows;
  KktColsEpi<V> cols;
  double* out;  // kSmallChecks scalar records of `slots` values (host memory), one per check
  int slots, s_rows, s_cols, s_fpe, s_fpe0;  // slots of the sums of the two passes and of the fixed-point error terms
  int* checks;  // number of checks made, and whether the last one is optimal (host memory)
};

// Checks in one launch, at most: the restart test, which the host makes, comes every 200
// iterations, and up to iteration 1 000 there is a check every 10.
constexpr int kSmallChecks = 20;
constexpr int kSmallCount  = 200;

// conditional_major of the check schedule, on the device.
__device__ inline long long small_cond_major(long long k)
{
  long long step = 10, threshold = 1000;
  while (k >= threshold) {
    step *= 10;
    threshold *= 10;
  }
  return step;
}

// Bytes of dynamic LDS: products, vectors and row pointers.
template <typename V>
inline size_t small_lds_bytes(int m, int n)
{
  const size_t vecs = (size_t)(6 * (size_t)n + 4 * (size_t)m) * sizeof(V);
  return (size_t)kSmallGroups * kSmallTile * 8 + vecs + sizeof(int) * ((size_t)m + n + 2) + 64;
}

template <typename V, int R>
__global__ __launch_bounds__(kSmallThreads) void small_block_kernel(SmallArgs<V> A)
{
  using V2   = typename Vec2<V>::type;
  using Elem = typename AccFor<V>::type::Elem;
  __shared__ V weight[kSmallCount];
  __shared__ double sums[7];
  __shared__ Tile tiles[2][kSmallTiles];
  __shared__ int meta[2][kSmallTiles];
  __shared__ double part[kSmallTiles * 4];
  __shared__ double red_lds[kSmallThreads / kWave][kMaxRed];
  extern __shared__ __align__(16) unsigned char small_lds[];
  const int tid = threadIdx.x, m = A.m, n = A.n;
  unsigned char* at = small_lds;
  auto take = [&](size_t bytes) {
    unsigned char* p = at;
    at += bytes;
    return p;
  };
  unsigned char* const prod_base = take((size_t)kSmallGroups * kSmallTile * 8) + (size_t)(tid / kBlock) * kSmallTile * 8;
  V2* const bnd = reinterpret_cast<V2*>(take(n * sizeof(V2)));
  V2* const cb  = reinterpret_cast<V2*>(take(m * sizeof(V2)));
  V* const x    = reinterpret_cast<V*>(take(n * sizeof(V)));
  V* const xbar = reinterpret_cast<V*>(take(n * sizeof(V)));
  V* const c    = reinterpret_cast<V*>(take(n * sizeof(V)));
  V* const x0   = reinterpret_cast<V*>(take(n * sizeof(V)));
  V* const y    = reinterpret_cast<V*>(take(m * sizeof(V)));
  V* const y0   = reinterpret_cast<V*>(take(m * sizeof(V)));
  int* const ap = reinterpret_cast<int*>(take((m + 1) * sizeof(int)));
  int* const tp = reinterpret_cast<int*>(take((n + 1) * sizeof(int)));
  for (int j = tid; j < n; j += kSmallThreads) {
    bnd[j] = A.bnd[j];
    x[j]   = A.x[j];
    c[j]   = A.c[j];
    x0[j]  = A.x0[j];
  }
  for (int i = tid; i < m; i += kSmallThreads) {
    cb[i] = A.cb[i];
    y[i]  = A.y[i];
    y0[i] = A.y0[i];
  }
  for (int i = tid; i <= m; i += kSmallThreads) ap[i] = A.aptr[i];
  for (int j = tid; j <= n; j += kSmallThreads) tp[j] = A.tptr[j];
  if (tid < A.natiles) {
    tiles[0][tid] = A.atiles[tid];
    meta[0][tid]  = A.ameta[tid];
  }
  if (tid < A.nttiles) {
    tiles[1][tid] = A.ttiles[tid];
    meta[1][tid]  = A.tmeta[tid];
  }
  __syncthreads();
  const SmallShape MA{ap, tiles[0], meta[0], A.natiles}, MT{tp, tiles[1], meta[1], A.nttiles};
  Elem* const prod = reinterpret_cast<Elem*>(prod_base);
  // Halpern weights of the launch's steps: an FP64 division each, all at once.
  for (int s = tid; s < A.count; s += kSmallThreads) weight[s] = halpern_weight<V>(&A.sc, s);
  SmallStream<V, R> sa, st;
  sa.load(MA, A.aidx, A.aw);
  st.load(MT, A.tidx, A.tw);
  __syncthreads();
  double* const prod64 = reinterpret_cast<double*>(prod_base);
  int checks   = 0;
  bool optimal = false;
  for (int s = 0;; ++s) {
    const long long k0 = A.k + s;  // iterations done
    if (s == A.count || (s > 0 && k0 % small_cond_major(k0) == 0)) {
      // ---- termination check (evaluate_kkt): FP64, unscaled matrix
      double* const out = A.out + (size_t)checks * A.slots;
      double unused[kMaxRed];
      for (int j = tid; j < n; j += kSmallThreads) A.point(j, unused);
      __syncthreads();
      SmallStream<double, R> so;
      small_pass<KktRowsEpi<V>, R, false>(MA, A.aidx, A.aorig, so, prod64, A.rows, part, red_lds);
      if (tid < 3) sums[tid] = small_tree(part + tid, A.natiles, 3);
      __syncthreads();
      small_pass<KktColsEpi<V>, R, false>(MT, A.tidx, A.torig, so, prod64, A.cols, part, red_lds);
      if (tid < 4) sums[3 + tid] = small_tree(part + tid, A.nttiles, 4);
      __syncthreads();
      if (tid < 3) out[A.s_rows + tid] = sums[tid];
      if (tid < 4) out[A.s_cols + tid] = sums[3 + tid];
      ++checks;
      double po = sums[4], du = sums[5] + sums[1];
      if (A.obj_sf != 1.0 || A.obj_off != 0.0) {
        po = A.obj_sf * (po + A.obj_off);
        du = A.obj_sf * (du + A.obj_off);
      }
      optimal = sqrt(sums[3]) <= A.tol_d && sqrt(sums[0]) <= A.tol_p &&
                fabs(po - du) <= A.abs_gap + A.rel_gap * (fabs(po) + fabs(du));
      if (s == A.count || (k0 > 1 && optimal) || s >= A.limit) break;
    }
    const long long k1 = k0 + 1, k2 = k1 + 1;
    const bool major   = k1 % 200 == 0 || k2 % small_cond_major(k2) == 0;
    const bool after   = A.restarted && s == 0;  // the first step after a restart
    const bool fpe     = k1 % 200 == 0 || after;
    if (fpe) {
      for (int j = tid; j < n; j += kSmallThreads) A.x_old[j] = x[j];
      __syncthreads();
    }
    auto primal = [&](auto MAJ, auto FP) {
      using E = PrimalStepEpi<V, decltype(MAJ)::value, decltype(FP)::value>;
      const OncePerPass<E> e(E{y, x, c, bnd, x0, xbar, x, A.xhat, A.slack, A.aty, nullptr, s, A.refine}, (V)A.sc.tau,
                             weight[s]);
      small_pass<OncePerPass<E>, R, true>(MT, A.tidx, A.tw, st, prod, e, part, red_lds);
    };
    auto dual = [&](auto MAJ, auto FP) {
      using E = DualStepEpi<V, decltype(MAJ)::value, decltype(FP)::value>;
      const OncePerPass<E> e(E{xbar, y, cb, y0, y, A.yhat, A.ybar, nullptr, s, A.kink}, (V)A.sc.sigma, weight[s]);
      small_pass<OncePerPass<E>, R, true>(MA, A.aidx, A.aw, sa, prod, e, part, red_lds);
    };
    using std::false_type;
    using std::true_type;
    if (!major && !fpe) {
      primal(false_type{}, false_type{});
      dual(false_type{}, false_type{});
    } else if (!fpe) {
      primal(true_type{}, false_type{});
      dual(true_type{}, false_type{});
    } else {  // (an FPE step that is not a major one stores x-hat, y-hat and the slack early)
      primal(true_type{}, true_type{});
      dual(true_type{}, true_type{});
      double* const f = A.out + (size_t)checks * A.slots + (after ? A.s_fpe0 : A.s_fpe);  // the next check's record
      if (tid == 0) f[0] = small_tree(part, A.natiles, 1);
      __syncthreads();
      const FpeEpi<V> e{A.ybar, A.aty, xbar, A.x_old};
      small_pass<FpeEpi<V>, R, true>(MT, A.tidx, A.tw, st, prod, e, part, red_lds);
      if (tid < 2) f[1 + tid] = small_tree(part + tid, A.nttiles, 2);
      __syncthreads();
    }
  }
  for (int j = tid; j < n; j += kSmallThreads) A.x[j] = x[j];
  for (int i = tid; i < m; i += kSmallThreads) A.y[i] = y[i];
  if (tid == 0) {
    A.checks[0] = checks;
    A.checks[1] = optimal;
  }
}

// ---- power iteration (FP64) ---------------------------------------------------
//
// All steps of PdlpSolver::power_iteration in one launch: the products as above, with
// z / ||z|| formed once per row, and the two reductions of power_step_small.

struct SmallSpmvEpi {
  using Mat = double;
  using Acc = AccSum64;
  static constexpr int NRED = 0;
  const double* vec;
  double* out;
  struct Pre {};
  __device__ double product(double v, int col, int) const { return v * vec[col]; }
  __device__ Pre load(int) const { return Pre{}; }
  __device__ void row(int r, const Acc& s, const Pre&, double (&)[kMaxRed]) const { out[r] = s.value(); }
};
struct SmallPowerAEpi {  // znew = A atq, red[0] = q . znew
  using Mat = double;
  using Acc = AccSum64;
  static constexpr int NRED = 1;
  const double* atq;
  const double* q;
  double* znew;
  struct Pre {
    double q;
  };
  __device__ double product(double v, int col, int) const { return v * atq[col]; }
  __device__ Pre load(int r) const { return Pre{q[r]}; }
  __device__ void row(int r, const Acc& sum, const Pre& p, double (&red)[kMaxRed]) const
  {
    const double s = sum.value();
    znew[r]        = s;
    red[0] += p.q * s;
  }
};

struct SmallPowerArgs {
  int m, n;
  const int *aptr, *aidx, *tptr, *tidx;
  const Tile *atiles, *ttiles;
  const int *ameta, *tmeta;
  int natiles, nttiles;
  const double *as, *ts;
  const double* z;  // start vector
  double nrm;       // its norm
  double tol;
  int limit;
  PowerState* out;  // host memory
};

inline size_t small_power_lds_bytes(int m, int n)
{
  return (size_t)kSmallGroups * kSmallTile * 8 + sizeof(double) * (2 * (size_t)m + n) + sizeof(int) * ((size_t)m + n + 2) +
         64;
}

template <int R>
__global__ __launch_bounds__(kSmallThreads) void small_power_kernel(SmallPowerArgs A)
{
  __shared__ Tile tiles[2][kSmallTiles];
  __shared__ int meta[2][kSmallTiles];
  __shared__ double part[kSmallTiles];
  __shared__ double red_lds[kSmallThreads / kWave][kMaxRed];
  __shared__ double sums[2];
  extern __shared__ __align__(16) unsigned char small_lds[];
  const int tid = threadIdx.x, m = A.m, n = A.n;
  double* const all = reinterpret_cast<double*>(small_lds);  // products, and the reductions' slots
  double* const prod = all + (size_t)(tid / kBlock) * kSmallTile;
  double* const q    = all + kSmallGroups * kSmallTile;
  double* const zn   = q + m;
  double* const atq  = zn + m;
  int* const ap      = reinterpret_cast<int*>(atq + n);
  int* const tp      = ap + m + 1;
  for (int i = tid; i < m; i += kSmallThreads) q[i] = A.z[i] / A.nrm;
  for (int i = tid; i <= m; i += kSmallThreads) ap[i] = A.aptr[i];
  for (int j = tid; j <= n; j += kSmallThreads) tp[j] = A.tptr[j];
  if (tid < A.natiles) {
    tiles[0][tid] = A.atiles[tid];
    meta[0][tid]  = A.ameta[tid];
  }
  if (tid < A.nttiles) {
    tiles[1][tid] = A.ttiles[tid];
    meta[1][tid]  = A.tmeta[tid];
  }
  __syncthreads();
  const SmallShape MA{ap, tiles[0], meta[0], A.natiles}, MT{tp, tiles[1], meta[1], A.nttiles};
  SmallStream<double, R> sa, st;
  sa.load(MA, A.aidx, A.as);
  st.load(MT, A.tidx, A.ts);
  double s2 = 0.0;
  int it    = 0;
  bool done = false;
  while (it < A.limit) {
    small_pass<SmallSpmvEpi, R, true>(MT, A.tidx, A.ts, st, prod, SmallSpmvEpi{q, atq}, part, red_lds);
    small_pass<SmallPowerAEpi, R, true>(MA, A.aidx, A.as, sa, prod, SmallPowerAEpi{atq, q, zn}, part, red_lds);
    s2        = small_tree(part, A.natiles, 1);
    double r2 = 0.0, z2 = 0.0;
    for (int i = tid; i < m; i += kSmallThreads) {
      const double z = zn[i];
      const double r = q[i] * -s2 + z;
      r2 += r * r;
      z2 += z * z;
    }
    all[tid]                 = r2;
    all[kSmallThreads + tid] = z2;
    __syncthreads();
    if (tid < 2 * kWave) {
      const double v = tree_1024(all + (tid / kWave) * kSmallThreads);
      if (tid % kWave == 0) sums[tid / kWave] = v;
    }
    __syncthreads();
    ++it;
    done = sqrt(sums[0]) < A.tol;
    if (done) break;
    const double nrm = sqrt(sums[1]);
    for (int i = tid; i < m; i += kSmallThreads) q[i] = zn[i] / nrm;
    __syncthreads();
  }
  if (tid == 0) {
    PowerState o{};
    o.s2    = s2;
    o.iters = it;
    o.done  = done ? 1.0 : 0.0;
    *A.out  = o;
  }
}

}  // namespace cuopt_amd
