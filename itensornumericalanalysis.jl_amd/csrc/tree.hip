// Batched evaluation of trees and wide chains (float64): one matrix product
// per vertex over many rows (src/itensornetworkfunction.jl:96-106, calculate_
// ind_values + project + scalar for a batch of points).
//
// The tree is cut at one edge (the centre).  Every vertex then has one output
// leg, toward the centre, and input legs away from it, and the vectors over
// its output leg are
//     out[row][n] = sum_k T[n][d(row)][k] A[row][k],
//     A[row][k]   = prod_legs u_leg[index_leg(row)][k_leg],
// k running over the combinations of the input legs.  A value is the dot
// product of the two vectors over the centre edge.
//
// Rows.  A vertex with few digits behind it has at most 2^nd different
// vectors, one per digit string, however many points there are: below a limit
// its rows are the digit strings (a table), and points that share digits share
// the work.  The tables depend only on the cores, so they are kept with the
// network, like its packed chain copy, until the cores change; they lie by
// number of digits, so a call that wants fewer finds its own among more, and one
// that wants more builds what is missing.  Above the limit the rows are the points.  A table's row index has the vertex's own digit as
// its top bit, then its input tables' indices.
//
// The product.  Rows of one digit use one slice of the core, so a workgroup
// sorts the 128 rows it takes by digit (two ballots) and cuts both halves into
// 16-row tiles: no slice is computed and thrown away.  Tiles are FP64 MFMA,
// v_mfma_f64_16x16x4f64 (lane l: A[l%16][l/16], B[l/16][l%16], D[l/16 + 4e]
// [l%16]).  The order of k inside a block of 16 is free as long as A and B
// agree: lane group l/16 takes the 4 consecutive entries 4 (l/16) .. + 3, one
// per MFMA.  A load is split into the lines that each 16 consecutive lanes
// touch, so 16 lanes on 16 different rows cost 16 accesses: the core is
// repacked once into 16 x 16 tiles in lane order (zero padded, kept with the
// network), and a wavefront brings its tile's rows of the input vectors into
// LDS with row-wise loads and reads its operands there.  A vertex with few rows and a long k (a comb's backbone:
// 128 x 128 combinations) splits k over workgroups and adds the parts in order.
//
// Measured against one lane per point walking every core entry: 20,011 points
// of a 3 x 16 comb of bond 32, 39.4 -> 0.10 ms (a network's first call 0.30
// ms); 256 points of the bond 128 comb, 1530 -> about 1 ms.  What bounds it: a
// chain of one launch per level (about 5 us each) while the rows are few, the
// FP64 matrix rate at the backbone.
#include "tree.h"

#include <algorithm>
#include <cstring>
#include <new>

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int TREE_MAX_IN = QTT_MAX_NDIM - 2;  // input legs of a vertex
constexpr int TREE_JOBS = 7;                   // vertices per launch (by value: under 4 KB of arguments)
constexpr int TREE_ROWS = 128;                 // most rows per workgroup
constexpr int TREE_TABLES = 24;                // tables per index launch
constexpr int TREE_BITS = 16;                  // most digits of a table

// One input leg: vectors u (row stride in doubles), and the row of u that a
// row of the vertex takes: idx[row] when idx is set (a point's table entry),
// else (row >> shift) & mask.
struct TreeLeg {
  const double* u;
  const int* idx;
  int stride, dim, shift, mask;
};

struct TreeJob {
  const double* P;   // packed core [digit][k block][npad / 16][256 in lane order]
  double* out;       // [R][npad], or partial sums [kc][R][npad]
  const double* xs;  // the points, when the vertex's rows are points and it has a digit
  int64_t dstride;   // doubles of one digit slice of P
  int R, n, npad, nt, ngrp;  // rows; output bond, padded; 16-column tiles per workgroup, groups of them
  int m, kbl, nk;    // input legs (the last one padded to kbl blocks of 16), k blocks in all
  int big;           // trees: the last leg's place among the vertex's own legs (it was exchanged with the
                     // last of them); -1: a chain (see tree_value)
  int rpw;           // rows per workgroup
  int ldu, ldw;      // LDS row strides of a tile's vectors (last leg, first of two legs); ldu 0: not staged
  int kc, kper;      // chunks of k blocks (one workgroup each) and blocks per chunk
  int dmode;         // digit of a row: 0 none (slice 0), 1 bit dshift of the row, 2 of a point's coordinate
  int dshift, coord, nc, ndig;
  // adjoint rows of a table (gradient): row i of the input table sums both
  // digit slices, slice d from row i + d R of the leg, where seen says that
  // this row's digit string occurs among the points; seen_out receives the
  // input table's own marks.  two: 0 off, else the number of slices
  int two;
  const unsigned char* seen;
  unsigned char* seen_out;
  TreeLeg leg[TREE_MAX_IN];
};

// (the arguments lie in host memory: unit0, the vertices' first workgroups,
// apart from the jobs, so that a workgroup finds its vertex with one load)
struct TreeJobs {
  int n;
  int unit0[TREE_JOBS];
  TreeJob job[TREE_JOBS];
};
static_assert(sizeof(TreeJobs) <= 4096, "kernel arguments");

__device__ __forceinline__ uint64_t tree_digit_word(double x, int L) {
  if (!(x >= 0.0)) return 0;  // negative or NaN: reported by the final kernel
  if (x >= 1.0) return (uint64_t(1) << L) - 1;
  return (uint64_t)(x * (double)(uint64_t(1) << L));
}

// The k blocks [k0, k1) of one 16-row tile against NT 16-column tiles.  ML: 0
// no input leg, 1 one, 2 two, 3 any number.  u: the last leg's row of this lane
// (offset to its 4 entries of a block), w: the first of two legs' row, lrow the
// vertex's row (for more legs).
//
// Three stages: two blocks' loads are in flight while a block is multiplied.
// No load stands behind a branch (past the end the last block is loaded again):
// at a join the compiler cannot tell how many loads are pending and would wait
// for all of them.  The other legs' factor is applied when the block is
// multiplied, so that loading waits for nothing.  The backbone of a comb of bond
// 32 (20,011 rows, k = 1024): 82 us with one block ahead and operands in row
// order, 46 us with the stages, the core in lane order and the rows in LDS.
typedef __attribute__((address_space(3))) double lds_f64;
typedef __attribute__((address_space(3))) f64x2 lds_f64x2;
template <int NT, int ML, typename UP, typename U2>
__device__ __forceinline__ void tree_tile(const TreeJob& J, const double* __restrict__ P, UP u, UP w, int lrow,
                                          int k0, int k1, f64x4 (&acc)[NT]) {
  const int lane = threadIdx.x & 63, lk = lane >> 4;
  const int kbl = J.kbl;
  const int64_t bstep = (int64_t)J.npad * 16;
  const double* __restrict__ pb = P + (int64_t)k0 * bstep;
  int q = k0 / kbl, kb = k0 - q * kbl, left = k1 - k0;
  auto coef = [&]() {  // product of the other legs' entries of combination q
    int r = q;
    double cf = 1.0;
    for (int j = J.m - 2; j >= 0; --j) {
      const TreeLeg& L = J.leg[j];
      const int nq = r / L.dim, i = r - nq * L.dim;
      r = nq;
      const int row = L.idx ? L.idx[lrow] : (lrow >> L.shift) & L.mask;
      cf *= L.u[(int64_t)row * L.stride + i];
    }
    return cf;
  };
  struct Stage {
    f64x2 a[2], b[NT][2];
    double f;
  };
  auto load = [&](Stage& g) {
    if constexpr (ML == 0) {
      g.a[0] = f64x2{lk == 0 ? 1.0 : 0.0, 0.0};
      g.a[1] = f64x2{0.0, 0.0};
    } else {
      g.a[0] = *(U2)(u + kb * 16);
      g.a[1] = *(U2)(u + kb * 16 + 2);
    }
    if constexpr (ML == 2) g.f = w[q];
    if constexpr (ML == 3) g.f = coef();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      g.b[t][0] = *(const f64x2*)(pb + t * 256);
      g.b[t][1] = *(const f64x2*)(pb + t * 256 + 128);
    }
    const int on = left > 1 ? 1 : 0;  // stay on the last block
    left -= on;
    pb += on * bstep;
    kb += on;
    const int wrap = kb == kbl ? 1 : 0;
    q += wrap;
    kb = wrap ? 0 : kb;
  };
  auto mul = [&](const Stage& g) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double a = ML >= 2 ? g.f * g.a[i >> 1][i & 1] : g.a[i >> 1][i & 1];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, g.b[t][i >> 1][i & 1], acc[t], 0, 0, 0);
    }
  };
  Stage s0, s1, s2;
  int n = k1 - k0;
  load(s0);
  load(s1);
  for (; n >= 3; n -= 3) {
    load(s2);
    mul(s0);
    load(s0);
    mul(s1);
    load(s1);
    mul(s2);
  }
  if (n > 0) mul(s0);
  if (n > 1) mul(s1);
}

// a tile from vectors staged in LDS, or (too long for it) read where they lie
template <int NT, int ML>
__device__ __forceinline__ void tree_tile_of(const TreeJob& J, const double* P, const double* u, const double* w,
                                             const lds_f64* lu, const lds_f64* lw, int lrow, int k0, int k1,
                                             f64x4 (&acc)[NT]) {
  if (J.ldu) tree_tile<NT, ML, const lds_f64*, const lds_f64x2*>(J, P, lu, lw, lrow, k0, k1, acc);
  else tree_tile<NT, ML, const double*, const f64x2*>(J, P, u, w, lrow, k0, k1, acc);
}

// One entry of a tree's vertex: row orow, output index n (slice P), k blocks
// [k0, k1).  A core entry of zero adds nothing whatever the legs hold, and
// neither does one whose legs, from the last, reach a zero: a sum of functions
// has zero blocks, and where one term overflows (inf) the other's entries must
// not become 0 inf = NaN.  A matrix product cannot leave products out, nor the
// padding of a leg beside an infinite factor, so an entry that comes out as NaN
// is formed again here.  (A chain's products are all formed, on every route.)
__device__ __forceinline__ double tree_value(const TreeJob& J, const double* __restrict__ P, int orow, int n, int k0,
                                             int k1) {
  double s = 0.0;
  for (int kb = k0; kb < k1; ++kb) {
    const int q = kb / J.kbl;
    const double* Pb = P + ((int64_t)kb * (J.npad >> 4) + (n >> 4)) * 256 + 2 * (n & 15);
    for (int kk = 0; kk < 16; ++kk) {
      double w = Pb[((kk >> 1) & 1) * 128 + (kk >> 2) * 32 + (kk & 1)];
      for (int o = J.m - 1; o >= 0 && w != 0.0; --o) {
        const int j = o == J.m - 1 ? J.big : o == J.big ? J.m - 1 : o;
        int i = (kb - q * J.kbl) * 16 + kk;
        if (j < J.m - 1) {
          i = q;
          for (int x = J.m - 2; x > j; --x) i /= J.leg[x].dim;
          i %= J.leg[j].dim;
        }
        const TreeLeg& L = J.leg[j];
        const int row = L.idx ? L.idx[orow] : (orow >> L.shift) & L.mask;
        w *= L.u[(int64_t)row * L.stride + i];
      }
      s += w;
    }
  }
  return s;
}

template <int NT>
__device__ __forceinline__ void tree_rows(const TreeJob& J, const int* rows, int n0, int n1, int ng, int kc, int k0,
                                          int k1, lds_f64* lds) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int t0 = (n0 + 15) >> 4, ntile = t0 + ((n1 + 15) >> 4);
  const int c0 = ng * NT * 16;
  double* out = J.out + (int64_t)kc * J.R * J.npad + c0;
  lds_f64* ub = lds + wv * 16 * (J.ldu + J.ldw);
  lds_f64* wb = ub + 16 * J.ldu;
  // row r's len doubles (len even, 16-byte aligned) from base + (x of lane r) stride
  auto stage = [&](lds_f64* dst, int ld, const double* base, int x, int stride, int len) {
    const int h = len >> 1;
    for (int e = lane; e < 16 * h; e += 64) {
      const int r = e / h, c = e - r * h;
      *(lds_f64x2*)(dst + r * ld + 2 * c) = *(const f64x2*)(base + (int64_t)__shfl(x, r) * stride + 2 * c);
    }
  };
  for (int t = wv; t < ntile; t += 4) {
    const int lrow = rows[t * 16 + li];
    const int r = lrow < 0 ? rows[t * 16] : lrow;  // a padding row repeats the tile's first
    const double* P = J.P + (t < t0 ? 0 : J.dstride) + (int64_t)c0 * 16 + 2 * lane;
    const double *u = nullptr, *w = nullptr;
    const lds_f64 *lu = ub + li * J.ldu + 4 * lk, *lw = wb + li * J.ldw;
    int xu = 0;
    if (J.m) {
      const TreeLeg& L = J.leg[J.m - 1];
      xu = L.idx ? L.idx[r] : (r >> L.shift) & L.mask;
      u = L.u + (int64_t)xu * L.stride + 4 * lk;
      if (J.ldu && !J.two) stage(ub, J.ldu, L.u, xu, L.stride, J.kbl * 16);
    }
    if (J.m == 2) {
      const TreeLeg& L = J.leg[0];
      const int x = L.idx ? L.idx[r] : (r >> L.shift) & L.mask;
      w = L.u + (int64_t)x * L.stride;
      if (J.ldu) stage(wb, J.ldw, L.u, x, L.stride, (L.dim + 1) & ~1);
    }
    f64x4 acc[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
    if (J.two) {
      // slice by slice; a digit string that no point has counts as zero even if
      // a core entry it meets is not finite
      for (int sl = 0; sl < J.two; ++sl) {
        f64x4 as[NT];
#pragma unroll
        for (int c = 0; c < NT; ++c) as[c] = f64x4{0.0, 0.0, 0.0, 0.0};
        const TreeLeg& L = J.leg[0];
        if (J.ldu) stage(ub, J.ldu, L.u, xu + sl * J.R, L.stride, J.kbl * 16);
        tree_tile_of<NT, 1>(J, P + sl * J.dstride, u + (int64_t)sl * J.R * L.stride, w, lu, lw, r, k0, k1, as);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int orow = rows[t * 16 + lk + 4 * e];
          if (orow >= 0 && J.seen[orow + sl * J.R]) {
#pragma unroll
            for (int c = 0; c < NT; ++c) acc[c][e] += as[c][e];
          }
        }
      }
    } else if (J.m == 0) tree_tile_of<NT, 0>(J, P, u, w, lu, lw, r, k0, k1, acc);
    else if (J.m == 1) tree_tile_of<NT, 1>(J, P, u, w, lu, lw, r, k0, k1, acc);
    else if (J.m == 2) tree_tile_of<NT, 2>(J, P, u, w, lu, lw, r, k0, k1, acc);
    else tree_tile_of<NT, 3>(J, P, u, w, lu, lw, r, k0, k1, acc);
    bool nan = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int orow = rows[t * 16 + lk + 4 * e];
      if (orow >= 0) {
#pragma unroll
        for (int c = 0; c < NT; ++c) {  // (the padding stays zero also for infinite values)
          const double x = c0 + 16 * c + li < J.n ? acc[c][e] : 0.0;
          out[(int64_t)orow * J.npad + 16 * c + li] = x;
          nan |= x != x;
        }
      }
    }
    if (__builtin_expect(J.big >= 0 && nan, 0)) {
#pragma clang loop unroll(disable)
      for (int x = 0; x < 4 * NT; ++x) {
        const int orow = rows[t * 16 + lk + 4 * (x & 3)], c = 16 * (x >> 2) + li;
        if (orow < 0 || c0 + c >= J.n) continue;
        double* o = out + (int64_t)orow * J.npad + c;
        if (*o != *o) *o = tree_value(J, J.P + (t < t0 ? 0 : J.dstride), orow, c0 + c, k0, k1);
      }
    }
  }
}

// WIDE: vertices with 3 or 4 column tiles (more registers, fewer wavefronts)
template <bool WIDE>
__global__ void __launch_bounds__(256, WIDE ? 2 : 3) tree_vertex_kernel(TreeJobs js) {
  extern __shared__ __align__(16) double lds_raw[];
  lds_f64* lds = (lds_f64*)lds_raw;
  __shared__ int rows[TREE_ROWS + 32];
  __shared__ int cnt[4];
  int jj = 0;
#pragma unroll
  for (int i = 1; i < TREE_JOBS; ++i) jj += (i < js.n && (int)blockIdx.x >= js.unit0[i]) ? 1 : 0;
  const TreeJob& J = js.job[jj];
  const int tid = threadIdx.x;
  int unit = (int)blockIdx.x - js.unit0[jj];
  const int kc = unit % J.kc;
  unit /= J.kc;
  const int ng = unit % J.ngrp, rb = unit / J.ngrp;
  // the workgroup's rows sorted by digit: digit 0 first, each half padded to
  // whole tiles with -1
  if (tid < TREE_ROWS + 32) rows[tid] = -1;
  const int row = rb * J.rpw + tid;
  const bool on = tid < J.rpw && row < J.R;
  int d = 0;
  if (on && J.dmode == 1) d = (row >> J.dshift) & 1;
  if (on && J.dmode == 2)
    d = (int)((tree_digit_word(J.xs[(int64_t)row * J.nc + J.coord], J.ndig) >> J.dshift) & 1);
  const uint64_t b0 = __ballot(on && d == 0), b1 = __ballot(on && d == 1);
  if (tid == 0 || tid == 64) {
    cnt[tid >> 5] = __popcll(b0);
    cnt[(tid >> 5) + 1] = __popcll(b1);
  }
  __syncthreads();
  const int n0 = cnt[0] + cnt[2], n1 = cnt[1] + cnt[3];
  if (on) {
    const uint64_t below = (uint64_t(1) << (tid & 63)) - 1;
    const int pos = __popcll((d ? b1 : b0) & below) + (tid >= 64 ? cnt[d] : 0);
    rows[d ? ((n0 + 15) & ~15) + pos : pos] = row;
  }
  __syncthreads();
  if (J.two && ng == 0 && on) J.seen_out[row] = J.seen[row] | (J.two > 1 ? J.seen[row + J.R] : 0);
  const int k0 = kc * J.kper, k1 = min(J.nk, k0 + J.kper);
  if constexpr (WIDE) {
    if (J.nt == 3) tree_rows<3>(J, rows, n0, n1, ng, kc, k0, k1, lds);
    else tree_rows<4>(J, rows, n0, n1, ng, kc, k0, k1, lds);
  } else {
    if (J.nt == 1) tree_rows<1>(J, rows, n0, n1, ng, kc, k0, k1, lds);
    else tree_rows<2>(J, rows, n0, n1, ng, kc, k0, k1, lds);
  }
}

// out[e] = the sum of the kc partial results at part + c n, in a fixed order
__global__ void tree_sum_kernel(const double* __restrict__ part, int kc, int64_t n, double* __restrict__ out) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int c = 0; c < kc; ++c) s += part[(int64_t)c * n + e];
    out[e] = s;
  }
}

// Table entry of every point for up to TREE_TABLES tables: bit b of the table
// (from the top) is bit shift[b] of coordinate coord[b]'s digit word.
struct TreeIndex {
  int* out;
  int nbits;
  unsigned short coord[TREE_BITS];
  unsigned char shift[TREE_BITS];
};
struct TreeIndexArgs {
  int n;
  TreeIndex t[TREE_TABLES];
};
static_assert(sizeof(TreeIndexArgs) <= 3072, "kernel arguments");

__global__ void __launch_bounds__(256)
tree_index_kernel(TreeIndexArgs a, const double* __restrict__ xs, int64_t npts, int nc,
                  const int* __restrict__ ndigits) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= npts) return;
  const double* x = xs + p * nc;
  uint64_t kw[QTT_MAX_COORD];  // the first coordinates' digits, read once
#pragma unroll
  for (int c = 0; c < QTT_MAX_COORD; ++c) kw[c] = c < nc ? tree_digit_word(x[c], ndigits[c]) : 0;
  for (int i = 0; i < a.n; ++i) {
    const TreeIndex& t = a.t[i];
    int r = 0;
    for (int b = 0; b < t.nbits; ++b) {
      const int c = t.coord[b];
      const uint64_t w = c == 0 ? kw[0] : c == 1 ? kw[1] : c == 2 ? kw[2] : c == 3 ? kw[3]
                                                       : tree_digit_word(x[c], ndigits[c]);
      r = 2 * r + (int)((w >> t.shift[b]) & 1);
    }
    t.out[p] = r;
  }
}

// f = <u_a, u_b> over the centre edge, 16 lanes per point (b null: u_a's only
// entry).  A point with a negative or NaN coordinate gives NaN and the flag.  On
// a tree a zero entry adds nothing (see tree_value).
__global__ void __launch_bounds__(256)
tree_dot_kernel(TreeLeg a, TreeLeg b, bool tree, const double* __restrict__ xs, int64_t npts, int nc,
                double* __restrict__ out, int* __restrict__ flag) {
  const int64_t p = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4;
  const int li = threadIdx.x & 15;
  if (p >= npts) return;  // whole 16-lane groups
  const int ra = a.idx ? a.idx[p] : ((int)p >> a.shift) & a.mask;
  const double* ua = a.u + (int64_t)ra * a.stride;
  double s = 0.0;
  if (b.u) {
    const int rb = b.idx ? b.idx[p] : ((int)p >> b.shift) & b.mask;
    const double* ub = b.u + (int64_t)rb * b.stride;
    double s1 = 0.0;
    int e = li;
    for (; e + 16 < a.dim; e += 32) {
      s = __builtin_fma(ua[e], ub[e], s);
      s1 = __builtin_fma(ua[e + 16], ub[e + 16], s1);
    }
    if (e < a.dim) s = __builtin_fma(ua[e], ub[e], s);
    s += s1;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (tree && s != s) {  // (the 16 lanes hold the same sum)
      s = 0.0;
      for (e = li; e < a.dim; e += 16)
        if (ua[e] != 0.0 && ub[e] != 0.0) s = __builtin_fma(ua[e], ub[e], s);
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o);
    }
  } else {
    s = ua[0];
  }
  if (li == 0) {
    bool bad = false;
    for (int c = 0; c < nc; ++c)
      if (!(xs[p * nc + c] >= 0.0)) bad = true;
    if (bad) flag[0] = 1;
    out[p] = bad ? __builtin_nan("") : s;
  }
}

// P[d][kb][n / 16][...] = T at output index n, input combination k = 16 kb + kk
// (the last leg padded to lpad entries), digit d; zero in the padding.  A 16 x
// 16 tile holds, for h = 0, 1, the lanes' entries kk = 4 (lane / 16) + 2 h + {0, 1}
// at n % 16 = lane % 16.
struct TreePackJob {
  const double* T;
  double* P;
  int64_t total;             // doubles of P
  int nd, nk, npad, n;       // digit slices, k blocks, padded and true output bond
  int m, lpad;               // input legs, padded size of the last one
  int64_t dstr, nstr;        // strides of the core's site and output indices
  int dim[TREE_MAX_IN];
  int64_t str[TREE_MAX_IN];
};
struct TreePackJobs {
  int n;
  TreePackJob job[16];
};
static_assert(sizeof(TreePackJobs) <= 4096, "kernel arguments");

__global__ void __launch_bounds__(256) tree_pack_kernel(TreePackJobs js) {
  const TreePackJob& J = js.job[blockIdx.y];
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < J.total; e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e & 255), ln = (i >> 1) & 63;
    const int kk = 4 * (ln >> 4) + 2 * (i >> 7) + (i & 1);
    int64_t r = e >> 8;
    const int n = (int)(r % (J.npad >> 4)) * 16 + (ln & 15);
    r /= J.npad >> 4;
    const int kb = (int)(r % J.nk), d = (int)(r / J.nk);
    const int64_t k = (int64_t)kb * 16 + kk;
    double val = 0.0;
    if (n < J.n) {
      int64_t o = d * J.dstr + n * J.nstr;
      bool in = true;
      if (J.m) {
        int64_t q = k / J.lpad;
        const int kl = (int)(k - q * J.lpad);
        in = kl < J.dim[J.m - 1];
        o += kl * J.str[J.m - 1];
        for (int j = J.m - 2; j >= 0; --j) {
          const int64_t nq = q / J.dim[j];
          o += (q - nq * J.dim[j]) * J.str[j];
          q = nq;
        }
      } else {
        in = k == 0;
      }
      if (in) val = J.T[o];
    }
    J.P[e] = val;
  }
}

// ---------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------
struct VPlan {
  int to = -1;               // neighbour on the output side (-1: the network's only vertex)
  std::vector<int> in;       // input neighbours; the last one is the padded leg
  int nd = 0;                // digits behind the output leg, this vertex included
  int level = 0;             // longest path of input vertices below
  int n = 1, npad = 16, nt = 1, ngrp = 1;
  int kbl = 1, nk = 1, slices = 1;
  int big = 0;               // the last input's place before it was exchanged with the last
  int64_t pack = 0;          // offset in the packed copy
  int64_t packT = 0;         // offset in the transposed copy (gradient)
  bool fits = false;         // its rows can be digit strings (they and its inputs' are few enough)
  int64_t tab = 0;           // then: offset in the table buffer
  bool table = false;        // this call's choice
  int64_t buf = 0;           // offset in the table buffer / point buffers (per row for points)
};

// dimension of the edge between neighbours v and w
int64_t edge_dim(const qtt_net* net, int v, int w) { return net->bond[net->t.parent[v] == w ? v : w]; }

std::vector<int> neighbours(const HostTopo& t, int v) {
  std::vector<int> r;
  if (t.parent[v] >= 0) r.push_back(t.parent[v]);
  for (int k = 0; k < t.nch[v]; k++) r.push_back(t.chs[t.choff[v] + k]);
  return r;
}

// The centre edge (c, parent[c]): the one that leaves the least work when a
// vertex with nd digits behind it costs its core times min(2^nd, 2^16) rows
// (2^16: a large call; the choice is the same for every call so that the
// packed copy and the tables are built once).
int choose_centre(const qtt_net* net) {
  const HostTopo& t = net->t;
  if (t.nv < 2) return -1;
  std::vector<int> below(t.nv, 0);
  int D = 0;
  for (int v = t.nv - 1; v >= 0; v--) {
    below[v] += t.vcoord[v] >= 0;
    D += t.vcoord[v] >= 0;
    if (v) below[t.parent[v]] += below[v];
  }
  auto rows = [](int nd) { return (double)(int64_t(1) << std::min(nd, 16)); };
  // every vertex toward the root first; a centre at edge (v, parent[v]) turns
  // the vertices from parent[v] up to the root toward v
  std::vector<double> down(t.nv), cost(t.nv, 0.0);
  double total = 0.0;
  for (int v = 0; v < t.nv; v++) {
    down[v] = (double)net->core_size(v) * rows(below[v]);
    total += down[v];
  }
  std::vector<double> path(t.nv, 0.0);
  int best = 1;
  for (int v = 1; v < t.nv; v++) {
    const int p = t.parent[v];
    // p turned toward v: the digits behind it are all but below[v]
    // (p's own parents were turned toward p already, counted in path[p])
    path[v] = path[p] - down[p] + (double)net->core_size(p) * rows(D - below[v]);
    cost[v] = total + path[v];
    if (v == 1 || cost[v] < cost[best]) best = v;
  }
  return best;
}

}  // namespace

// Packed cores and table rows of a network, built for one centre edge.
struct TreeState {
  int centre = -1;
  bool packed = false;
  std::vector<VPlan> vp;
  std::vector<int> order;    // input vertices before the vertices that use them
  double* d_pack = nullptr;
  int64_t pack_cap = 0;
  bool packedT = false;      // the copy with output and input exchanged (gradient)
  double* d_packT = nullptr;
  int64_t packT_cap = 0;
  double* d_tab = nullptr;   // vectors of every table vertex
  int64_t tab_cap = 0;
  int tab_digits = 0;        // tables of fewer digits than this are built
  // what was queued last to make any of the above: ev follows it on ev_stream
  hipEvent_t ev = nullptr;
  hipStream_t ev_stream = nullptr;
  bool making = false;       // something was queued since
  ~TreeState() {
    if (ev) (void)hipEventDestroy(ev);
    if (d_pack) (void)hipFree(d_pack);
    if (d_packT) (void)hipFree(d_packT);
    if (d_tab) (void)hipFree(d_tab);
  }
};

void tree_state_free(TreeState* s) { delete s; }
void tree_state_stale(TreeState* s) {
  if (s) {
    s->packed = false;
    s->packedT = false;
    s->tab_digits = 0;
  }
}

// A network's packed cores and tables may be used from any stream (and through
// another context) right after the call that queued them: a call on another
// stream waits on the device for what was made last.  Nothing built is written
// again while it is valid, so uses need no such mark.
static int tree_enter(qtt_ctx* ctx, qtt_net* net) {
  if (!net->tree && !(net->tree = new (std::nothrow) TreeState)) return qtt_fail(ctx, QTT_ENOMEM, "host allocation");
  TreeState& S = *net->tree;
  if (!S.ev_stream || S.ev_stream == ctx->stream) return QTT_OK;
  if (hipEventQuery(S.ev) == hipSuccess) {
    S.ev_stream = nullptr;
    return QTT_OK;
  }
  (void)hipGetLastError();  // not ready
  return qtt_hip_check(ctx, hipStreamWaitEvent(ctx->stream, S.ev, 0), "tree event");
}

// after a call's work is queued, also when it failed on the way
static int tree_leave(qtt_ctx* ctx, qtt_net* net) {
  TreeState& S = *net->tree;
  if (!S.making) return QTT_OK;
  int rc = QTT_OK;
  if (!S.ev) rc = qtt_hip_check(ctx, hipEventCreateWithFlags(&S.ev, hipEventDisableTiming), "tree event");
  if (!rc) rc = qtt_hip_check(ctx, hipEventRecord(S.ev, ctx->stream), "tree event");
  if (!rc) {
    S.ev_stream = ctx->stream;
    S.making = false;
  }
  return rc;
}

namespace {

int64_t core_stride(const qtt_net* net, int v, int w) {  // stride in core v of the leg toward w
  const HostTopo& t = net->t;
  int64_t s = 1;
  for (int k = t.nch[v] - 1; k >= 0; k--) {
    const int c = t.chs[t.choff[v] + k];
    if (c == w) return s;
    s *= net->bond[c];
  }
  return s * t.sdim[v];  // the parent leg
}

int64_t site_stride(const qtt_net* net, int v) {
  const HostTopo& t = net->t;
  int64_t s = 1;
  for (int k = 0; k < t.nch[v]; k++) s *= net->bond[t.chs[t.choff[v] + k]];
  return s;
}

// Orientation, shapes and the packed copy (once per network state).
int tree_pack(qtt_ctx* ctx, qtt_net* net) {
  TreeState& S = *net->tree;
  if (S.packed) return QTT_OK;
  const HostTopo& t = net->t;
  S.tab_digits = 0;
  S.centre = choose_centre(net);
  S.vp.assign(t.nv, VPlan());
  S.order.clear();
  // breadth first from the centre, then reversed: inputs come before users
  std::vector<int> bfs;
  if (S.centre < 0) {
    bfs.push_back(0);
  } else {
    const int a = S.centre, b = t.parent[a];
    S.vp[a].to = b;
    S.vp[b].to = a;
    bfs = {a, b};
  }
  for (size_t h = 0; h < bfs.size(); h++) {
    const int v = bfs[h];
    for (int w : neighbours(t, v))
      if (w != S.vp[v].to) {
        S.vp[v].in.push_back(w);
        S.vp[w].to = v;
        bfs.push_back(w);
      }
  }
  S.order.assign(bfs.rbegin(), bfs.rend());
  int64_t tot = 0;
  for (int v : S.order) {
    VPlan& p = S.vp[v];
    p.n = p.to < 0 ? 1 : (int)edge_dim(net, v, p.to);
    const int tiles = (p.n + 15) / 16;
    p.ngrp = (tiles + 3) / 4;
    p.nt = (tiles + p.ngrp - 1) / p.ngrp;
    p.npad = p.ngrp * p.nt * 16;
    p.nd = t.vcoord[v] >= 0;
    p.level = 0;
    int64_t q = 1;
    if (!p.in.empty()) {  // the largest input leg last (the padded one)
      size_t big = 0;
      for (size_t i = 0; i < p.in.size(); i++)
        if (edge_dim(net, v, p.in[i]) > edge_dim(net, v, p.in[big])) big = i;
      std::swap(p.in[big], p.in.back());
      p.big = (int)big;
    }
    for (size_t i = 0; i < p.in.size(); i++) {
      const int w = p.in[i];
      p.nd += S.vp[w].nd;
      p.level = std::max(p.level, S.vp[w].level + 1);
      const int64_t dim = edge_dim(net, v, w);
      if (i + 1 < p.in.size()) q *= dim;
      else p.kbl = (int)((dim + 15) / 16);
    }
    if (q * p.kbl >= (int64_t(1) << 30)) return qtt_fail(ctx, QTT_EINVAL, "evaluate: a core is too large");
    p.nk = (int)(q * p.kbl);
    p.slices = t.vcoord[v] >= 0 ? 2 : 1;
    p.pack = tot;
    tot += (int64_t)p.slices * p.nk * p.npad * 16;
    p.fits = p.nd <= TREE_BITS && (int64_t(p.npad) << p.nd) <= (int64_t(1) << 21);
    for (int w : p.in) p.fits = p.fits && S.vp[w].fits;
  }
  int64_t tabs = 0;
  for (int nd = 0; nd <= TREE_BITS; nd++)
    for (int v : S.order) {
      VPlan& p = S.vp[v];
      if (!p.fits || p.nd != nd) continue;
      p.tab = tabs;
      tabs += int64_t(p.npad) << nd;
    }
  S.making = true;
  if (S.pack_cap < tot) {
    if (S.d_pack) (void)hipFree(S.d_pack);
    S.d_pack = nullptr;
    S.pack_cap = 0;
    const int rc = qtt_hip_check(ctx, hipMalloc(&S.d_pack, tot * sizeof(double)), "hipMalloc packed tree");
    if (rc) return rc;
    S.pack_cap = tot;
  }
  for (int i0 = 0; i0 < t.nv; i0 += 16) {
    TreePackJobs js;
    js.n = std::min(16, t.nv - i0);
    int64_t most = 1;
    for (int i = 0; i < js.n; i++) {
      const int v = i0 + i;
      const VPlan& p = S.vp[v];
      TreePackJob& J = js.job[i];
      J.T = net->d_data + net->off[v];
      J.P = S.d_pack + p.pack;
      J.total = (int64_t)p.slices * p.nk * p.npad * 16;
      J.nd = p.slices;
      J.nk = p.nk;
      J.npad = p.npad;
      J.n = p.n;
      J.m = (int)p.in.size();
      J.lpad = p.kbl * 16;
      J.dstr = site_stride(net, v);
      J.nstr = p.to < 0 ? 0 : core_stride(net, v, p.to);
      for (int j = 0; j < J.m; j++) {
        J.dim[j] = (int)edge_dim(net, v, p.in[j]);
        J.str[j] = core_stride(net, v, p.in[j]);
      }
      most = std::max(most, J.total);
    }
    const unsigned nb = (unsigned)std::min<int64_t>((most + 255) / 256, 4096);
    tree_pack_kernel<<<dim3(nb, js.n), 256, 0, ctx->stream>>>(js);
    const int rc = qtt_hip_check(ctx, hipGetLastError(), "tree_pack_kernel");
    if (rc) return rc;
  }
  S.packed = true;
  return QTT_OK;
}

// LDS strides of a job's staged vectors (odd multiples of 16 bytes, so rows
// fall in different banks), 0 where the four wavefronts' rows do not fit
constexpr int TREE_LDS = 18 * 1024;  // doubles
void stage_strides(TreeJob& J) {
  J.ldu = J.m ? J.kbl * 16 + 2 : 0;
  J.ldw = J.m == 2 ? ((J.leg[0].dim + 1) & ~1) + 2 : 0;
  if (64 * (J.ldu + J.ldw) > TREE_LDS) J.ldu = J.ldw = 0;
}
int launch_vertices(qtt_ctx* ctx, const TreeJobs& js, int units) {
  int lds = 0;
  for (int i = 0; i < js.n; i++) lds = std::max(lds, 64 * (js.job[i].ldu + js.job[i].ldw));
  const size_t bytes = lds * sizeof(double);
  const bool wide = js.job[0].nt > 2;
  if (bytes > 60 * 1024) {
    const int rc = qtt_hip_check(ctx, hipFuncSetAttribute(wide ? (const void*)tree_vertex_kernel<true> : (const void*)tree_vertex_kernel<false>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes),
                                 "tree LDS attribute");
    if (rc) return rc;
  }
  if (wide) tree_vertex_kernel<true><<<units, 256, bytes, ctx->stream>>>(js);
  else tree_vertex_kernel<false><<<units, 256, bytes, ctx->stream>>>(js);
  return qtt_hip_check(ctx, hipGetLastError(), "tree_vertex_kernel");
}

// A batch of vertices whose inputs are ready; launched when full or flushed.
struct Level {
  qtt_ctx* ctx;
  TreeJobs js;
  int units = 0;
  double* part;         // partial sums of split products
  int64_t part_used = 0, part_cap;
  struct Sum {
    const double* part;
    int kc;
    int64_t n;
    double* out;
  };
  std::vector<Sum> sums;
  Level(qtt_ctx* c, double* p, int64_t cap) : ctx(c), part(p), part_cap(cap) { js.n = 0; }
  int flush() {
    if (js.n) {
      const int rc = launch_vertices(ctx, js, units);
      if (rc) return rc;
    }
    for (const Sum& s : sums) {
      const unsigned nb = (unsigned)std::min<int64_t>((s.n + 255) / 256, 2048);
      tree_sum_kernel<<<nb, 256, 0, ctx->stream>>>(s.part, s.kc, s.n, s.out);
      int rc = qtt_hip_check(ctx, hipGetLastError(), "tree_sum_kernel");
      if (rc) return rc;
    }
    js.n = 0;
    units = 0;
    part_used = 0;
    sums.clear();
    return QTT_OK;
  }
  // Rows per workgroup.  Table rows of one digit are whole tiles: 128 rows are
  // two tiles per wavefront, and 64, one, while that leaves compute units idle
  // (a level is then one chain of loads and products shorter: 13.5 -> 8.3 us
  // for 2^8 .. 2^13 rows of bond 32).  Point rows, split by digit, leave a part
  // tile: 112 rows are 8 tiles at most, 48 are 4 (128 rows were 9, three rounds
  // of the four wavefronts).
  static int rows_per(const qtt_ctx* ctx, int64_t R, int ngrp, bool points) {
    const bool few = ((R + 111) / 112) * ngrp < ctx->cus;
    return points ? (few ? 48 : 112) : ((R + 127) / 128) * ngrp < 2 * ctx->cus ? 64 : 128;
  }
  // chunks of a vertex's k blocks: more workgroups when its rows and columns
  // alone leave compute units idle, each with at least 8 blocks of 16
  static int chunks(const qtt_ctx* ctx, const VPlan& p, int64_t R) {
    const int rpw = rows_per(ctx, R, p.ngrp, !p.table);
    const int64_t u = ((R + rpw - 1) / rpw) * p.ngrp;
    const int64_t want = (2 * (int64_t)ctx->cus) / std::max<int64_t>(1, u);
    return (int)std::max<int64_t>(1, std::min<int64_t>(want, p.nk / 8));
  }
  int add(const VPlan& p, TreeJob& J) {
    const int64_t R = J.R;
    J.kc = chunks(ctx, p, R);
    J.kper = (p.nk + J.kc - 1) / J.kc;
    J.kc = (p.nk + J.kper - 1) / J.kper;
    J.rpw = rows_per(ctx, R, p.ngrp, !p.table);
    stage_strides(J);
    const int64_t n = R * p.npad;
    if (js.n == TREE_JOBS || (js.n && (js.job[0].nt > 2) != (J.nt > 2)) || (J.kc > 1 && part_used + n * J.kc > part_cap)) {
      const int rc = flush();
      if (rc) return rc;
    }
    if (J.kc > 1) {
      sums.push_back({part + part_used, J.kc, n, J.out});
      J.out = part + part_used;
      part_used += n * J.kc;
    }
    js.unit0[js.n] = units;
    units += (int)((R + J.rpw - 1) / J.rpw) * p.ngrp * J.kc;
    js.job[js.n++] = J;
    return QTT_OK;
  }
};

// the digits behind v's output leg in the order of its table index, top first
void table_digits(const qtt_net* net, const TreeState& S, int v, std::vector<int>& out) {
  if (net->t.vcoord[v] >= 0) out.push_back(v);
  for (int w : S.vp[v].in) table_digits(net, S, w, out);
}

// One call's rows: which vertices are tables, where the vectors of point rows,
// table entries and partial sums lie in the scratch.
struct Call {
  qtt_ctx* ctx;
  qtt_net* net;
  TreeState& S;
  int64_t npts, chunk = 0, per = 0, kpart = 0;
  int digits = 0, most_level = 0;
  bool any_point = false;
  std::vector<int> frontier, front_of;  // tables used by a point vertex or the final product
  double *pbuf = nullptr, *part = nullptr;
  int* idx = nullptr;
  Call(qtt_ctx* c, qtt_net* n, int64_t np) : ctx(c), net(n), S(*n->tree), npts(np) {}

  // Tables: a vertex with nd digits behind it is a table when 2^nd <= npts / 2
  // (its rows then cost at most half of a row per point, also on a call that
  // builds them), nd <= 16 and the table holds at most 2^21 doubles (the choice
  // does not depend on what is built already, so neither do the values).  copies:
  // buffers per point vertex (the chunk of points keeps them near 512 MiB).
  int plan(int copies) {
    const HostTopo& t = net->t;
    int limit = 0;
    while (limit < TREE_BITS && (int64_t(4) << limit) <= npts) ++limit;
    int64_t tabs = 0;
    front_of.assign(t.nv, -1);
    for (int v : S.order) {
      VPlan& p = S.vp[v];
      p.table = p.fits && p.nd <= limit;
      if (p.table) {
        p.buf = p.tab;
        tabs += int64_t(p.npad) << p.nd;  // (the tables of at most this many digits lie in front)
        digits = std::max(digits, p.nd + 1);
      } else {
        any_point = true;
        p.buf = per;
        per += p.npad;
      }
      most_level = std::max(most_level, p.level);
    }
    for (int v : S.order) {
      const VPlan& p = S.vp[v];
      const bool last = p.to < 0 || v == S.centre || t.parent[S.centre] == v;
      if (p.table && (last || !S.vp[p.to].table)) {
        front_of[v] = (int)frontier.size();
        frontier.push_back(v);
      }
    }
    if (S.tab_cap < tabs) {
      if (S.d_tab) (void)hipFree(S.d_tab);
      S.d_tab = nullptr;
      S.tab_cap = 0;
      S.tab_digits = 0;
      const int rc = qtt_hip_check(ctx, hipMalloc(&S.d_tab, tabs * sizeof(double)), "hipMalloc tree tables");
      if (rc) return rc;
      S.tab_cap = tabs;
    }
    chunk = npts;
    if (per > 0)
      chunk = std::max<int64_t>(TREE_ROWS, std::min<int64_t>(npts, ((int64_t(1) << 26) / (per * copies)) & ~int64_t(TREE_ROWS - 1)));
    chunk = std::min<int64_t>(chunk, int64_t(1) << 24);
    // (Level::chunks: rows x chunks is at most 2 cus TREE_ROWS per column group)
    for (int v : S.order)
      if (S.vp[v].nk >= 16) kpart = std::max<int64_t>(kpart, 2 * (int64_t)ctx->cus * TREE_ROWS * 16 * S.vp[v].nt);
    kpart = std::max<int64_t>(kpart * 2, 16);
    return QTT_OK;
  }
  size_t bytes() const {
    return (size_t)(per * chunk + kpart) * sizeof(double) + (size_t)frontier.size() * chunk * sizeof(int) + 256;
  }
  char* place(char* p) {
    pbuf = (double*)p;
    part = pbuf + per * chunk;
    idx = (int*)(part + kpart);
    return p + bytes();
  }

  TreeJob make_job(int v, int64_t nrows, const double* x0) const {
    const HostTopo& t = net->t;
    const VPlan& p = S.vp[v];
    TreeJob J;
    std::memset(&J, 0, sizeof(J));
    J.P = S.d_pack + p.pack;
    J.dstride = (int64_t)p.nk * p.npad * 16;
    J.R = p.table ? 1 << p.nd : (int)nrows;
    J.n = p.n;
    J.npad = p.npad;
    J.nt = p.nt;
    J.ngrp = p.ngrp;
    J.m = (int)p.in.size();
    J.kbl = p.kbl;
    J.nk = p.nk;
    J.big = t.chain ? -1 : p.big;
    const int c = t.vcoord[v];
    J.out = p.table ? S.d_tab + p.buf : pbuf + p.buf * nrows;
    if (c >= 0) {
      J.dmode = p.table ? 1 : 2;
      J.dshift = p.table ? p.nd - 1 : t.ndigits[c] - t.vdigit[v];
      J.coord = c;
      J.nc = t.ncoord;
      J.ndig = t.ndigits[c];
      J.xs = x0;
    }
    int sh = p.nd - (c >= 0);
    for (int j = 0; j < J.m; j++) {
      const VPlan& pw = S.vp[p.in[j]];
      if (p.table) {
        sh -= pw.nd;
        J.leg[j] = {S.d_tab + pw.buf, nullptr, pw.npad, pw.n, sh, (1 << pw.nd) - 1};
      } else {
        J.leg[j] = point_leg(p.in[j], nrows);
      }
    }
    return J;
  }
  // the vectors of vertex v per point
  TreeLeg point_leg(int v, int64_t nrows) const {
    const VPlan& p = S.vp[v];
    if (p.table) return {S.d_tab + p.buf, idx + front_of[v] * chunk, p.npad, p.n, 0, 0};
    return {pbuf + p.buf * nrows, nullptr, p.npad, p.n, 0, -1};
  }
  // the vertices whose rows are points, or tables of at least `from` digits
  int forward(bool table, int from, int64_t nrows, const double* x0) {
    Level lv(ctx, part, kpart);
    for (int l = 0; l <= most_level; l++) {
      for (int v : S.order) {
        const VPlan& p = S.vp[v];
        if (p.level != l || p.table != table || p.nd < from) continue;
        TreeJob J = make_job(v, nrows, x0);
        const int r = lv.add(p, J);
        if (r) return r;
      }
      const int r = lv.flush();
      if (r) return r;
    }
    return QTT_OK;
  }
  int tables() {  // once per network state
    if (S.tab_digits >= digits) return QTT_OK;
    S.making = true;
    const int rc = forward(true, S.tab_digits, 0, nullptr);
    if (!rc) S.tab_digits = digits;
    return rc;
  }
  int index(int64_t np, const double* x0) {
    const HostTopo& t = net->t;
    for (size_t f0 = 0; f0 < frontier.size(); f0 += TREE_TABLES) {
      TreeIndexArgs a;
      a.n = (int)std::min<size_t>(TREE_TABLES, frontier.size() - f0);
      for (int i = 0; i < a.n; i++) {
        std::vector<int> ds;
        table_digits(net, S, frontier[f0 + i], ds);
        a.t[i].out = idx + (f0 + i) * chunk;
        a.t[i].nbits = (int)ds.size();
        for (size_t b = 0; b < ds.size(); b++) {
          const int c = t.vcoord[ds[b]];
          a.t[i].coord[b] = (unsigned short)c;
          a.t[i].shift[b] = (unsigned char)(t.ndigits[c] - t.vdigit[ds[b]]);
        }
      }
      tree_index_kernel<<<(unsigned)((np + 255) / 256), 256, 0, ctx->stream>>>(a, x0, np, t.ncoord,
                                                                            net->view().ndigits);
      const int rc = qtt_hip_check(ctx, hipGetLastError(), "tree_index_kernel");
      if (rc) return rc;
    }
    return QTT_OK;
  }
};

}  // namespace

static int eval_tree(qtt_ctx* ctx, qtt_net* net, const double* xs, int64_t npts, double* out) {
  const HostTopo& t = net->t;
  int rc = tree_pack(ctx, net);
  if (rc) return rc;
  Call c(ctx, net, npts);
  if ((rc = c.plan(1))) return rc;
  char* scr = (char*)qtt_scratch(ctx, c.bytes());
  if (!scr) return qtt_fail(ctx, QTT_ENOMEM, "evaluate: scratch");
  c.place(scr);
  if ((rc = c.tables())) return rc;
  const int nc = t.ncoord, centre = c.S.centre;
  for (int64_t p0 = 0; p0 < npts; p0 += c.chunk) {
    const int64_t np = std::min(c.chunk, npts - p0);
    const double* x0 = xs + p0 * nc;
    if ((rc = c.index(np, x0))) return rc;
    if (c.any_point && (rc = c.forward(false, 0, np, x0))) return rc;
    const TreeLeg a = c.point_leg(centre < 0 ? 0 : centre, np);
    TreeLeg b;
    std::memset(&b, 0, sizeof(b));
    if (centre >= 0) b = c.point_leg(t.parent[centre], np);
    tree_dot_kernel<<<(unsigned)((np + 15) / 16), 256, 0, ctx->stream>>>(a, b, !t.chain, x0, np, nc, out + p0,
                                                                   ctx->flags());
    if ((rc = qtt_hip_check(ctx, hipGetLastError(), "tree_dot_kernel"))) return rc;
  }
  return QTT_OK;
}

int launch_eval_tree(qtt_ctx* ctx, qtt_net* net, const double* xs, int64_t npts, double* out) {
  int rc = tree_enter(ctx, net);
  if (rc) return rc;
  rc = eval_tree(ctx, net, xs, npts, out);
  // queued only: work on another stream that takes the scratch, or what was made
  // for the network, waits for it
  const int rl = tree_leave(ctx, net), rq = qtt_scratch_queued(ctx);
  return rc ? rc : rl ? rl : rq;
}

// ---------------------------------------------------------------------------
// Gradient of sum_m ybar_m f(x_m) with respect to the cores of a chain: the
// reverse of the vertex products above.  With S_v the derivative with respect
// to v's vectors (one row per row of v),
//     at the centre      S_a[row] = sum over the points with that row of ybar u_b,
//     dT_v[n][d][k]    = sum over the rows with digit d of S_v[row][n] A_v[row][k],
//     S_w[row of w][k] = sum over v's rows on it of sum_n S_v[row][n] T_v[n][d][k].
// On table rows all points that share the digits are one row, so only the
// sites between the two tables are worked through per point.
//
// Points are gathered onto table rows without atomics: a stable radix sort of
// the points by table entry, then runs of equal entries summed in point order
// (pieces of a run that spans several groups of lanes added in order), so the
// result does not depend on timing.
//
// 2^20 points of a 28-site chain of bond 32 (tables of 14 digits on both
// sides): 0.40 ms (0.59 with the tables built) against 24.3 ms with every environment formed per point
// (168 GFLOP and both digit slices).
// ---------------------------------------------------------------------------
namespace {

constexpr int SORT_BITS = 8, SORT_BINS = 1 << SORT_BITS;
constexpr int GRAD_KEYS = 2;       // tables that points meet (one per side of the centre)
constexpr int RUN = 64;            // sorted positions summed by one group of lanes

// ybar, zero (and the flag) at points with a negative or NaN coordinate.  An
// infinite weight sets *inf, a word of host memory that is read once the call
// has waited: here a weight meets the row of one side before that row passes
// the other side's cores, whose sums would turn infinities of both signs into NaN.
__global__ void __launch_bounds__(256)
grad_weight_kernel(const double* __restrict__ xs, const double* __restrict__ ybar, int64_t npts, int nc,
                   double* __restrict__ w, int* __restrict__ flag, int* __restrict__ inf) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= npts) return;
  bool bad = false;
  for (int c = 0; c < nc; ++c)
    if (!(xs[p * nc + c] >= 0.0)) bad = true;
  if (bad) flag[0] = 1;
  const double y = bad ? 0.0 : ybar[p];
  if (isinf(y)) *inf = 1;
  w[p] = y;
}

__global__ void grad_zero_kernel(double* __restrict__ a, int64_t na, unsigned char* __restrict__ b, int64_t nb) {
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, st = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = i0; i < na; i += st) a[i] = 0.0;
  for (int64_t i = i0; i < nb; i += st) b[i] = 0;
}

// One pass of the sort: a wavefront counts the digits of its seg consecutive
// positions; one wavefront per digit scans that digit's counts over the
// wavefronts; a wavefront then places its positions 64 at a time, a lane's
// rank among equal digits from ballots.  What the sums read of a point (the row
// of the other side's vectors, the weight) travels with its key, 16 bytes in
// all, so nothing is gathered by point afterwards.
struct SortRec {  // table row, row of u, weight
  int key, r;
  double w;
};
struct SortArgs {
  const int* key[GRAD_KEYS];     // first pass (in null): keys,
  const int* idx[GRAD_KEYS];     // rows of u (null: the point itself),
  const double* w[GRAD_KEYS];    // weights (null: 1)
  const SortRec* in[GRAD_KEYS];
  SortRec* out[GRAD_KEYS];
  int* cnt[GRAD_KEYS];           // [bin][wavefront], then the digits' totals
  int n, seg, nw, shift;
};

__global__ void __launch_bounds__(256) sort_count_kernel(SortArgs a) {
  __shared__ int h[4][SORT_BINS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, w = blockIdx.x * 4 + wv;
  const int* __restrict__ key = a.key[blockIdx.y];
  const SortRec* __restrict__ in = a.in[blockIdx.y];
  for (int b = lane; b < SORT_BINS; b += 64) h[wv][b] = 0;
  __syncthreads();
  const int p0 = w * a.seg, p1 = min(a.n, p0 + a.seg);
  for (int p = p0 + lane; p < p1; p += 64)
    atomicAdd(&h[wv][((in ? in[p].key : key[p]) >> a.shift) & (SORT_BINS - 1)], 1);
  __syncthreads();
  if (w < a.nw)
    for (int b = lane; b < SORT_BINS; b += 64) a.cnt[blockIdx.y][b * a.nw + w] = h[wv][b];
}

// counts of one digit -> exclusive sums over the wavefronts, and their total
__global__ void __launch_bounds__(256) sort_scan_kernel(SortArgs a) {
  const int lane = threadIdx.x & 63, b = blockIdx.x * 4 + (threadIdx.x >> 6);
  int* __restrict__ c = a.cnt[blockIdx.y] + (int64_t)b * a.nw;
  int run = 0;
  for (int i0 = 0; i0 < a.nw; i0 += 64) {
    const int v = i0 + lane < a.nw ? c[i0 + lane] : 0;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (i0 + lane < a.nw) c[i0 + lane] = run + x - v;
    run += __shfl(x, 63);
  }
  if (lane == 0) a.cnt[blockIdx.y][(int64_t)SORT_BINS * a.nw + b] = run;
}

__global__ void __launch_bounds__(256) sort_place_kernel(SortArgs a) {
  __shared__ int at[4][SORT_BINS];
  __shared__ int ws[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, w = blockIdx.x * 4 + wv, k = blockIdx.y;
  const SortRec* __restrict__ in = a.in[k];
  {  // where each digit starts: exclusive sums of the 256 totals
    const int v = a.cnt[k][(int64_t)SORT_BINS * a.nw + tid];
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (lane == 63) ws[wv] = x;
    __syncthreads();
    int base = x - v;
    for (int i = 0; i < wv; ++i) base += ws[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ww = blockIdx.x * 4 + i;
      if (ww < a.nw) at[i][tid] = base + a.cnt[k][(int64_t)tid * a.nw + ww];
    }
  }
  __syncthreads();
  const int p0 = w * a.seg, p1 = min(a.n, p0 + a.seg);
  for (int q = p0; q < p1; q += 64) {
    const int p = q + lane;
    const bool on = p < p1;
    SortRec rec = {0, 0, 0.0};
    if (on) {
      if (in) rec = in[p];
      else rec = {a.key[k][p], a.idx[k] ? a.idx[k][p] : p, a.w[k] ? a.w[k][p] : 1.0};
    }
    const int d = (rec.key >> a.shift) & (SORT_BINS - 1);
    uint64_t same = __ballot(on);
#pragma unroll
    for (int b = 0; b < SORT_BITS; ++b) {
      const uint64_t m = __ballot((d >> b) & 1);
      same &= ((d >> b) & 1) ? m : ~m;
    }
    const int rank = __popcll(same & ((uint64_t(1) << lane) - 1));
    int base = 0;
    if (on) base = at[wv][d];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // every lane has read before the count moves on
    if (on && rank == 0) at[wv][d] = base + __popcll(same);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (on) a.out[k][base + rank] = rec;
  }
}

// Sums of runs of equal keys: S[row][e] += sum over the run of w u[r][e].  A
// group of G lanes (e = lane) takes RUN sorted positions; a run that began
// in an earlier group goes to head[group], one that continues in the next to
// tail[group], a run inside the group straight to S.  seen[row] = 1.
struct RunArgs {
  const SortRec* rec;
  const double* u;
  int stride;
  int n, width;     // sorted positions; doubles per row (16, 32, 48 or 64)
  int dim;          // entries of u's rows (a row's padding stays zero beside an infinite weight)
  double *S, *head, *tail;
  unsigned char* seen;
};
struct RunJobs {
  RunArgs j[GRAD_KEYS];
};

template <int G>
__device__ __forceinline__ void run_group(const RunArgs& a, int grp, int e) {
  const int q0 = grp * RUN, q1 = min(a.n, q0 + RUN);
  if (q0 >= a.n) return;
  const bool eon = e < a.width, uon = e < a.dim;
  const int before = q0 ? a.rec[q0 - 1].key : -1, after = q1 < a.n ? a.rec[q1].key : -1;
  int cur = a.rec[q0].key;
  bool first = true;  // still in the group's first run
  double acc = 0.0;
  auto flush = [&](bool last) {
    if (first && cur == before) {
      if (eon) a.head[(int64_t)grp * a.width + e] = acc;
    } else if (last && cur == after) {
      if (eon) a.tail[(int64_t)grp * a.width + e] = acc;
    } else if (eon) {
      a.S[(int64_t)cur * a.width + e] += acc;
    }
    if (e == 0) a.seen[cur] = 1;
    first = false;
  };
  for (int q = q0; q < q1; q += 8) {
    int row[8];
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int qq = min(q + i, q1 - 1);
      const SortRec rec = a.rec[qq];
      row[i] = rec.key;
      x[i] = uon ? rec.w * a.u[(int64_t)rec.r * a.stride + e] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (q + i < q1) {
        if (row[i] != cur) {
          flush(false);
          cur = row[i];
          acc = 0.0;
        }
        acc += x[i];
      }
    }
  }
  flush(true);
}

template <int G>
__global__ void __launch_bounds__(256) run_sum_kernel(RunJobs js) {
  const RunArgs& a = js.j[blockIdx.y];
  run_group<G>(a, (int)blockIdx.x * (256 / G) + (int)threadIdx.x / G, threadIdx.x & (G - 1));
}

// the runs that span groups: the group where such a run begins adds its pieces in order
template <int G>
__global__ void __launch_bounds__(256) run_join_kernel(RunJobs js) {
  const RunArgs& a = js.j[blockIdx.y];
  const int grp = (int)blockIdx.x * (256 / G) + (int)threadIdx.x / G, e = threadIdx.x & (G - 1);
  const int q0 = grp * RUN, q1 = q0 + RUN;
  if (q1 >= a.n) return;
  const int row = a.rec[q1 - 1].key;
  if (a.rec[q1].key != row) return;                              // the last run ends here
  if (q0 && a.rec[q0].key == row && a.rec[q0 - 1].key == row) return;  // and began before this group
  double s = e < a.width ? a.tail[(int64_t)grp * a.width + e] : 0.0;
  const int last = (a.n + RUN - 1) / RUN - 1;
  for (int g = grp + 1; g <= last && a.rec[(int64_t)g * RUN].key == row; g += 8) {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int gg = min(g + i, last);
      x[i] = (g + i <= last && e < a.width && a.rec[(int64_t)gg * RUN].key == row) ? a.head[(int64_t)gg * a.width + e] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) s += x[i];
  }
  if (e < a.width) a.S[(int64_t)row * a.width + e] += s;
}

// S[p][e] = w[p] u(p)[e] for point rows at the centre (zero in the padding)
__global__ void __launch_bounds__(256)
point_scale_kernel(const double* __restrict__ w, TreeLeg u, int64_t n, double* __restrict__ S) {
  const int64_t total = n * u.stride;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t p = i / u.stride;
    const int e = (int)(i - p * u.stride);
    const int r = u.idx ? u.idx[p] : (int)p;
    S[i] = e < u.dim ? w[p] * u.u[(int64_t)r * u.stride + e] : 0.0;
  }
}

// S[p][0] = w[p], the rest of the 16-wide row zero: a network of one vertex
__global__ void __launch_bounds__(256)
point_unit_kernel(const double* __restrict__ w, int64_t n, double* __restrict__ S) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < 16 * n) S[i] = (i & 15) ? 0.0 : w[i >> 4];
}

// dT of one vertex: part[c][d][n][k] = sum over this part's rows with digit d
// of S[row][n] A[row][k], as FP64 MFMA tiles with the rows as k.  A workgroup
// takes blocks of 128 rows sorted by digit (as tree_vertex_kernel); wavefronts
// 0, 1 have digit 0, wavefronts 2, 3 digit 1, alternate 16-row groups, every
// tile of the slice in registers; each writes its own part.
struct CoreJob {
  const double* S;
  TreeLeg u;           // A's rows (u null: A = 1, a leaf)
  const double* xs;
  const unsigned char* seen;  // table rows that occur, or null
  double* part;
  int R, lds, tn, tk;  // rows; S's row stride; tiles of n and k
  int dmode, dshift, coord, nc, ndig;
  int blocks, nwg;     // 128-row blocks per workgroup, workgroups
};
constexpr int CORE_JOBS = 32;
struct CoreJobs {
  int n;
  int unit0[CORE_JOBS];
  CoreJob job[CORE_JOBS];
};
static_assert(sizeof(CoreJobs) <= 4096, "kernel arguments");

template <int T>
__device__ __forceinline__ void core_tiles(const CoreJob& J, const int* rows, int n0, int n1, f64x4 (&acc)[T][T]) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int t0 = (n0 + 15) >> 4, t1 = (n1 + 15) >> 4;
  const int g0 = wv >> 1 ? t0 : 0, g1 = wv >> 1 ? t0 + t1 : t0;
  for (int g = g0 + (wv & 1); g < g1; g += 2) {
    double a[T][4], b[T][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rows[g * 16 + 4 * lk + i];
      const bool on = r >= 0 && (!J.seen || J.seen[r]);  // a row without points counts as zero
      const int rr = r < 0 ? 0 : r;
      const double* s = J.S + (int64_t)rr * J.lds + li;
      const int x = J.u.idx ? J.u.idx[rr] : (rr >> J.u.shift) & J.u.mask;
      const double* u = J.u.u ? J.u.u + (int64_t)x * J.u.stride + li : nullptr;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        a[t][i] = (on && t < J.tn) ? s[16 * t] : 0.0;
        b[t][i] = !on || t >= J.tk ? 0.0 : u ? u[16 * t] : (t == 0 && li == 0) ? 1.0 : 0.0;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int x = 0; x < T; ++x)
#pragma unroll
        for (int y = 0; y < T; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x][i], b[y][i], acc[x][y], 0, 0, 0);
  }
}

template <int T>
__device__ __forceinline__ void core_block(const CoreJob& J, int wg, int* rows, int* cnt) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lk = lane >> 4;
  f64x4 acc[T][T];
#pragma unroll
  for (int x = 0; x < T; ++x)
#pragma unroll
    for (int y = 0; y < T; ++y) acc[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
  for (int bl = 0; bl < J.blocks; ++bl) {
    const int base = (wg * J.blocks + bl) * TREE_ROWS;
    if (base >= J.R) break;
    __syncthreads();
    if (tid < TREE_ROWS + 32) rows[tid] = -1;
    const int row = base + tid;
    const bool on = tid < TREE_ROWS && row < J.R;
    int d = 0;
    if (on && J.dmode == 1) d = (row >> J.dshift) & 1;
    if (on && J.dmode == 2)
      d = (int)((tree_digit_word(J.xs[(int64_t)row * J.nc + J.coord], J.ndig) >> J.dshift) & 1);
    const uint64_t b0 = __ballot(on && d == 0), b1 = __ballot(on && d == 1);
    if (lane == 0 && wv < 2) {
      cnt[2 * wv] = __popcll(b0);
      cnt[2 * wv + 1] = __popcll(b1);
    }
    __syncthreads();
    const int n0 = cnt[0] + cnt[2], n1 = cnt[1] + cnt[3];
    if (on) {
      const uint64_t below = (uint64_t(1) << lane) - 1;
      const int pos = __popcll((d ? b1 : b0) & below) + (wv ? cnt[d] : 0);
      rows[d ? ((n0 + 15) & ~15) + pos : pos] = row;
    }
    __syncthreads();
    core_tiles<T>(J, rows, n0, n1, acc);
  }
  const int np = 16 * J.tn, kp = 16 * J.tk;
  double* out = J.part + ((int64_t)(2 * wg + (wv & 1)) * 2 + (wv >> 1)) * np * kp;
#pragma unroll
  for (int x = 0; x < T; ++x)
#pragma unroll
    for (int y = 0; y < T; ++y)
      if (x < J.tn && y < J.tk)
#pragma unroll
        for (int e = 0; e < 4; ++e) out[(16 * x + lk + 4 * e) * kp + 16 * y + li] = acc[x][y][e];
}

__global__ void __launch_bounds__(256) tree_core_kernel(CoreJobs js) {
  __shared__ int rows[TREE_ROWS + 32];
  __shared__ int cnt[4];
  int jj = 0;
#pragma unroll
  for (int i = 1; i < CORE_JOBS; ++i) jj += (i < js.n && (int)blockIdx.x >= js.unit0[i]) ? 1 : 0;
  const CoreJob& J = js.job[jj];
  const int wg = (int)blockIdx.x - js.unit0[jj], t = max(J.tn, J.tk);
  if (t == 1) core_block<1>(J, wg, rows, cnt);
  else if (t == 2) core_block<2>(J, wg, rows, cnt);
  else if (t == 3) core_block<3>(J, wg, rows, cnt);
  else core_block<4>(J, wg, rows, cnt);
}

// the parts of every vertex added in order into its core's gradient (add: to
// what earlier points left there)
struct CoreSum {
  const double* part;
  double* g;
  int C, n, k, np, kp, sd, slices;
  int64_t nstr, kstr, dstr;
};
struct CoreSums {
  int n, add;
  CoreSum job[CORE_JOBS];
};

__global__ void __launch_bounds__(256) tree_core_sum_kernel(CoreSums js) {
  const CoreSum& J = js.job[blockIdx.y];
  const int total = J.sd * J.n * J.k;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    const int k = i % J.k, r = i / J.k, n = r % J.n, d = r / J.n;
    double s = 0.0;
    if (d < J.slices) {  // (a site without a digit has only its first slice in the values)
      const double* p = J.part + ((int64_t)d * J.np + n) * J.kp + k;
      const int64_t st = (int64_t)2 * J.np * J.kp;
      int c = 0;
      for (; c + 8 <= J.C; c += 8) {
        double x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = p[(c + q) * st];
#pragma unroll
        for (int q = 0; q < 8; ++q) s += x[q];
      }
      for (; c < J.C; ++c) s += p[c * st];
    }
    double* g = J.g + d * J.dstr + n * J.nstr + k * J.kstr;
    *g = js.add ? *g + s : s;
  }
}

// The copy of the cores with output and input leg exchanged (chains: at most
// one input), packed as tree_pack does with k over the output leg.
int tree_pack_transposed(qtt_ctx* ctx, qtt_net* net) {
  TreeState& S = *net->tree;
  if (S.packedT) return QTT_OK;
  S.making = true;
  int64_t tot = 0;
  for (int v : S.order) {
    VPlan& p = S.vp[v];
    p.packT = tot;
    if (!p.in.empty()) tot += (int64_t)p.slices * ((p.n + 15) / 16) * S.vp[p.in[0]].npad * 16;
  }
  if (S.packT_cap < tot) {
    if (S.d_packT) (void)hipFree(S.d_packT);
    S.d_packT = nullptr;
    S.packT_cap = 0;
    const int rc = qtt_hip_check(ctx, hipMalloc(&S.d_packT, tot * sizeof(double)), "hipMalloc packed chain");
    if (rc) return rc;
    S.packT_cap = tot;
  }
  TreePackJobs js;
  js.n = 0;
  int64_t most = 1;
  auto flush = [&]() {
    if (!js.n) return QTT_OK;
    tree_pack_kernel<<<dim3((unsigned)std::min<int64_t>((most + 255) / 256, 4096), js.n), 256, 0, ctx->stream>>>(js);
    js.n = 0;
    most = 1;
    return qtt_hip_check(ctx, hipGetLastError(), "tree_pack_kernel");
  };
  for (int v : S.order) {
    const VPlan& p = S.vp[v];
    if (p.in.empty()) continue;
    const VPlan& pw = S.vp[p.in[0]];
    TreePackJob& J = js.job[js.n++];
    J.T = net->d_data + net->off[v];
    J.P = S.d_packT + p.packT;
    J.nd = p.slices;
    J.nk = (p.n + 15) / 16;
    J.npad = pw.npad;
    J.n = pw.n;
    J.total = (int64_t)J.nd * J.nk * J.npad * 16;
    J.m = 1;
    J.lpad = J.nk * 16;
    J.dstr = site_stride(net, v);
    J.nstr = core_stride(net, v, p.in[0]);
    J.dim[0] = p.n;
    J.str[0] = p.to < 0 ? 0 : core_stride(net, v, p.to);
    most = std::max(most, J.total);
    if (js.n == 16) {
      const int rc = flush();
      if (rc) return rc;
    }
  }
  const int rc = flush();
  if (!rc) S.packedT = true;
  return rc;
}

}  // namespace

static int grad_chain(qtt_ctx* ctx, qtt_net* net, const double* xs, const double* ybar, int64_t npts, double* grad) {
  const HostTopo& t = net->t;
  if (npts == 0) {
    grad_zero_kernel<<<256, 256, 0, ctx->stream>>>(grad, qtt_net_size(net), nullptr, 0);
    return qtt_hip_check(ctx, hipGetLastError(), "grad_zero_kernel");
  }
  int rc = tree_pack(ctx, net);
  if (!rc) rc = tree_pack_transposed(ctx, net);
  if (rc) return rc;
  Call c(ctx, net, npts);
  if ((rc = c.plan(2))) return rc;
  TreeState& S = c.S;
  const int nc = t.ncoord, centre = S.centre, nf = (int)c.frontier.size();
  // scratch after the forward's: the derivatives of point rows and of table
  // rows (both laid out as the vectors), marks of table rows, weights, the
  // sorts, the sums of runs, the parts of the cores' gradients
  int64_t tabs = 0, marks = 0;
  std::vector<int64_t> mark(t.nv, 0), goff(t.nv, 0);
  int64_t o = 0;
  for (int v = 0; v < t.nv; v++) {
    goff[v] = o;
    o += net->core_size(v);
  }
  for (int v : S.order)
    if (S.vp[v].table) {
      tabs += int64_t(S.vp[v].npad) << S.vp[v].nd;
      mark[v] = marks;
      marks += int64_t(1) << S.vp[v].nd;
    }
  const int64_t chunk = c.chunk;
  // a wavefront's share of the sort: at most 1024 wavefronts (2^20 points: 1024 each)
  const int seg = (int)std::max<int64_t>(256, ((chunk + 1023) / 1024 + 63) & ~int64_t(63));
  const int nw = (int)((chunk + seg - 1) / seg);
  const int64_t groups = (chunk + RUN - 1) / RUN;
  int width = 16;
  for (int v : c.frontier) width = std::max(width, S.vp[v].npad);
  // parts: per vertex 2 workgroup halves x 2 digits x the padded slice; at most
  // 64 workgroups per vertex (all vertices of a kind run together), two
  // 128-row blocks each while there are fewer
  auto most_wgs = [](int64_t R) {
    return std::max<int64_t>(1, std::min<int64_t>(64, ((R + TREE_ROWS - 1) / TREE_ROWS + 1) / 2));
  };
  auto core_wgs = [&](int64_t R, int& blocks) {
    const int64_t nb = (R + TREE_ROWS - 1) / TREE_ROWS, wgs = most_wgs(R);
    blocks = (int)((nb + wgs - 1) / wgs);
    return (int)((nb + blocks - 1) / blocks);
  };
  std::vector<int64_t> poff(t.nv, 0);
  int64_t parts = 0;
  for (int v : S.order) {
    const VPlan& p = S.vp[v];
    const int64_t wgs = most_wgs(p.table ? int64_t(1) << p.nd : chunk);
    poff[v] = parts;
    parts += 2 * wgs * 2 * ((p.n + 15) / 16 * 16) * 16 * p.kbl;
  }
  auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t b_sp = al((size_t)c.per * chunk * 8), b_st = al((size_t)tabs * 8), b_mk = al((size_t)marks),
               b_w = al((size_t)chunk * 8), b_srt = al((size_t)chunk * sizeof(SortRec)), b_cnt = al((size_t)SORT_BINS * (nw + 1) * 4),
               b_run = al((size_t)groups * width * 8), b_tmp = al((size_t)chunk * width * 8),
               b_part = al((size_t)parts * 8);
  const bool tmp_needed = c.any_point || centre < 0;  // point rows on their way to a table
  size_t bytes = al(c.bytes()) + b_sp + b_st + b_mk + b_w + b_part + (size_t)nf * (2 * b_srt + b_cnt + 2 * b_run) +
                 (tmp_needed ? (size_t)nf * b_tmp : 0) + 1024;
  char* scr = (char*)qtt_scratch(ctx, bytes);
  if (!scr) return qtt_fail(ctx, QTT_ENOMEM, "gradient scratch");
  c.place(scr);
  char* q = scr + al(c.bytes());
  auto take = [&](size_t b) {
    char* r = q;
    q += b;
    return r;
  };
  double* Sp = (double*)take(b_sp);
  double* St = (double*)take(b_st);
  unsigned char* mk = (unsigned char*)take(b_mk);
  double* wts = (double*)take(b_w);
  double* part = (double*)take(b_part);
  SortRec *ra[GRAD_KEYS], *rb[GRAD_KEYS];
  int* cnt[GRAD_KEYS];
  double *head[GRAD_KEYS], *tail[GRAD_KEYS], *tmp[GRAD_KEYS];
  for (int f = 0; f < nf; f++) {
    ra[f] = (SortRec*)take(b_srt);
    rb[f] = (SortRec*)take(b_srt);
    cnt[f] = (int*)take(b_cnt);
    head[f] = (double*)take(b_run);
    tail[f] = (double*)take(b_run);
    tmp[f] = tmp_needed ? (double*)take(b_tmp) : nullptr;
  }
  if ((rc = c.tables())) return rc;
  for (int v : c.frontier) {  // the tables that points add to (the others' rows are written whole)
    const int64_t rows = int64_t(1) << S.vp[v].nd;
    grad_zero_kernel<<<256, 256, 0, ctx->stream>>>(St + S.vp[v].buf, rows * S.vp[v].npad, mk + mark[v], rows);
    if ((rc = qtt_hip_check(ctx, hipGetLastError(), "grad_zero_kernel"))) return rc;
  }

  std::vector<int> ends;  // the centre's two vertices, or the only one
  if (centre < 0) ends = {0};
  else ends = {centre, t.parent[centre]};
  // the gradient of some vertices' cores (all of point rows, or of table rows)
  auto cores_of = [&](bool table, int64_t np, const double* x0, bool add) -> int {
    std::vector<int> vs;
    for (int v : S.order)
      if (S.vp[v].table == table) vs.push_back(v);
    for (size_t i0 = 0; i0 < vs.size(); i0 += CORE_JOBS) {
      CoreJobs js;
      CoreSums ss;
      js.n = ss.n = (int)std::min<size_t>(CORE_JOBS, vs.size() - i0);
      ss.add = add ? 1 : 0;
      int units = 0, most = 1;
      for (int i = 0; i < js.n; i++) {
        const int v = vs[i0 + i];
        const VPlan& p = S.vp[v];
        const TreeJob f = c.make_job(v, np, x0);
        CoreJob& J = js.job[i];
        std::memset(&J, 0, sizeof(J));
        J.S = table ? St + p.buf : Sp + p.buf * np;
        if (f.m) J.u = f.leg[0];
        J.xs = f.xs;
        J.seen = table ? mk + mark[v] : nullptr;
        J.part = part + poff[v];
        J.R = f.R;
        J.lds = p.npad;
        J.tn = (p.n + 15) / 16;
        J.tk = p.kbl;
        J.dmode = f.dmode;
        J.dshift = f.dshift;
        J.coord = f.coord;
        J.nc = f.nc;
        J.ndig = f.ndig;
        J.nwg = core_wgs(J.R, J.blocks);
        js.unit0[i] = units;
        units += J.nwg;
        CoreSum& Q = ss.job[i];
        Q.part = J.part;
        Q.g = grad + goff[v];
        Q.C = 2 * J.nwg;
        Q.n = p.n;
        Q.k = f.m ? f.leg[0].dim : 1;
        Q.np = 16 * J.tn;
        Q.kp = 16 * J.tk;
        Q.sd = t.sdim[v];
        Q.slices = p.slices;
        Q.dstr = site_stride(net, v);
        Q.nstr = p.to < 0 ? 0 : core_stride(net, v, p.to);
        Q.kstr = f.m ? core_stride(net, v, p.in[0]) : 0;
        most = std::max(most, Q.sd * Q.n * Q.k);
      }
      tree_core_kernel<<<units, 256, 0, ctx->stream>>>(js);
      int r = qtt_hip_check(ctx, hipGetLastError(), "tree_core_kernel");
      if (r) return r;
      tree_core_sum_kernel<<<dim3((most + 255) / 256, ss.n), 256, 0, ctx->stream>>>(ss);
      if ((r = qtt_hip_check(ctx, hipGetLastError(), "tree_core_sum_kernel"))) return r;
    }
    return QTT_OK;
  };
  // the derivative rows of v's input from v's own (points: one row each; tables: both digits)
  auto back_job = [&](int v, int64_t np, const double* x0, double* out) {
    const VPlan& p = S.vp[v];
    const VPlan& pw = S.vp[p.in[0]];
    TreeJob J;
    std::memset(&J, 0, sizeof(J));
    J.P = S.d_packT + p.packT;
    J.nk = J.kbl = (p.n + 15) / 16;
    J.dstride = (int64_t)J.nk * pw.npad * 16;
    J.n = pw.n;
    J.npad = pw.npad;
    J.nt = pw.nt;
    J.ngrp = pw.ngrp;
    J.m = 1;
    J.big = -1;
    J.kc = 1;
    J.kper = J.nk;
    J.out = out;
    if (p.table) {
      J.R = 1 << pw.nd;
      J.two = p.slices;
      J.seen = mk + mark[v];
      J.seen_out = mk + mark[p.in[0]];
      J.leg[0] = {St + p.buf, nullptr, p.npad, p.n, 0, -1};
    } else {
      const TreeJob f = c.make_job(v, np, x0);
      J.R = (int)np;
      J.dmode = f.dmode;
      J.dshift = f.dshift;
      J.coord = f.coord;
      J.nc = f.nc;
      J.ndig = f.ndig;
      J.xs = f.xs;
      J.leg[0] = {Sp + p.buf * np, nullptr, p.npad, p.n, 0, -1};
    }
    return J;
  };
  auto launch_back = [&](std::vector<TreeJob>& jobs) -> int {
    for (size_t i = 0; i < jobs.size();) {  // (at most one vertex per side; equal kernels together)
      TreeJobs js;
      js.n = 0;
      int units = 0;
      const bool wide = jobs[i].nt > 2;
      for (; i < jobs.size() && (jobs[i].nt > 2) == wide; i++) {
        js.unit0[js.n] = units;
        TreeJob& J = js.job[js.n++];
        J = jobs[i];
        J.rpw = Level::rows_per(ctx, J.R, J.ngrp, !J.two);
        stage_strides(J);
        units += (J.R + J.rpw - 1) / J.rpw * J.ngrp;
      }
      const int r = launch_vertices(ctx, js, units);
      if (r) return r;
    }
    jobs.clear();
    return QTT_OK;
  };

  for (int64_t p0 = 0; p0 < npts; p0 += chunk) {
    const int64_t np = std::min(chunk, npts - p0);
    const double* x0 = xs + p0 * nc;
    const unsigned nb = (unsigned)((np + 255) / 256);
    grad_weight_kernel<<<nb, 256, 0, ctx->stream>>>(x0, ybar + p0, np, nc, wts, ctx->flags(), ctx->h_inf);
    if ((rc = qtt_hip_check(ctx, hipGetLastError(), "grad_weight_kernel"))) return rc;
    if ((rc = c.index(np, x0))) return rc;
    if (c.any_point && (rc = c.forward(false, 0, np, x0))) return rc;
    // the values that reach each table, by point
    std::vector<TreeLeg> into(nf);
    std::vector<const double*> wof(nf, nullptr);
    std::vector<int> wave;  // point vertices whose derivative rows are ready
    for (size_t i = 0; i < ends.size(); i++) {
      const int v = ends[i];
      if (ends.size() == 1) {  // its value is its only entry: the derivative is the weight
        const bool table = S.vp[v].table;
        double* dst = table ? tmp[c.front_of[v]] : Sp + S.vp[v].buf * np;
        point_unit_kernel<<<(unsigned)((16 * np + 255) / 256), 256, 0, ctx->stream>>>(wts, np, dst);
        if ((rc = qtt_hip_check(ctx, hipGetLastError(), "point_unit_kernel"))) return rc;
        if (table) into[c.front_of[v]] = {dst, nullptr, 16, 1, 0, -1};
        continue;
      }
      const TreeLeg other = c.point_leg(ends[1 - i], np);
      if (S.vp[v].table) {
        into[c.front_of[v]] = other;
        wof[c.front_of[v]] = wts;
      } else {
        const unsigned g = (unsigned)std::min<int64_t>((np * other.stride + 255) / 256, 65536);
        point_scale_kernel<<<g, 256, 0, ctx->stream>>>(wts, other, np, Sp + S.vp[v].buf * np);
        if ((rc = qtt_hip_check(ctx, hipGetLastError(), "point_scale_kernel"))) return rc;
        wave.push_back(v);
      }
    }
    while (!wave.empty()) {
      std::vector<TreeJob> jobs;
      std::vector<int> next;
      for (int v : wave) {
        if (S.vp[v].in.empty()) continue;
        const int w = S.vp[v].in[0];
        double* out;
        if (S.vp[w].table) {
          const int f = c.front_of[w];
          out = tmp[f];
          into[f] = {out, nullptr, S.vp[w].npad, S.vp[w].n, 0, -1};
        } else {
          out = Sp + S.vp[w].buf * np;
          next.push_back(w);
        }
        jobs.push_back(back_job(v, np, x0, out));
      }
      if ((rc = launch_back(jobs))) return rc;
      wave = next;
    }
    // points sorted by the entry of each table they meet
    int digits = 0;
    for (int v : c.frontier) digits = std::max(digits, S.vp[v].nd);
    const int passes = std::max(1, (digits + SORT_BITS - 1) / SORT_BITS);
    const int nws = (int)((np + seg - 1) / seg);
    for (int ps = 0; ps < passes && nf; ps++) {
      SortArgs a;
      std::memset(&a, 0, sizeof(a));
      for (int f = 0; f < nf; f++) {
        const bool toa = ((passes - 1 - ps) & 1) == 0;  // the last pass leaves the result in ra
        a.key[f] = c.idx + f * chunk;
        a.idx[f] = into[f].idx;
        a.w[f] = wof[f];
        a.in[f] = ps == 0 ? nullptr : toa ? rb[f] : ra[f];
        a.out[f] = toa ? ra[f] : rb[f];
        a.cnt[f] = cnt[f];
      }
      a.n = (int)np;
      a.seg = seg;
      a.nw = nws;
      a.shift = ps * SORT_BITS;
      const dim3 g((nws + 3) / 4, nf);
      sort_count_kernel<<<g, 256, 0, ctx->stream>>>(a);
      sort_scan_kernel<<<dim3(SORT_BINS / 4, nf), 256, 0, ctx->stream>>>(a);
      sort_place_kernel<<<g, 256, 0, ctx->stream>>>(a);
      if ((rc = qtt_hip_check(ctx, hipGetLastError(), "gradient sort"))) return rc;
    }
    for (int f0 = 0; f0 < nf;) {  // tables of equal row width share a launch
      RunJobs js;
      std::memset(&js, 0, sizeof(js));
      const int wd = S.vp[c.frontier[f0]].npad;
      int n = 0, f = f0;
      for (; f < nf && S.vp[c.frontier[f]].npad == wd; f++, n++) {
        RunArgs& a = js.j[n];
        a.rec = ra[f];
        a.u = into[f].u;
        a.stride = into[f].stride;
        a.n = (int)np;
        a.width = wd;
        a.dim = into[f].dim;
        a.S = St + S.vp[c.frontier[f]].buf;
        a.head = head[f];
        a.tail = tail[f];
        a.seen = mk + mark[c.frontier[f]];
      }
      f0 = f;
      const int64_t grps = (np + RUN - 1) / RUN;
      auto blocks = [&](int G) { return dim3((unsigned)((grps + 256 / G - 1) / (256 / G)), n); };
      if (wd == 16) {
        run_sum_kernel<16><<<blocks(16), 256, 0, ctx->stream>>>(js);
        run_join_kernel<16><<<blocks(16), 256, 0, ctx->stream>>>(js);
      } else if (wd == 32) {
        run_sum_kernel<32><<<blocks(32), 256, 0, ctx->stream>>>(js);
        run_join_kernel<32><<<blocks(32), 256, 0, ctx->stream>>>(js);
      } else {
        run_sum_kernel<64><<<blocks(64), 256, 0, ctx->stream>>>(js);
        run_join_kernel<64><<<blocks(64), 256, 0, ctx->stream>>>(js);
      }
      if ((rc = qtt_hip_check(ctx, hipGetLastError(), "run_sum_kernel"))) return rc;
    }
    if (c.any_point && (rc = cores_of(false, np, x0, p0 > 0))) return rc;
  }
  // down the tables, both sides together
  std::vector<int> wave;
  for (int v : c.frontier) wave.push_back(v);
  while (!wave.empty()) {
    std::vector<TreeJob> jobs;
    std::vector<int> next;
    for (int v : wave) {
      if (S.vp[v].in.empty()) continue;
      const int w = S.vp[v].in[0];
      jobs.push_back(back_job(v, 0, nullptr, St + S.vp[w].buf));
      next.push_back(w);
    }
    if ((rc = launch_back(jobs))) return rc;
    wave = next;
  }
  if ((rc = cores_of(true, 0, nullptr, false))) return rc;
  rc = qtt_hip_check(ctx, hipStreamSynchronize(ctx->stream), "grad sync");
  if (!rc) {  // what it made, and what it waited for in tree_enter, is done: nothing to order by an event
    S.making = false;
    S.ev_stream = nullptr;
  }
  return rc;
}

int launch_grad_chain(qtt_ctx* ctx, qtt_net* net, const double* xs, const double* ybar, int64_t npts, double* grad,
                      bool* inf_weight) {
  int rc = tree_enter(ctx, net);
  if (rc) return rc;
  *ctx->h_inf = 0;  // (a call that failed half-way may set it late: the other kernel runs, the results are right)
  rc = grad_chain(ctx, net, xs, ybar, npts, grad);
  const int rl = tree_leave(ctx, net);
  if (!rc) {
    *inf_weight = *(volatile int*)ctx->h_inf != 0;
    return rl;
  }
  const int rq = qtt_scratch_queued(ctx);  // it may have failed with work queued
  (void)rq;
  return rc;
}
