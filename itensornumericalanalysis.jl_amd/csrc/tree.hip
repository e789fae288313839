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
// network, like its packed chain copy, until the cores change.  Above the limit
// the rows are the points.  A table's row index has the vertex's own digit as
// its top bit, then its input tables' indices.
//
// The product.  Rows of one digit use one slice of the core, so a workgroup
// sorts the 128 rows it takes by digit (two ballots) and cuts both halves into
// 16-row tiles: no slice is computed and thrown away.  Tiles are FP64 MFMA,
// v_mfma_f64_16x16x4f64 (lane l: A[l%16][l/16], B[l/16][l%16], D[l/16 + 4e]
// [l%16]).  The order of k inside a block of 16 is free as long as A and B
// agree: lane group l/16 takes the 4 consecutive entries 4 (l/16) .. + 3, one
// per MFMA, so both operands come as 32-byte pieces of 128-byte lines.  The
// core is repacked once into 16 x 16 tiles in that order (zero padded, kept
// with the network).  A vertex with few rows and a long k (a comb's backbone:
// 128 x 128 combinations) splits k over workgroups and adds the parts in order.
//
// Measured against one lane per point walking every core entry: 20,011 points
// of a 3 x 16 comb of bond 32, 39.4 -> 0.14 ms (a network's first call 0.35
// ms); 256 points of the bond 128 comb, 1530 -> about 1 ms.  What bounds it: a
// chain of one launch per level (about 5 us each) while the rows are few, the
// FP64 matrix rate at the backbone.
#include "tree.h"

#include <algorithm>
#include <cstring>

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int TREE_MAX_IN = QTT_MAX_NDIM - 2;  // input legs of a vertex
constexpr int TREE_JOBS = 7;                   // vertices per launch (by value: under 4 KB of arguments)
constexpr int TREE_ROWS = 128;                 // rows per workgroup
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
  const double* P;   // packed core [digit][k block][npad][16]
  double* out;       // [R][npad], or partial sums [kc][R][npad]
  const double* xs;  // the points, when the vertex's rows are points and it has a digit
  int64_t dstride;   // doubles of one digit slice of P
  int R, n, npad, nt, ngrp;  // rows; output bond, padded; 16-column tiles per workgroup, groups of them
  int m, kbl, nk;    // input legs (the last one padded to kbl blocks of 16), k blocks in all
  int kc, kper;      // chunks of k blocks (one workgroup each) and blocks per chunk
  int dmode;         // digit of a row: 0 none (slice 0), 1 bit dshift of the row, 2 of a point's coordinate
  int dshift, coord, nc, ndig;
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

// The k blocks [k0, k1) of one 16-row tile against NT 16-column tiles.  ML: 1
// one input leg (or none), 2 two legs, 3 any number.  u: the last leg's row
// of this lane (offset to its 4 entries of a block), w: the other legs' rows
// (row position q of the workgroup's list in wrow).
template <int NT, int ML>
__device__ __forceinline__ void tree_tile(const TreeJob& J, const double* __restrict__ P, const double* __restrict__ u,
                                          const double* __restrict__ w, int lrow, int k0, int k1,
                                          f64x4 (&acc)[NT]) {
  const int lane = threadIdx.x & 63, lk = lane >> 4;
  const int kbl = J.kbl;
  const int64_t bstep = (int64_t)J.npad * 16;
  const double* __restrict__ pb = P + (int64_t)k0 * bstep;
  int q = k0 / kbl, kb = k0 - q * kbl;
  double cf = 1.0;
  auto coef = [&]() {  // product of the other legs' entries of combination q
    if (ML == 1) return;
    if (ML == 2) {
      cf = w[q];
      return;
    }
    int r = q;
    cf = 1.0;
    for (int j = J.m - 2; j >= 0; --j) {
      const TreeLeg& L = J.leg[j];
      const int nq = r / L.dim, i = r - nq * L.dim;
      r = nq;
      const int row = L.idx ? L.idx[lrow] : (lrow >> L.shift) & L.mask;
      cf *= L.u[(int64_t)row * L.stride + i];
    }
  };
  f64x2 a0[2], a1[2], b0[NT][2], b1[NT][2];
  auto load = [&](f64x2 (&a)[2], f64x2 (&b)[NT][2]) {
    if (ML >= 2 && kb == 0) coef();
    if (J.m) {
      a[0] = *(const f64x2*)(u + kb * 16);
      a[1] = *(const f64x2*)(u + kb * 16 + 2);
    } else {
      a[0] = f64x2{lk == 0 ? 1.0 : 0.0, 0.0};
      a[1] = f64x2{0.0, 0.0};
    }
    if (ML >= 2) {
      a[0] *= cf;
      a[1] *= cf;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      b[t][0] = *(const f64x2*)(pb + t * 256);
      b[t][1] = *(const f64x2*)(pb + t * 256 + 2);
    }
    pb += bstep;
    if (++kb == kbl) {
      kb = 0;
      ++q;
    }
  };
  auto mul = [&](const f64x2 (&a)[2], const f64x2 (&b)[NT][2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i >> 1][i & 1], b[t][i >> 1][i & 1], acc[t], 0, 0, 0);
  };
  if (ML >= 2 && kb != 0) coef();
  // the next block's loads are issued before this block's products
  int k = k0;
  load(a0, b0);
  for (; k + 2 <= k1; k += 2) {
    load(a1, b1);
    mul(a0, b0);
    if (k + 2 < k1) load(a0, b0);
    mul(a1, b1);
  }
  if (k < k1) mul(a0, b0);
}

template <int NT>
__device__ __forceinline__ void tree_rows(const TreeJob& J, const int* rows, int n0, int n1, int ng, int kc, int k0,
                                          int k1) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int t0 = (n0 + 15) >> 4, ntile = t0 + ((n1 + 15) >> 4);
  const int c0 = ng * NT * 16;
  double* out = J.out + (int64_t)kc * J.R * J.npad + c0;
  for (int t = wv; t < ntile; t += 4) {
    const int lrow = rows[t * 16 + li];
    const int r = lrow < 0 ? rows[t * 16] : lrow;  // a padding row repeats the tile's first
    const double* P = J.P + (t < t0 ? 0 : J.dstride) + (int64_t)(c0 + li) * 16 + 4 * lk;
    const double *u = nullptr, *w = nullptr;
    if (J.m) {
      const TreeLeg& L = J.leg[J.m - 1];
      const int x = L.idx ? L.idx[r] : (r >> L.shift) & L.mask;
      u = L.u + (int64_t)x * L.stride + 4 * lk;
    }
    if (J.m == 2) {
      const TreeLeg& L = J.leg[0];
      const int x = L.idx ? L.idx[r] : (r >> L.shift) & L.mask;
      w = L.u + (int64_t)x * L.stride;
    }
    f64x4 acc[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
    if (J.m <= 1) tree_tile<NT, 1>(J, P, u, w, r, k0, k1, acc);
    else if (J.m == 2) tree_tile<NT, 2>(J, P, u, w, r, k0, k1, acc);
    else tree_tile<NT, 3>(J, P, u, w, r, k0, k1, acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int orow = rows[t * 16 + lk + 4 * e];
      if (orow >= 0) {
#pragma unroll
        for (int c = 0; c < NT; ++c)  // (the padding stays zero also for infinite values)
          out[(int64_t)orow * J.npad + 16 * c + li] = c0 + 16 * c + li < J.n ? acc[c][e] : 0.0;
      }
    }
  }
}

__global__ void __launch_bounds__(256) tree_vertex_kernel(TreeJobs js) {
  __shared__ int rows[TREE_ROWS + 32];
  __shared__ int cnt[2];
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
  const int row = rb * TREE_ROWS + tid;
  const bool on = tid < TREE_ROWS && row < J.R;
  int d = 0;
  if (on && J.dmode == 1) d = (row >> J.dshift) & 1;
  if (on && J.dmode == 2)
    d = (int)((tree_digit_word(J.xs[(int64_t)row * J.nc + J.coord], J.ndig) >> J.dshift) & 1);
  const uint64_t b0 = __ballot(on && d == 0), b1 = __ballot(on && d == 1);
  if (tid == 0) {
    cnt[0] = __popcll(b0);
    cnt[1] = __popcll(b1);
  }
  __syncthreads();
  const int f0 = cnt[0], f1 = cnt[1];  // digit counts of the first wavefront
  __syncthreads();
  if (tid == 64) {
    cnt[0] = f0 + __popcll(b0);
    cnt[1] = f1 + __popcll(b1);
  }
  __syncthreads();
  const int n0 = cnt[0], n1 = cnt[1];
  if (on) {
    const uint64_t below = (uint64_t(1) << (tid & 63)) - 1;
    const int pos = __popcll((d ? b1 : b0) & below) + (tid >= 64 ? (d ? f1 : f0) : 0);
    rows[d ? ((n0 + 15) & ~15) + pos : pos] = row;
  }
  __syncthreads();
  const int k0 = kc * J.kper, k1 = min(J.nk, k0 + J.kper);
  if (J.nt == 1) tree_rows<1>(J, rows, n0, n1, ng, kc, k0, k1);
  else if (J.nt == 2) tree_rows<2>(J, rows, n0, n1, ng, kc, k0, k1);
  else if (J.nt == 3) tree_rows<3>(J, rows, n0, n1, ng, kc, k0, k1);
  else tree_rows<4>(J, rows, n0, n1, ng, kc, k0, k1);
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
  for (int i = 0; i < a.n; ++i) {
    const TreeIndex& t = a.t[i];
    int r = 0, last = -1;
    uint64_t w = 0;
    for (int b = 0; b < t.nbits; ++b) {
      const int c = t.coord[b];
      if (c != last) {
        w = tree_digit_word(x[c], ndigits[c]);
        last = c;
      }
      r = 2 * r + (int)((w >> t.shift[b]) & 1);
    }
    t.out[p] = r;
  }
}

// f = <u_a, u_b> over the centre edge, 16 lanes per point (b null: u_a's only
// entry).  A point with a negative or NaN coordinate gives NaN and the flag.
__global__ void __launch_bounds__(256)
tree_dot_kernel(TreeLeg a, TreeLeg b, const double* __restrict__ xs, int64_t npts, int nc, double* __restrict__ out,
                int* __restrict__ flag) {
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

// P[d][kb][n][kk] = T at output index n, input combination k = 16 kb + kk
// (the last leg padded to lpad entries), digit d; zero in the padding.
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
    const int kk = (int)(e & 15);
    int64_t r = e >> 4;
    const int n = (int)(r % J.npad);
    r /= J.npad;
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
  int64_t pack = 0;          // offset in the packed copy
  bool table = false;
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
  double* d_tab = nullptr;   // vectors of every table vertex
  int64_t tab_cap = 0;
  int tab_digits = -1;       // largest table's digits in the buffer (-1: none built)
  ~TreeState() {
    if (d_pack) (void)hipFree(d_pack);
    if (d_tab) (void)hipFree(d_tab);
  }
};

void tree_state_free(TreeState* s) { delete s; }
void tree_state_stale(TreeState* s) {
  if (s) {
    s->packed = false;
    s->tab_digits = -1;
  }
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
  if (!net->tree) net->tree = new TreeState;
  TreeState& S = *net->tree;
  if (S.packed) return QTT_OK;
  const HostTopo& t = net->t;
  S.tab_digits = -1;
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
    }
    for (size_t i = 0; i < p.in.size(); i++) {
      const int w = p.in[i];
      p.nd += S.vp[w].nd;
      p.level = std::max(p.level, S.vp[w].level + 1);
      const int64_t dim = edge_dim(net, v, w);
      if (i + 1 < p.in.size()) q *= dim;
      else p.kbl = (int)((dim + 15) / 16);
    }
    if (q * p.kbl >= (int64_t(1) << 27)) return qtt_fail(ctx, QTT_EINVAL, "evaluate: a core is too large");
    p.nk = (int)(q * p.kbl);
    p.slices = t.vcoord[v] >= 0 ? 2 : 1;
    p.pack = tot;
    tot += (int64_t)p.slices * p.nk * p.npad * 16;
  }
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
      tree_vertex_kernel<<<units, 256, 0, ctx->stream>>>(js);
      int rc = qtt_hip_check(ctx, hipGetLastError(), "tree_vertex_kernel");
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
  // chunks of a vertex's k blocks: more workgroups when its rows and columns
  // alone leave compute units idle, each with at least 8 blocks of 16
  static int chunks(const qtt_ctx* ctx, const VPlan& p, int64_t R) {
    const int64_t u = ((R + TREE_ROWS - 1) / TREE_ROWS) * p.ngrp;
    const int64_t want = (2 * (int64_t)ctx->cus) / std::max<int64_t>(1, u);
    return (int)std::max<int64_t>(1, std::min<int64_t>(want, p.nk / 8));
  }
  int add(const VPlan& p, TreeJob& J) {
    const int64_t R = J.R;
    J.kc = chunks(ctx, p, R);
    J.kper = (p.nk + J.kc - 1) / J.kc;
    J.kc = (p.nk + J.kper - 1) / J.kper;
    const int64_t n = R * p.npad;
    if (js.n == TREE_JOBS || (J.kc > 1 && part_used + n * J.kc > part_cap)) {
      const int rc = flush();
      if (rc) return rc;
    }
    if (J.kc > 1) {
      sums.push_back({part + part_used, J.kc, n, J.out});
      J.out = part + part_used;
      part_used += n * J.kc;
    }
    js.unit0[js.n] = units;
    units += (int)((R + TREE_ROWS - 1) / TREE_ROWS) * p.ngrp * J.kc;
    js.job[js.n++] = J;
    return QTT_OK;
  }
};

// the digits behind v's output leg in the order of its table index, top first
void table_digits(const qtt_net* net, const TreeState& S, int v, std::vector<int>& out) {
  if (net->t.vcoord[v] >= 0) out.push_back(v);
  for (int w : S.vp[v].in) table_digits(net, S, w, out);
}

}  // namespace

int launch_eval_tree(qtt_ctx* ctx, qtt_net* net, const double* xs, int64_t npts, double* out) {
  const HostTopo& t = net->t;
  int rc = tree_pack(ctx, net);
  if (rc) return rc;
  TreeState& S = *net->tree;
  const int nc = t.ncoord;
  // Tables: a vertex with nd digits behind it is a table when 2^nd <= npts / 2
  // (its rows then cost at most half of a row per point, also on a call that
  // builds them), nd <= 16 and the table holds at most 2^21 doubles.
  int limit = 0;
  while (limit < TREE_BITS && (int64_t(4) << limit) <= npts) ++limit;
  int64_t tabs = 0;
  int digits = 0;  // of the largest table: names the set of tables
  bool any_point = false;
  for (int v : S.order) {
    VPlan& p = S.vp[v];
    p.table = p.nd <= limit && (int64_t(p.npad) << p.nd) <= (int64_t(1) << 21);
    for (int w : p.in) p.table = p.table && S.vp[w].table;
    if (p.table) {
      p.buf = tabs;
      tabs += int64_t(p.npad) << p.nd;
      digits = std::max(digits, p.nd);
    } else {
      any_point = true;
    }
  }
  if (S.tab_cap < tabs) {
    if (S.d_tab) (void)hipFree(S.d_tab);
    S.d_tab = nullptr;
    S.tab_cap = 0;
    S.tab_digits = -1;
    rc = qtt_hip_check(ctx, hipMalloc(&S.d_tab, tabs * sizeof(double)), "hipMalloc tree tables");
    if (rc) return rc;
    S.tab_cap = tabs;
  }
  // point rows: buffers of every point vertex for a chunk of points (at most
  // about 512 MiB), the table entries of every point, partial sums
  int64_t per = 0, kpart = 0;
  std::vector<int> frontier;  // tables used by a point vertex or the final product
  std::vector<int> front_of(t.nv, -1);
  int most_level = 0;
  for (int v : S.order) {
    VPlan& p = S.vp[v];
    most_level = std::max(most_level, p.level);
    const bool final_leg = p.to < 0 || v == S.centre || t.parent[S.centre] == v;
    if (p.table && (final_leg || !S.vp[p.to].table)) {
      front_of[v] = (int)frontier.size();
      frontier.push_back(v);
    }
    if (!p.table) {
      p.buf = per;
      per += p.npad;
    }
  }
  int64_t chunk = npts;
  if (per > 0) chunk = std::max<int64_t>(TREE_ROWS, std::min<int64_t>(npts, ((int64_t(1) << 26) / per) & ~int64_t(TREE_ROWS - 1)));
  chunk = std::min<int64_t>(chunk, int64_t(1) << 24);
  // (Level::chunks: rows x chunks is at most 2 cus TREE_ROWS per column group)
  for (int v : S.order)
    if (S.vp[v].nk >= 16) kpart = std::max<int64_t>(kpart, 2 * (int64_t)ctx->cus * TREE_ROWS * 16 * S.vp[v].nt);
  kpart = std::max<int64_t>(kpart * 2, 16);
  const int64_t nidx = (int64_t)frontier.size() * chunk;
  double* scr = qtt_scratch(ctx, (size_t)(per * chunk + kpart) * sizeof(double) + (size_t)nidx * sizeof(int) + 256);
  if (!scr) return qtt_fail(ctx, QTT_ENOMEM, "evaluate: scratch");
  double* pbuf = scr;
  double* part = pbuf + per * chunk;
  int* idx = (int*)(part + kpart);
  const int* d_ndigits = net->view().ndigits;

  auto make_job = [&](int v, int64_t R, int64_t nrows, const double* x0) {
    const VPlan& p = S.vp[v];
    TreeJob J;
    std::memset(&J, 0, sizeof(J));
    J.P = S.d_pack + p.pack;
    J.dstride = (int64_t)p.nk * p.npad * 16;
    J.R = (int)R;
    J.n = p.n;
    J.npad = p.npad;
    J.nt = p.nt;
    J.ngrp = p.ngrp;
    J.m = (int)p.in.size();
    J.kbl = p.kbl;
    J.nk = p.nk;
    const int c = t.vcoord[v];
    J.out = p.table ? S.d_tab + p.buf : pbuf + p.buf * nrows;
    if (c >= 0) {
      J.dmode = p.table ? 1 : 2;
      J.dshift = p.table ? p.nd - 1 : t.ndigits[c] - t.vdigit[v];
      J.coord = c;
      J.nc = nc;
      J.ndig = t.ndigits[c];
      J.xs = x0;
    }
    int sh = p.nd - (c >= 0);
    for (int j = 0; j < J.m; j++) {
      const int w = p.in[j];
      const VPlan& pw = S.vp[w];
      TreeLeg& L = J.leg[j];
      L.dim = pw.n;
      L.stride = pw.npad;
      if (p.table) {
        sh -= pw.nd;
        L.u = S.d_tab + pw.buf;
        L.shift = sh;
        L.mask = (1 << pw.nd) - 1;
      } else if (pw.table) {
        L.u = S.d_tab + pw.buf;
        L.idx = idx + front_of[w] * chunk;
      } else {
        L.u = pbuf + pw.buf * nrows;
        L.mask = -1;
      }
    }
    return J;
  };
  auto run_level = [&](bool table, int64_t nrows, const double* x0) -> int {
    Level lv(ctx, part, kpart);
    for (int l = 0; l <= most_level; l++) {
      for (int v : S.order) {
        const VPlan& p = S.vp[v];
        if (p.level != l || p.table != table) continue;
        TreeJob J = make_job(v, table ? int64_t(1) << p.nd : nrows, nrows, x0);
        const int r = lv.add(p, J);
        if (r) return r;
      }
      const int r = lv.flush();
      if (r) return r;
    }
    return QTT_OK;
  };
  if (S.tab_digits != digits && tabs > 0) {
    if ((rc = run_level(true, chunk, xs))) return rc;
    S.tab_digits = digits;
  }
  for (int64_t p0 = 0; p0 < npts; p0 += chunk) {
    const int64_t np = std::min(chunk, npts - p0);
    const double* x0 = xs + p0 * nc;
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
      tree_index_kernel<<<(unsigned)((np + 255) / 256), 256, 0, ctx->stream>>>(a, x0, np, nc, d_ndigits);
      if ((rc = qtt_hip_check(ctx, hipGetLastError(), "tree_index_kernel"))) return rc;
    }
    if (any_point && (rc = run_level(false, np, x0))) return rc;
    auto leg_of = [&](int v) {
      const VPlan& p = S.vp[v];
      TreeLeg L;
      L.dim = p.n;
      L.stride = p.npad;
      L.shift = 0;
      L.mask = -1;
      L.idx = p.table ? idx + front_of[v] * chunk : nullptr;
      L.u = p.table ? S.d_tab + p.buf : pbuf + p.buf * np;
      return L;
    };
    TreeLeg a = leg_of(S.centre < 0 ? 0 : S.centre), b;
    std::memset(&b, 0, sizeof(b));
    if (S.centre >= 0) b = leg_of(t.parent[S.centre]);
    tree_dot_kernel<<<(unsigned)((np + 15) / 16), 256, 0, ctx->stream>>>(a, b, x0, np, nc, out + p0, ctx->flags());
    if ((rc = qtt_hip_check(ctx, hipGetLastError(), "tree_dot_kernel"))) return rc;
  }
  // queued only: work on another stream that takes the scratch (or this
  // network's tables, through this function) waits for it
  return qtt_scratch_queued(ctx);
}
