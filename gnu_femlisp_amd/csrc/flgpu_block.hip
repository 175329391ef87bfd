// Vertex-centred block smoothers: <geometric-ssc> and <geometric-psc>
// (src/iteration/blockit.lisp:41-203, src/iteration/geoblock.lisp:37-157).
//
// femlisp's vertex-centred block of a mesh vertex v holds v and every DOF of a cell containing
// v that is not Dirichlet (find-vertex-centered-block, geoblock.lisp:65-91).  On the lattice of
// a Q`order` discretisation (M = order n + 1 points per axis) v sits at order a, a in
// [0, n]^dim, and its block is the points v + d with |d_k| <= order - 1: W = (2 order - 1)^dim
// slots, slot s = the digits of s in base 2 order - 1, axis 0 most significant.  A slot is
// absent when its point lies outside the lattice or is Dirichlet (v itself always counts).
//
// Blocks are swept colour by colour, colour = the parity of a per axis (axis 0 most
// significant).  The vertices of two blocks of one colour are at least 2 order lattice steps
// apart along some axis.  The rows of a block couple only DOFs of the cells around its vertex,
// within order steps of it, while the other block's DOFs are at least order + 1 steps away:
// neither block reads what the other writes, and the sequential sweep over one colour equals
// its parallel update.
//
// The blocks are symmetric positive definite (principal submatrices of the SPD operator, the
// Dirichlet vertex an identity row), so their inverses are formed once by Gauss-Jordan without
// pivoting in FP64 and stored (femlisp's store-p t, blockit.lisp:118-121), per vertex in
// lattice vertex order as inv[v][i][j] = (A_BB^-1)_ij, rows padded to 16 bytes, identity rows and
// columns at absent slots.  One iterate then costs per block the residual of its rows (<ssc>
// only; from the element matrices of the cells around the vertex where the matrix has them,
// else from its CSR rows) and the W x W inverse; order-1 blocks are single DOFs and take one
// lane each.
#include "flgpu_internal.h"

namespace flgpu {

namespace {


struct BlkGeom {
  int dim, order, n, M, W, w1, h;
  int par[3];  // colour parity per axis
  int cnt[3];  // vertices of that parity per axis
  Div1 dcnt[3];
};

BlkGeom blk_geom(const flgpu_mat *A, int colour) {
  BlkGeom g{};
  g.dim = A->lat_dim;
  g.order = A->lat_order;
  g.n = A->lat_n;
  g.M = g.order * g.n + 1;
  g.w1 = 2 * g.order - 1;
  g.h = g.order - 1;
  g.W = 1;
  for (int k = 0; k < g.dim; k++) g.W *= g.w1;
  for (int k = 0; k < 3; k++) {
    g.par[k] = 0;
    g.cnt[k] = 1;
  }
  for (int k = 0; k < g.dim; k++) {
    g.par[k] = (colour >> (g.dim - 1 - k)) & 1;
    g.cnt[k] = (g.n + 2 - g.par[k]) / 2;
  }
  for (int k = 0; k < 3; k++) g.dcnt[k] = div1(g.cnt[k]);
  return g;
}

long blk_count(const BlkGeom &g) {
  long c = 1;
  for (int k = 0; k < g.dim; k++) c *= g.cnt[k];
  return c;
}

// vertex coordinates a of the w-th vertex of the colour (last axis fastest)
__device__ __forceinline__ void blk_vertex(const BlkGeom &g, long w, int *a) {
  for (int k = g.dim - 1; k >= 0; k--) {
    int j = (int)(w % g.cnt[k]);
    w /= g.cnt[k];
    a[k] = 2 * j + g.par[k];
  }
}

__device__ __forceinline__ long blk_vertex_id(const BlkGeom &g, const int *a) {
  long v = 0;
  for (int k = 0; k < g.dim; k++) v = v * (g.n + 1) + a[k];
  return v;
}

// the DOF of the slot with digits dg (axis k's offset dg[k] - h) of vertex a, or -1
__device__ __forceinline__ int blk_key_d(const BlkGeom &g, const int *a, const int *dg) {
  int key = 0;
  bool centre = true, bdry = false;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if (k >= g.dim) break;
    int c = g.order * a[k] + dg[k] - g.h;
    if (c < 0 || c >= g.M) return -1;
    if (dg[k] != g.h) centre = false;
    if (c == 0 || c == g.M - 1) bdry = true;
    key = key * g.M + c;
  }
  return (bdry && !centre) ? -1 : key;
}

// the DOF of slot s of vertex a, or -1
__device__ __forceinline__ int blk_key(const BlkGeom &g, const int *a, int s) {
  int dg[3] = {0, 0, 0};
  for (int k = g.dim - 1; k >= 0; k--) {
    dg[k] = s % g.w1;
    s /= g.w1;
  }
  return blk_key_d(g, a, dg);
}

// entries of a stored row of a block's inverse: W padded to 16 bytes
template <class T>
__host__ __device__ constexpr int blk_pad(int W) {
  const int v = 16 / (int)sizeof(T);
  return (W + v - 1) / v * v;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Block inverses of order 2, one wave per vertex (grid: all (n+1)^dim vertices, colour 0's
// geometry with the parities ignored).  The block matrix is gathered into LDS from the CSR rows
// of the block's DOFs (a column belongs to the block when its offset from v is within the block),
// four rows' entries in flight at a time.  Then lane j holds column j and a Gauss-Jordan step k is
// in registers: the pivot and column k's entries come from lane k, and column k itself becomes
// the inverse's.  Bound by the instructions of the W^3 steps.  24^3 cells (15 625 blocks of 27)
// FP64 186 us, 837 with [A|I] and the steps in LDS.
template <class T, int DIM>
__global__ __launch_bounds__(64) void k_blk_invert(BlkGeom g, Div1 dM,
                                                   const int *__restrict__ rowptr,
                                                   const int *__restrict__ colidx,
                                                   const T *__restrict__ vals, T *__restrict__ inv) {
  constexpr int W = DIM == 3 ? 27 : DIM == 2 ? 9 : 3, WP = blk_pad<T>(W);
  __shared__ double a[W][W + 1];
  __shared__ int sb[W], se[W];
  const int lane = threadIdx.x;
  const long v = blockIdx.x;
  int av[3] = {0, 0, 0}, c0[DIM];
  {
    unsigned t = (unsigned)v;
#pragma unroll
    for (int k = DIM - 1; k >= 0; k--) {
      av[k] = (int)(t % (unsigned)(g.n + 1));
      t /= (unsigned)(g.n + 1);
      c0[k] = 2 * av[k] - 1;
    }
  }
  for (int e = lane; e < W * W; e += 64) a[e / W][e % W] = 0.0;
  __syncthreads();
  if (lane < W) {
    const int ks = blk_key(g, av, lane);
    sb[lane] = ks < 0 ? 0 : rowptr[ks];
    se[lane] = ks < 0 ? 0 : rowptr[ks + 1];
    if (ks < 0) a[lane][lane] = 1.0;  // absent slot: identity row
  }
  __syncthreads();
  constexpr int RB = W % 3 == 0 ? 3 : 1, CH = 2;  // rows and chunks of 64 entries in flight
#pragma unroll 1
  for (int s0 = 0; s0 < W; s0 += RB) {
    int b[RB], n[RB], most = 0;
#pragma unroll
    for (int u = 0; u < RB; u++) {
      b[u] = sb[s0 + u];
      n[u] = se[s0 + u] - b[u];
      most = max(most, n[u]);
    }
    for (int o = lane; o < most + lane; o += 64 * CH) {
      int cl[RB][CH];
      T vl[RB][CH];
#pragma unroll
      for (int u = 0; u < RB; u++)
#pragma unroll
        for (int c = 0; c < CH; c++) {
          const int e = b[u] + max(min(o + c * 64, n[u] - 1), 0);
          cl[u][c] = n[u] > 0 ? colidx[e] : 0;
          vl[u][c] = n[u] > 0 ? vals[e] : (T)0;
        }
#pragma unroll
      for (int u = 0; u < RB; u++)
#pragma unroll
        for (int c = 0; c < CH; c++) {
          unsigned col = (unsigned)cl[u][c];
          int t = 0;
          bool in = o + c * 64 < n[u], centre = true, bdry = false;
#pragma unroll
          for (int k = DIM - 1, mul = 1; k >= 0; k--, mul *= 3) {
            const unsigned cq = k > 0 ? fdiv(col, dM) : 0u;
            const int ck = (int)(col - cq * (unsigned)g.M), d = ck - c0[k];
            col = cq;
            in &= d >= 0 && d < 3;
            centre &= d == 1;
            bdry |= ck == 0 || ck == g.M - 1;
            t += d * mul;
          }
          if (in && (centre || !bdry)) a[s0 + u][t] = (double)vl[u][c];
        }
    }
  }
  __syncthreads();
  double c[W];
#pragma unroll
  for (int i = 0; i < W; i++) c[i] = a[i][min(lane, W - 1)];
#pragma unroll
  for (int k = 0; k < W; k++) {
    const bool own = lane == k;
    const double p = lane_value(c[k], k);
    const double pr = (own ? 1.0 : c[k]) / p;
#pragma unroll
    for (int i = 0; i < W; i++)
      if (i != k) {
        const double f = lane_value(c[i], k);
        c[i] = (own ? 0.0 : c[i]) - f * pr;
      }
    c[k] = pr;
  }
  T *out = inv + v * W * WP;
  if (lane < WP)
#pragma unroll
    for (int i = 0; i < W; i++) out[i * WP + lane] = lane < W ? (T)c[i] : (T)0;
}

// The LDS traffic of one wave is in order; this keeps the compiler from moving accesses across.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A block's inverse in the registers of the G lanes that share the block, as 16-byte pieces of
// its padded rows (piece f = k G + gl), and y = A_BB^-1 r from it: every lane multiplies its
// pieces with the matching entries of r from LDS, and a slot's lane sums the pieces of its row
// in order.  All of a block's 16-byte loads are independent and coalesced (27 loads of 4 bytes
// by 27 of 64 lanes, and 27 broadcasts, as one column per step).
template <class T, int W, int G>
struct BlkInverse {
  static constexpr int VL = 16 / (int)sizeof(T), WP = (W + VL - 1) / VL * VL, CPR = WP / VL,
                       NC = W * CPR, K = (NC + G - 1) / G;
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  vec a[K];
  __device__ __forceinline__ void load(const T *__restrict__ iv, int gl) {
#pragma unroll
    for (int k = 0; k < K; k++) a[k] = *(const vec *)(iv + (long)min(k * G + gl, NC - 1) * VL);
  }
  // rv: r in LDS, WP values (zero beyond W); part: NC values of LDS
  __device__ __forceinline__ void multiply(const T *rv, T *part, int gl) const {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int f = k * G + gl;
      const vec r = *(const vec *)(rv + (f % CPR) * VL);
      T p = 0;
#pragma unroll
      for (int j = 0; j < VL; j++) p += a[k][j] * r[j];
      if (f < NC) part[f] = p;
    }
  }
  static __device__ __forceinline__ T row(const T *part, int slot) {
    T y = 0;
#pragma unroll
    for (int j = 0; j < CPR; j++) y += part[slot * CPR + j];
    return y;
  }
};

constexpr int kBlkWaves = 2;  // waves per workgroup of k_blk_sweep

// Order-2 blocks in DIM dimensions: W = 3^DIM slots, slot digits base 3, last axis fastest.
// Slots 3q, 3q + 1, 3q + 2 are three lattice neighbours along the last axis: their CSR rows
// are contiguous, a run of at most 11 * 3^(DIM-1-z) * 5^z entries, z = the number of the first
// DIM - 1 digits of q that sit on the vertex's planes.
constexpr int pow_i(int b, int e) { return e == 0 ? 1 : b * pow_i(b, e - 1); }
template <int DIM>
constexpr int run_chunks(int q) {  // 64-entry chunks of run q
  int z = 0;
  for (int k = 0; k < DIM - 1; k++, q /= 3) z += (q % 3) == 1;
  return (11 * pow_i(3, DIM - 1 - z) * pow_i(5, z) + 63) / 64;
}
template <int DIM>
constexpr int range_chunks(int q0, int q1) {
  int c = 0;
  for (int q = q0; q < q1; q++) c += run_chunks<DIM>(q);
  return c;
}

// runs [Q0, Q1) of a block: every chunk's entries loaded, then the x values they name, then
// the products added into the slots' partial sums
template <class T, int DIM, int Q0, int Q1>
__device__ __forceinline__ void blk_runs(const int *__restrict__ colidx,
                                         const T *__restrict__ vals, const T *x, int lane,
                                         const int *ta, const int *e0, const int *e1,
                                         const int *e2, const int *e3, T *acc) {
  constexpr int NCH = range_chunks<DIM>(Q0, Q1);
  int cc[NCH];
  T vv[NCH];
#pragma unroll
  for (int q = Q0, c = 0; q < Q1; q++)
#pragma unroll
    for (int i = 0; i < run_chunks<DIM>(q); i++, c++) {
      int e = e0[q] + 64 * i + lane;
      int ec = max(min(e, e3[q] - 1), 0);
      cc[c] = colidx[ec];
      vv[c] = vals[ec];
    }
  T xv[NCH];
#pragma unroll
  for (int c = 0; c < NCH; c++) xv[c] = x[cc[c]];
#pragma unroll
  for (int q = Q0, c = 0; q < Q1; q++)
#pragma unroll
    for (int i = 0; i < run_chunks<DIM>(q); i++, c++) {
      int e = e0[q] + 64 * i + lane;
      T p = e < e3[q] ? vv[c] * xv[c] : (T)0;
      int t = ta[q] + (e >= e1[q]) + (e >= e2[q]);
      acc[3 * q] += t == 0 ? p : (T)0;
      acc[3 * q + 1] += t == 1 ? p : (T)0;
      acc[3 * q + 2] += t == 2 ? p : (T)0;
    }
}

// One colour of an iterate with order-2 blocks, one wave per block.
// <ssc>: r_k = b_k - (A x)_k for the block's DOFs k (stored in r, as femlisp stores the block
// residual), then x_B += omega A_BB^-1 r_B.  <psc>: x_B += omega A_BB^-1 r_B with r as given.
// b may be r.  The memory reads of a block are issued in batches of independent loads: the
// row bounds; the CSR entries of the runs, 64 at a time and every lane its own entry; the x
// values they name; then the block inverse, while the partial sums are reduced.  Every lane adds
// its products into per-slot partial sums, and the 64 partials of each slot are summed in lane
// order through LDS by the slot's own lane.
template <class T, bool SSC, int DIM>
__global__ __launch_bounds__(64 * kBlkWaves) void k_blk_sweep(BlkGeom g, long cnt,
                                                              const int *__restrict__ rowptr,
                                                              const int *__restrict__ colidx,
                                                              const T *__restrict__ vals,
                                                              const T *__restrict__ inv, T omega,
                                                              T *x, const T *b, T *r) {
  constexpr int W = pow_i(3, DIM), NRUN = W / 3;
  typedef BlkInverse<T, W, 64> Inv;
  // the partial sums, then r (32 values) and the inverse's products.  <psc> has no partial sums:
  // with room for them only ten waves a CU were resident, and at Q2 32^3 FP64 an iterate took 73
  // us instead of 60
  constexpr int kPart = SSC ? 64 * (W + 1) : 32 + (Inv::NC + Inv::VL - 1) / Inv::VL * Inv::VL;
  static_assert(kPart >= 32 + Inv::NC && Inv::WP <= 32, "r and the products fit");
  __shared__ __align__(16) T part[kBlkWaves][kPart];
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int wv = threadIdx.x >> 6;
  long w = (long)lb * kBlkWaves + wv;
  if (w >= cnt) return;  // uniform over the wave
  const int lane = threadIdx.x & 63;
  int av[3];
  blk_vertex(g, w, av);
  int key = lane < W ? blk_key(g, av, lane) : -1;
  const T *iv = inv + blk_vertex_id(g, av) * W * Inv::WP;
  Inv A;
  typename Inv::vec row[Inv::CPR];  // 1D: the slot's row, a lane's own; else the block's pieces
  auto load_inverse = [&] {
    if constexpr (DIM == 1) {
#pragma unroll
      for (int k = 0; k < Inv::CPR; k++)
        row[k] = ((const typename Inv::vec *)iv)[min(lane, W - 1) * Inv::CPR + k];
    } else {
      A.load(iv, lane);
    }
  };
  T myr = 0;
  if (SSC) {
    int rs = 0, re = 0;
    if (key >= 0) {
      rs = rowptr[key];
      re = rowptr[key + 1];
    }
    // per run: first present slot, and the entry bounds [e0, e3) with the ends e1, e2 of its
    // first two rows (present rows are consecutive lattice points; none present: empty run)
    int ta[NRUN], e0[NRUN], e1[NRUN], e2[NRUN], e3[NRUN];
#pragma unroll
    for (int q = 0; q < NRUN; q++) {
      int k0 = __builtin_amdgcn_readlane(key, 3 * q);
      int k1 = __builtin_amdgcn_readlane(key, 3 * q + 1);
      int k2 = __builtin_amdgcn_readlane(key, 3 * q + 2);
      int a = k0 >= 0 ? 0 : (k1 >= 0 ? 1 : (k2 >= 0 ? 2 : -1));
      int z = k2 >= 0 ? 2 : (k1 >= 0 ? 1 : 0);
      ta[q] = a < 0 ? 0 : a;
      e0[q] = a < 0 ? 0 : __builtin_amdgcn_readlane(rs, 3 * q + a);
      e3[q] = a < 0 ? 0 : __builtin_amdgcn_readlane(re, 3 * q + z);
      e1[q] = (a >= 0 && a < z) ? __builtin_amdgcn_readlane(re, 3 * q + a) : e3[q];
      e2[q] = (a >= 0 && a + 1 < z) ? __builtin_amdgcn_readlane(re, 3 * q + a + 1) : e3[q];
    }
    T acc[W];
#pragma unroll
    for (int s = 0; s < W; s++) acc[s] = 0;
    blk_runs<T, DIM, 0, NRUN>(colidx, vals, x, lane, ta, e0, e1, e2, e3, acc);
#pragma unroll
    for (int s = 0; s < W; s++) part[wv][lane * (W + 1) + s] = acc[s];
    load_inverse();  // in flight during the reduction, in the registers acc held
    wave_sync();
    if (key >= 0) {
      T sum = 0;
      for (int l = 0; l < 64; l++) sum += part[wv][l * (W + 1) + lane];
      myr = b[key] - sum;
    }
  } else {
    load_inverse();
    if (key >= 0) myr = r[key];
  }
  T y = 0;
  if constexpr (DIM == 1) {
    // three products a slot, without the LDS round trips (200 000 cells FP64: 103 us, 110 with)
#pragma unroll
    for (int j = 0; j < W; j++) y += row[j / Inv::VL][j % Inv::VL] * lane_value(myr, j);
  } else {
    wave_sync();  // part is free for r and the products
    T *rv = part[wv], *pr = part[wv] + 32;
    if (lane < Inv::WP) rv[lane] = myr;
    wave_sync();
    A.multiply(rv, pr, lane);
    wave_sync();
    if (lane < W) y = Inv::row(pr, lane);
  }
  if (key >= 0) {
    if (SSC) r[key] = myr;
    x[key] += omega * y;
  }
}

// One colour of an iterate with order-2 blocks from the element matrices of the cells around
// each vertex: (A x)_i over the block's rows i is the sum, over the 2^DIM cells, of the cell's
// element row times the cell's 3^DIM values of x, so the columns and row bounds of the CSR, which
// cost two more dependent round trips to memory, are not read.  rows: with ALPHA one reference
// matrix, scaled by the cell's factor alpha[cell] (a coefficient constant per cell), else
// every cell's own matrix (`elem`).
//
// G = 4^DIM lanes share a block: lane = (cell s around the vertex, node t of that cell within
// the block), bits per axis, axis 0 most significant.  A lane multiplies its element row
// (registers) with the cell's part of the x patch (LDS, 5^DIM values around the vertex, zero at
// Dirichlet points as the eliminated columns are); a node shared by several cells is summed by
// exchanges across the cell bits, both partners forming the same sum.  The rows, the patch, b,
// the old x and the block's inverse are all loaded at once, one round trip.
//
// Issue, not bytes, bounds the 3D sweep, so everything that depends on the lane alone (offsets
// from the vertex, the reference row) is formed once per wave; a vertex costs its coordinates
// (uniform in 3D) and one bit test per axis for what the boundary cuts off.  A wave takes `per`
// consecutive vertices and loads the next one's values before it works on the current one.
// Q2 48^3, one fine colour (14 700 blocks): FP32 16.2 us (17.5 us with the indices formed anew
// for every block); 51 us from the CSR rows, 10.6 KB of entries per block where this reads 32
// bytes of alpha.
template <class T, bool SSC, int DIM, bool ALPHA>
struct BlkCell {
  static constexpr int W = pow_i(3, DIM), G = pow_i(4, DIM), NP = pow_i(5, DIM);
  typedef BlkInverse<T, W, G> Inv;
  typedef typename Inv::vec vec;
  // what depends on the lane alone
  int gl, dk, po[2], pp[2][3], ps[3], sb[3], dc, erow, pbase, slot;
  bool canon, centre;
  vec e[Inv::CPR];  // element row
  // what a vertex's loads give
  struct Vals {
    int key;
    bool present, exists, vb;
    T xo, bo, al, pv[2];
    Inv A;
    vec e[ALPHA ? 1 : Inv::CPR];
  };

  __device__ __forceinline__ void init(const BlkGeom &g, int gl_, const T *__restrict__ rows) {
    gl = gl_;
    dk = dc = erow = pbase = slot = 0;
    canon = centre = true;
#pragma unroll
    for (int k = 0; k < DIM; k++) {
      const int s = (gl >> (DIM + DIM - 1 - k)) & 1, t = (gl >> (DIM - 1 - k)) & 1;
      const int d = s ? t : -t;
      sb[k] = s;
      ps[k] = d + 2;
      dk = dk * g.M + d;
      dc = dc * g.n + s - 1;
      erow = erow * 3 + (s ? t : 2 - t);
      pbase = pbase * 5 + 2 * s;
      slot = slot * 3 + d + 1;
      canon = canon && (s || t);
      centre = centre && d == 0;
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int q = gl + u * G;
      po[u] = 0;
#pragma unroll
      for (int k = 0; k < DIM; k++) {
        pp[u][k] = q < NP ? (q / pow_i(5, DIM - 1 - k)) % 5 : 5;  // 5: no such value
        po[u] = po[u] * g.M + pp[u][k] - 2;
      }
    }
    if (SSC && ALPHA)
#pragma unroll
      for (int j = 0; j < Inv::CPR; j++)
        e[j] = *(const vec *)(rows + erow * Inv::WP + j * Inv::VL);
  }

  // every load of vertex w of the colour
  __device__ __forceinline__ Vals load(const BlkGeom &g, unsigned w, bool live,
                                       const T *__restrict__ rows, const T *__restrict__ alpha,
                                       const T *__restrict__ inv, const T *x, const T *b,
                                       const T *r) const {
    Vals v;
    int vk = 0, vc = 0, vcl = 0, vid = 0;
    int in = 1, ex = 1;  // the slot's point is interior, the cell exists
    int ip[2] = {1, 1};
    v.vb = false;
    int av[3] = {0, 0, 0};
#pragma unroll
    for (int k = DIM - 1; k >= 0; k--) {
      const unsigned q = k > 0 ? fdiv(w, g.dcnt[k]) : 0u;
      av[k] = 2 * (int)(w - q * (unsigned)g.cnt[k]) + g.par[k];
      w = q;
    }
#pragma unroll
    for (int k = 0; k < DIM; k++) {
      const int a = av[k];
      // bit p: the point 2 a - 2 + p lies inside (0, M - 1); bit s: the cell a - 1 + s exists
      int vm = 0x1f;
      vm = a == 0 ? vm & 0x18 : vm;
      vm = a == 1 ? vm & 0x1e : vm;
      vm = a == g.n ? vm & 0x03 : vm;
      vm = a == g.n - 1 ? vm & 0x0f : vm;
      const int em = (a > 0 ? 1 : 0) | (a < g.n ? 2 : 0);
      in &= vm >> ps[k];
      ex &= em >> sb[k];
      ip[0] &= vm >> pp[0][k];
      ip[1] &= vm >> pp[1][k];
      v.vb = v.vb || a == 0 || a == g.n;
      vk = vk * g.M + 2 * a;
      vc = vc * g.n + a;
      vcl = vcl * g.n + min(a, g.n - 1);
      vid = vid * (g.n + 1) + a;
    }
    v.exists = ex & 1;
    v.present = live && (centre || (in & 1));
    v.key = vk + ((centre || (in & 1)) ? dk : 0);
    v.xo = x[v.key];
    v.bo = SSC ? b[v.key] : r[v.key];
    v.A.load(inv + (long)vid * (W * Inv::WP), gl);
    if (SSC) {
      const int cell = v.exists ? vc + dc : vcl;
      if (ALPHA) {
        v.al = alpha[cell];
      } else {
        const T *rp = rows + (long)cell * (W * Inv::WP) + erow * Inv::WP;
#pragma unroll
        for (int j = 0; j < Inv::CPR; j++) v.e[j] = *(const vec *)(rp + j * Inv::VL);
      }
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const T t = x[vk + ((ip[u] & 1) ? po[u] : 0)];
        v.pv[u] = (ip[u] & 1) ? t : (T)0;
      }
    }
    return v;
  }

  // the update of the vertex whose loads gave v; lds: the block's LDS
  __device__ __forceinline__ void update(const Vals &v, T omega, T *lds, T *x, T *r) const {
    T *px = lds, *rv = px + kPatch, *part = rv + Inv::WP;
    T sum = 0;
    if (SSC) {
      px[gl] = v.pv[0];
      if (gl + G < NP) px[gl + G] = v.pv[1];
      wave_sync();
#pragma unroll
      for (int j = 0; j < W; j++) {
        // node j of the cell, digits base 3: its place in the patch
        int o = 0, q = j, mul = 1;
#pragma unroll
        for (int k = 0; k < DIM; k++) {
          o += (q % 3) * mul;
          q /= 3;
          mul *= 5;
        }
        sum += (ALPHA ? e : v.e)[j / Inv::VL][j % Inv::VL] * px[pbase + o];
      }
      if (ALPHA) sum *= v.al;
      if (!v.exists) sum = 0;
#pragma unroll
      for (int k = 0; k < DIM; k++) {
        const T other = __shfl_xor(sum, 1 << (DIM + DIM - 1 - k), 64);
        if (!((gl >> (DIM - 1 - k)) & 1)) sum += other;
      }
      if (centre && v.vb) sum = v.xo;  // a Dirichlet vertex: identity row
    }
    const T res = v.present ? (SSC ? v.bo - sum : v.bo) : (T)0;
    if (canon) rv[slot] = res;
    if (gl < Inv::WP - W) rv[W + gl] = 0;
    wave_sync();
    v.A.multiply(rv, part, gl);
    wave_sync();
    if (canon && v.present) {
      const T y = Inv::row(part, slot);
      if (SSC) r[v.key] = res;
      x[v.key] = v.xo + omega * y;
    }
    wave_sync();
  }
  static constexpr int kPatch = (NP + Inv::VL - 1) / Inv::VL * Inv::VL;
  static constexpr int kLds = kPatch + Inv::WP + (Inv::NC + Inv::VL - 1) / Inv::VL * Inv::VL;
};

template <class T, bool SSC, int DIM, bool ALPHA>
__global__ __launch_bounds__(256) void k_blk_cell(BlkGeom g, long cnt, int per,
                                                  const T *__restrict__ rows,
                                                  const T *__restrict__ alpha,
                                                  const T *__restrict__ inv, T omega, T *x,
                                                  const T *b, T *r) {
  typedef BlkCell<T, SSC, DIM, ALPHA> B;
  constexpr int NB = 64 / B::G;  // blocks side by side in a wave
  __shared__ __align__(16) T lds[4 * NB][B::kLds];
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // the wave's groups of NB blocks [w0, w1)
  const int groups = (int)((cnt + NB - 1) / NB), w0 = (int)(lb * 4 + wv) * per,
            w1 = min(w0 + per, groups);
  if (w0 >= w1) return;
  const int sub = lane / B::G;
  B blk;
  blk.init(g, lane & (B::G - 1), rows);
  T *my = lds[wv * NB + sub];
  auto load = [&](int w) {
    const int id = w * NB + (NB > 1 ? sub : 0);
    const bool live = NB == 1 || id < (int)cnt;
    return blk.load(g, (unsigned)(live ? id : 0), live, rows, alpha, inv, x, b, r);
  };
  typename B::Vals cur = load(w0);
  for (int w = w0 + 1; w < w1; w++) {
    typename B::Vals next = load(w);
    blk.update(cur, omega, my, x, r);
    cur = next;
  }
  blk.update(cur, omega, my, x, r);
}

// One colour of an iterate with one-DOF blocks (order 1), one lane per block: gesv! of the
// 1 x 1 block is the division by the diagonal.
template <class T, bool SSC>
__global__ __launch_bounds__(256) void k_blk_point(BlkGeom g, long cnt,
                                                   const int *__restrict__ rowptr,
                                                   const int *__restrict__ colidx,
                                                   const T *__restrict__ vals,
                                                   const T *__restrict__ diag, T omega, T *x,
                                                   const T *b, T *r) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  long w = (long)lb * 256 + threadIdx.x;
  if (w >= cnt) return;
  int av[3];
  blk_vertex(g, w, av);
  int key = blk_key(g, av, 0);
  T res;
  if (SSC) {
    T acc = 0;
    for (int e = rowptr[key]; e < rowptr[key + 1]; e++) acc += vals[e] * x[colidx[e]];
    res = b[key] - acc;
    r[key] = res;
  } else {
    res = r[key];
  }
  x[key] += omega * (res / diag[key]);
}

}  // namespace

void blocks_prepare(flgpu_mat *A) {
  FLGPU_REQUIRE(A->lat_dim >= 1 && A->lat_dim <= 3 && A->lat_order >= 1 && A->lat_order <= 2,
                "block smoothers need a matrix assembled on a lattice (dim 1-3, order 1-2)");
  BlkGeom g = blk_geom(A, 0);
  long nv = 1;
  for (int k = 0; k < g.dim; k++) nv *= g.n + 1;
  long N = 1;
  for (int k = 0; k < g.dim; k++) N *= g.M;
  FLGPU_REQUIRE(A->nrows == N && A->ncols == N, "matrix size differs from its lattice");
  if (g.W == 1) return;  // one-DOF blocks use the diagonal
  const int wp = A->prec == FLGPU_F64 ? blk_pad<double>(g.W) : blk_pad<float>(g.W);
  size_t bytes = (size_t)nv * g.W * wp * prec_bytes(A->prec);
  if (!A->blk_inv) {
    A->blk_inv = dev_alloc(bytes);
    layout_changed(A);
  }
  auto invert = [&](auto t) {
    using T = decltype(t);
    auto launch = [&](auto kern) {
      kern<<<(unsigned)nv, 64, 0, A->ctx->stream>>>(g, div1((unsigned)g.M), A->rowptr, A->colidx,
                                                    (const T *)A->vals, (T *)A->blk_inv);
    };
    if (g.dim == 3) launch(k_blk_invert<T, 3>);
    else if (g.dim == 2) launch(k_blk_invert<T, 2>);
    else launch(k_blk_invert<T, 1>);
  };
  if (A->prec == FLGPU_F64) invert(0.0);
  else invert(0.0f);
  FLGPU_HIP(hipGetLastError());
}

void blocks_drop(flgpu_mat *A) {
  if (A->blk_inv) layout_changed(A);
  dev_free(A->blk_inv);
  A->blk_inv = nullptr;
}

template <class T>
static void block_sweep_t(const flgpu_mat *A, bool ssc, T omega, int backwards, T *x, const T *b,
                          T *r, bool cells) {
  int ncol = 1 << A->lat_dim;
  for (int k = 0; k < ncol; k++) {
    BlkGeom g = blk_geom(A, backwards ? ncol - 1 - k : k);
    long cnt = blk_count(g);
    hipStream_t st = A->ctx->stream;
    if (g.W == 1) {
      unsigned grid = xcd_grid(grid_for(cnt, 256));
      if (ssc)
        k_blk_point<T, true><<<grid, 256, 0, st>>>(g, cnt, A->rowptr, A->colidx,
                                                   (const T *)A->vals, (const T *)A->diag, omega,
                                                   x, b, r);
      else
        k_blk_point<T, false><<<grid, 256, 0, st>>>(g, cnt, A->rowptr, A->colidx,
                                                    (const T *)A->vals, (const T *)A->diag,
                                                    omega, x, b, r);
    } else if (cells && (A->cell || A->elem)) {
      // groups of vertices (one per wave at a time), shared out evenly over at most five
      // waves per SIMD, the kernel's occupancy
      const int nb = 64 >> (2 * g.dim);
      const long groups = (cnt + nb - 1) / nb, waves = 20L * A->ctx->cus;
      const int per = (int)((groups + waves - 1) / waves);
      unsigned grid = xcd_grid(grid_for((groups + per - 1) / per, 4));
      auto launch = [&](auto kern, const void *rows) {
        kern<<<grid, 256, 0, st>>>(g, cnt, per, (const T *)rows, (const T *)A->cell,
                                   (const T *)A->blk_inv, omega, x, b, r);
      };
#define FLGPU_BLK(DIM)                                                               \
  if (A->cell)                                                                       \
    launch(ssc ? k_blk_cell<T, true, DIM, true> : k_blk_cell<T, false, DIM, true>,   \
           A->kref);                                                                 \
  else                                                                               \
    launch(ssc ? k_blk_cell<T, true, DIM, false> : k_blk_cell<T, false, DIM, false>, \
           A->elem)
      if (g.dim == 3) FLGPU_BLK(3);
      else if (g.dim == 2) FLGPU_BLK(2);
      else FLGPU_BLK(1);
#undef FLGPU_BLK
    } else {
      unsigned grid = xcd_grid(grid_for(cnt, kBlkWaves));
      auto launch = [&](auto kern) {
        kern<<<grid, 64 * kBlkWaves, 0, st>>>(g, cnt, A->rowptr, A->colidx, (const T *)A->vals,
                                              (const T *)A->blk_inv, omega, x, b, r);
      };
      if (g.dim == 3)
        launch(ssc ? k_blk_sweep<T, true, 3> : k_blk_sweep<T, false, 3>);
      else if (g.dim == 2)
        launch(ssc ? k_blk_sweep<T, true, 2> : k_blk_sweep<T, false, 2>);
      else
        launch(ssc ? k_blk_sweep<T, true, 1> : k_blk_sweep<T, false, 1>);
    }
    FLGPU_HIP(hipGetLastError());
  }
}

void block_sweep(const flgpu_mat *A, bool ssc, double omega, int backwards, void *x,
                 const void *b, void *r, bool cells) {
  BlkGeom g = blk_geom(A, 0);
  if (g.W > 1 && !A->blk_inv) blocks_prepare(const_cast<flgpu_mat *>(A));
  if (A->prec == FLGPU_F64)
    block_sweep_t<double>(A, ssc, omega, backwards, (double *)x, (const double *)b, (double *)r,
                          cells);
  else
    block_sweep_t<float>(A, ssc, (float)omega, backwards, (float *)x, (const float *)b,
                         (float *)r, cells);
}

}  // namespace flgpu

using namespace flgpu;

static void check_block_vec(const flgpu_mat *A, const flgpu_vec *v, const char *what) {
  FLGPU_REQUIRE(v != nullptr, std::string(what) + " must not be NULL");
  FLGPU_REQUIRE(v->ctx == A->ctx, std::string(what) + " belongs to another context");
  FLGPU_REQUIRE(v->n == A->nrows, std::string(what) + ": length mismatch");
  FLGPU_REQUIRE(v->prec == A->prec, std::string(what) + ": precision differs from the matrix");
}

extern "C" int flgpu_block_iterate(const flgpu_mat *A, int kind, double omega, int backwards,
                                   flgpu_vec *x, const flgpu_vec *b, flgpu_vec *r) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    FLGPU_REQUIRE(kind == FLGPU_SMOOTH_SSC || kind == FLGPU_SMOOTH_PSC,
                  "kind must be FLGPU_SMOOTH_SSC or FLGPU_SMOOTH_PSC");
    check_block_vec(A, x, "x");
    check_block_vec(A, b, "b");
    check_block_vec(A, r, "r");
    FLGPU_REQUIRE(x != b && x != r, "x must differ from b and r");
    CTX_LOCK(A->ctx);
    flgpu_mat *M = const_cast<flgpu_mat *>(A);
    if (!M->blk_inv) blocks_prepare(M);
    // a single iterate sums the CSR entries in their order, whatever else A holds, so that a
    // caller's copy of a lattice matrix gives the same values
    block_sweep(A, kind == FLGPU_SMOOTH_SSC, omega, backwards, x->d, b->d, r->d, false);
    return 0;
  });
}
