// Sparse matrices of libflgpu.so: CSR as handed over by femlisp, streamed by
// the kernels in SELL-64 form (one wavefront per 64-row slice, column-major
// entries so that each load instruction of a wavefront reads 64 consecutive
// values and 64 consecutive column indices).
//
// Restates femlisp's <sparse-matrix> operations for scalar (1x1-block) DOFs:
//   gemm-nn!/gemm-tn!      src/matlisp/sparse-matrix.lisp:378-442
//   compute-residual       src/iteration/linit.lisp:73-80
//   <jacobi> iterate       src/iteration/linit.lisp:220-250
//   <sor> iterate          src/iteration/linit.lisp:288-323
// Row sums accumulate like femlisp's template: start from beta*x_i and add
// (alpha*y_j)*A_ij in ascending column order (femlisp's order is hash order).
#include <algorithm>
#include <cstring>
#include <numeric>

#include "flgpu_internal.h"

namespace flgpu {

// ---- SELL construction ----------------------------------------------------------

__global__ void k_slice_width(int nsub, const int *rows, const int *rowptr, int *width) {
  int li = blockIdx.x * blockDim.x + threadIdx.x;
  int len = 0;
  if (li < nsub) {
    int r = rows ? rows[li] : li;
    len = rowptr[r + 1] - rowptr[r];
  }
  for (int off = 32; off > 0; off >>= 1) len = max(len, __shfl_down(len, off, 64));
  if ((threadIdx.x & 63) == 0 && (li - (int)(threadIdx.x & 63)) < nsub)
    width[li >> 6] = len;
}

template <class T>
__global__ void k_sell_fill(int nsub, const int *rows, const int *rowptr, const int *colidx,
                            const T *vals, const long *slice_ptr, int *scol, T *sval,
                            int fill_cols) {
  int li = blockIdx.x * blockDim.x + threadIdx.x;
  int s = li >> 6, lane = li & 63;
  int nslices = (nsub + 63) >> 6;
  if (s >= nslices) return;
  long base = slice_ptr[s];
  int w = (int)((slice_ptr[s + 1] - base) >> 6);
  int r = -1, b = 0, len = 0;
  if (li < nsub) {
    r = rows ? rows[li] : li;
    b = rowptr[r];
    len = rowptr[r + 1] - b;
  }
  int padc = (len > 0) ? colidx[b + len - 1] : 0;
  for (int k = 0; k < w; k++) {
    long p = base + (long)k * 64 + lane;
    if (k < len) {
      if (fill_cols) scol[p] = colidx[b + k];
      sval[p] = vals[b + k];
    } else {
      if (fill_cols) scol[p] = padc;
      sval[p] = (T)0;
    }
  }
}

// The same for all rows (rows == nullptr) and rows of at most kSellLdsW entries: a block takes
// one slice, reads the slice's CSR entries (contiguous) into LDS with coalesced loads, and
// writes the slice column by column.
constexpr int kSellLdsW = 32;

template <class T>
__global__ __launch_bounds__(64) void k_sell_fill_lds(int nrows, const int *__restrict__ rowptr,
                                                      const int *__restrict__ colidx,
                                                      const T *__restrict__ vals,
                                                      const long *__restrict__ slice_ptr,
                                                      int *scol, T *sval, int fill_cols) {
  __shared__ T sv[64 * kSellLdsW];
  __shared__ int sc[64 * kSellLdsW];
  const int s = blockIdx.x, lane = threadIdx.x;
  const int r0 = s * 64, r = r0 + lane;
  const int e0 = rowptr[r0], e1 = rowptr[min(r0 + 64, nrows)];
  for (int e = e0 + lane; e < e1; e += 64) {
    sv[e - e0] = vals[e];
    sc[e - e0] = colidx[e];
  }
  int b = 0, len = 0;
  if (r < nrows) {
    b = rowptr[r] - e0;
    len = rowptr[r + 1] - rowptr[r];
  }
  __syncthreads();
  const long base = slice_ptr[s];
  const int w = (int)((slice_ptr[s + 1] - base) >> 6);
  const int padc = len > 0 ? sc[b + len - 1] : 0;
  for (int k = 0; k < w; k++) {
    const long p = base + (long)k * 64 + lane;
    if (k < len) {
      if (fill_cols) scol[p] = sc[b + k];
      sval[p] = sv[b + k];
    } else {
      if (fill_cols) scol[p] = padc;
      sval[p] = (T)0;
    }
  }
}

static bool csr_irregular(const flgpu_mat *A);
static int csr_lanes(const flgpu_mat *A);
// the CSR bounds of a colour's rows (below)
__global__ void k_row_span(int nsub, const int *__restrict__ rows, const int *__restrict__ rowptr,
                           int2 *__restrict__ span);

void sell_free(Sell &s) {
  dev_free(s.rows);
  dev_free(s.slice_ptr);
  dev_free(s.col);
  dev_free(s.val);
  dev_free(s.span);
  s = Sell();
}

template <class T>
static void sell_fill(flgpu_ctx *ctx, const flgpu_mat *A, Sell &s, int fill_cols) {
  if (s.nrows == 0 || s.span) return;
  if (!s.rows && s.maxw <= kSellLdsW) {
    k_sell_fill_lds<T><<<s.nslices, 64, 0, ctx->stream>>>(s.nrows, A->rowptr, A->colidx,
                                                          (const T *)A->vals, s.slice_ptr, s.col,
                                                          (T *)s.val, fill_cols);
    FLGPU_HIP(hipGetLastError());
    return;
  }
  int nthreads = s.nslices * 64;
  k_sell_fill<T><<<grid_for(nthreads, 256), 256, 0, ctx->stream>>>(
      s.nrows, s.rows, A->rowptr, A->colidx, (const T *)A->vals, s.slice_ptr, s.col, (T *)s.val,
      fill_cols);
  FLGPU_HIP(hipGetLastError());
}

// rows_host: row ids of the subset (nullptr: all rows).  A colour's rows that are long or irregular
// (csr_irregular, or over 27 entries) are swept from the CSR: they get their bounds (span) instead
// of stored entries.
static Sell sell_build(flgpu_mat *A, const std::vector<int> *rows_host) {
  flgpu_ctx *ctx = A->ctx;
  Sell s;
  s.nrows = rows_host ? (int)rows_host->size() : A->nrows;
  s.nslices = (s.nrows + 63) / 64;
  if (rows_host && s.nrows > 0) {
    s.rows = (int *)dev_alloc(sizeof(int) * s.nrows);
    FLGPU_HIP(hipMemcpyAsync(s.rows, rows_host->data(), sizeof(int) * s.nrows,
                             hipMemcpyHostToDevice, ctx->stream));
  }
  std::vector<int> w(s.nslices);
  std::vector<long> sp(s.nslices + 1, 0);
  if (s.nslices > 0) {
    int *dw = (int *)dev_alloc(sizeof(int) * s.nslices);
    k_slice_width<<<grid_for((long)s.nslices * 64, 256), 256, 0, ctx->stream>>>(
        s.nrows, s.rows, A->rowptr, dw);
    FLGPU_HIP(hipGetLastError());
    FLGPU_HIP(hipMemcpyAsync(w.data(), dw, sizeof(int) * s.nslices, hipMemcpyDeviceToHost,
                             ctx->stream));
    FLGPU_HIP(hipStreamSynchronize(ctx->stream));
    dev_free(dw);
  }
  for (int i = 0; i < s.nslices; i++) {
    sp[i + 1] = sp[i] + 64L * w[i];
    s.maxw = std::max(s.maxw, w[i]);
  }
  if (rows_host && s.nrows > 0 && (csr_irregular(A) || s.maxw > 27)) {
    s.span = dev_alloc(sizeof(int2) * (size_t)s.nrows);
    k_row_span<<<grid_for(s.nrows, 256), 256, 0, ctx->stream>>>(s.nrows, s.rows, A->rowptr,
                                                                (int2 *)s.span);
    FLGPU_HIP(hipGetLastError());
    return s;
  }
  s.nstored = sp[s.nslices];
  s.slice_ptr = (long *)dev_alloc(sizeof(long) * (s.nslices + 1));
  FLGPU_HIP(hipMemcpyAsync(s.slice_ptr, sp.data(), sizeof(long) * (s.nslices + 1),
                           hipMemcpyHostToDevice, ctx->stream));
  s.col = (int *)dev_alloc(sizeof(int) * s.nstored);
  s.val = dev_alloc(prec_bytes(A->prec) * s.nstored);
  if (A->prec == FLGPU_F64) sell_fill<double>(ctx, A, s, 1);
  else sell_fill<float>(ctx, A, s, 1);
  FLGPU_HIP(hipStreamSynchronize(ctx->stream));
  return s;
}

Sell sell_build_rows(flgpu_mat *A, const std::vector<int> &rows) { return sell_build(A, &rows); }

// ---- diagonal -----------------------------------------------------------------------

// pos[r] = the position of A(r, r) in the CSR (the last one if repeated), -1 if absent: 32
// lanes per row read the row's columns side by side (coalesced)
__global__ __launch_bounds__(256) void k_diagpos32(int n, const int *__restrict__ rowptr,
                                                   const int *__restrict__ colidx, int *pos) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = (int)(t >> 5), k = (int)(t & 31);
  if (r >= n) return;  // the 32 lanes of a row leave together
  int p = -1;
  for (int e = rowptr[r] + k; e < rowptr[r + 1]; e += 32)
    if (colidx[e] == r) p = e;
  for (int off = 16; off > 0; off >>= 1) p = max(p, __shfl_xor(p, off, 32));
  if (k == 0) pos[r] = p;
}

template <class T>
__global__ void k_diag(int n, const int *pos, const T *vals, T *diag) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int p = pos[r];
  diag[r] = p >= 0 ? vals[p] : (T)0;
}

// T = A^T with T's pattern already built: T_cf = A_fc (row c of T, column f)
template <class T>
__global__ void k_transpose_gather(int nrows_t, const int *__restrict__ trowptr,
                                   const int *__restrict__ tcolidx, T *tvals,
                                   const int *__restrict__ rowptr, const int *__restrict__ colidx,
                                   const T *__restrict__ vals) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrows_t) return;
  for (int p = trowptr[c]; p < trowptr[c + 1]; p++) {
    int f = tcolidx[p];
    T v = (T)0;
    for (int e = rowptr[f]; e < rowptr[f + 1]; e++)
      if (colidx[e] == c) {
        v = vals[e];
        break;
      }
    tvals[p] = v;
  }
}

static void diag_refresh(flgpu_mat *A) {
  int n = std::min(A->nrows, A->ncols);
  if (n == 0) return;
  if (A->prec == FLGPU_F64)
    k_diag<double><<<grid_for(n, 256), 256, 0, A->ctx->stream>>>(n, A->diagpos, (const double *)A->vals,
                                                                 (double *)A->diag);
  else
    k_diag<float><<<grid_for(n, 256), 256, 0, A->ctx->stream>>>(n, A->diagpos, (const float *)A->vals,
                                                                (float *)A->diag);
  FLGPU_HIP(hipGetLastError());
}

flgpu_mat *mat_new(flgpu_ctx *ctx, int nrows, int ncols, long nnz, int prec) {
  FLGPU_REQUIRE(nrows >= 0 && ncols >= 0 && nnz >= 0, "negative matrix dimensions");
  FLGPU_REQUIRE(nnz <= 0x7fffffffL, "nnz exceeds the int32 index range");
  FLGPU_REQUIRE(prec == FLGPU_F64 || prec == FLGPU_F32, "precision must be FLGPU_F64 or FLGPU_F32");
  flgpu_mat *A = new flgpu_mat;
  A->ctx = ctx;
  A->nrows = nrows;
  A->ncols = ncols;
  A->nnz = nnz;
  A->prec = prec;
  A->rowptr = (int *)dev_alloc(sizeof(int) * (nrows + 1));
  A->colidx = (int *)dev_alloc(sizeof(int) * nnz);
  A->vals = dev_alloc(prec_bytes(prec) * nnz);
  return A;
}

void mat_finish(flgpu_mat *A) {
  flgpu_ctx *ctx = A->ctx;
  int n = std::min(A->nrows, A->ncols);
  A->diagpos = (int *)dev_alloc(sizeof(int) * std::max(n, 1));
  A->diag = dev_alloc(prec_bytes(A->prec) * std::max(n, 1));
  if (n > 0) {
    k_diagpos32<<<grid_for(32L * n, 256), 256, 0, ctx->stream>>>(n, A->rowptr, A->colidx,
                                                                 A->diagpos);
    FLGPU_HIP(hipGetLastError());
    diag_refresh(A);
  }
  A->sell = sell_build(A, nullptr);
  A->lanes = csr_lanes(A);
  if (is_q1_lattice(A)) {
    A->val27 = dev_alloc(prec_bytes(A->prec) * 27 * (size_t)A->nrows);
    stencil_refresh(A);
  }
}

void mat_free(flgpu_mat *A) {
  if (!A) return;
  dev_free(A->rowptr);
  dev_free(A->colidx);
  dev_free(A->vals);
  dev_free(A->diagpos);
  dev_free(A->diag);
  sell_free(A->sell);
  for (auto &s : A->colour_sell) sell_free(s);
  if (A->transpose) mat_free(A->transpose);
  dev_free(A->alpha);
  dev_free(A->cell);
  dev_free(A->kref);
  dev_free(A->elem);
  dev_free(A->sor_work);
  dev_free(A->val27);
  dev_free(A->tp27);
  dev_free(A->blk_inv);
  dev_free(A->dot_part);
  delete A;
}

// values no longer follow the per-cell form (new values or another ordering)
void drop_alpha(flgpu_mat *A) {
  if (A->alpha) layout_changed(A);
  dev_free(A->alpha);
  A->alpha = nullptr;
}

// new values that are no sum over the lattice's cells
void drop_cells(flgpu_mat *A) {
  if (A->cell || A->elem) layout_changed(A);
  for (void **p : {&A->cell, &A->kref, &A->elem}) {
    dev_free(*p);
    *p = nullptr;
  }
}

void mat_refresh_values(flgpu_mat *A) {
  if (A->q2t || A->tp_geo) layout_changed(A);
  A->q2t = 0;  // other values than the interpolation's
  A->tp_geo = false;
  diag_refresh(A);
  stencil_refresh(A);
  if (A->tp_kind) tp_prepare(A);
  if (A->blk_inv) blocks_prepare(A);
  if (A->prec == FLGPU_F64) {
    sell_fill<double>(A->ctx, A, A->sell, 0);
    for (auto &s : A->colour_sell) sell_fill<double>(A->ctx, A, s, 0);
  } else {
    sell_fill<float>(A->ctx, A, A->sell, 0);
    for (auto &s : A->colour_sell) sell_fill<float>(A->ctx, A, s, 0);
  }
  if (A->transpose) {
    // same pattern: the transpose's values are gathered from the new ones
    flgpu_mat *T = A->transpose;
    if (T->nrows > 0) {
      if (A->prec == FLGPU_F64)
        k_transpose_gather<double><<<grid_for(T->nrows, 256), 256, 0, A->ctx->stream>>>(
            T->nrows, T->rowptr, T->colidx, (double *)T->vals, A->rowptr, A->colidx,
            (const double *)A->vals);
      else
        k_transpose_gather<float><<<grid_for(T->nrows, 256), 256, 0, A->ctx->stream>>>(
            T->nrows, T->rowptr, T->colidx, (float *)T->vals, A->rowptr, A->colidx,
            (const float *)A->vals);
      FLGPU_HIP(hipGetLastError());
    }
    mat_refresh_values(T);
  }
}

static void download_csr(const flgpu_mat *A, std::vector<int> &rp, std::vector<int> &ci,
                         std::vector<double> *v) {
  flgpu_ctx *ctx = A->ctx;
  rp.resize(A->nrows + 1);
  ci.resize(A->nnz);
  FLGPU_HIP(hipMemcpyAsync(rp.data(), A->rowptr, sizeof(int) * (A->nrows + 1),
                           hipMemcpyDeviceToHost, ctx->stream));
  FLGPU_HIP(hipMemcpyAsync(ci.data(), A->colidx, sizeof(int) * A->nnz, hipMemcpyDeviceToHost,
                           ctx->stream));
  if (v) {
    v->resize(A->nnz);
    if (A->prec == FLGPU_F64) {
      FLGPU_HIP(hipMemcpyAsync(v->data(), A->vals, sizeof(double) * A->nnz,
                               hipMemcpyDeviceToHost, ctx->stream));
    } else {
      double *tmp = (double *)dev_alloc(sizeof(double) * A->nnz);
      vcopy(ctx, A->nnz, FLGPU_F32, A->vals, FLGPU_F64, tmp);
      FLGPU_HIP(hipMemcpyAsync(v->data(), tmp, sizeof(double) * A->nnz, hipMemcpyDeviceToHost,
                               ctx->stream));
      FLGPU_HIP(hipStreamSynchronize(ctx->stream));
      dev_free(tmp);
    }
  }
  FLGPU_HIP(hipStreamSynchronize(ctx->stream));
}

static void upload_vals(flgpu_mat *A, const double *vals) {
  flgpu_ctx *ctx = A->ctx;
  if (A->nnz == 0) return;
  if (A->prec == FLGPU_F64) {
    FLGPU_HIP(hipMemcpyAsync(A->vals, vals, sizeof(double) * A->nnz, hipMemcpyHostToDevice,
                             ctx->stream));
    FLGPU_HIP(hipStreamSynchronize(ctx->stream));
  } else {
    double *tmp = (double *)dev_alloc(sizeof(double) * A->nnz);
    FLGPU_HIP(hipMemcpyAsync(tmp, vals, sizeof(double) * A->nnz, hipMemcpyHostToDevice,
                             ctx->stream));
    vcopy(ctx, A->nnz, FLGPU_F64, tmp, FLGPU_F32, A->vals);
    FLGPU_HIP(hipStreamSynchronize(ctx->stream));
    dev_free(tmp);
  }
}

// Transpose via the host (setup only): columns of A become rows, row
// indices ascending within each new row.
void mat_build_transpose(const flgpu_mat *A) {
  if (A->transpose) return;
  std::vector<int> rp, ci, trp(A->ncols + 1, 0), tci(A->nnz);
  std::vector<double> v, tv(A->nnz);
  download_csr(A, rp, ci, &v);
  for (long e = 0; e < A->nnz; e++) trp[ci[e] + 1]++;
  for (int c = 0; c < A->ncols; c++) trp[c + 1] += trp[c];
  std::vector<int> fill(trp.begin(), trp.end() - 1);
  for (int r = 0; r < A->nrows; r++)
    for (int e = rp[r]; e < rp[r + 1]; e++) {
      int p = fill[ci[e]]++;
      tci[p] = r;
      tv[p] = v[e];
    }
  flgpu_mat *T = mat_new(A->ctx, A->ncols, A->nrows, A->nnz, A->prec);
  FLGPU_HIP(hipMemcpyAsync(T->rowptr, trp.data(), sizeof(int) * (A->ncols + 1),
                           hipMemcpyHostToDevice, A->ctx->stream));
  FLGPU_HIP(hipMemcpyAsync(T->colidx, tci.data(), sizeof(int) * A->nnz, hipMemcpyHostToDevice,
                           A->ctx->stream));
  upload_vals(T, tv.data());
  mat_finish(T);
  const_cast<flgpu_mat *>(A)->transpose = T;
  layout_changed(const_cast<flgpu_mat *>(A));
}

flgpu_mat *mat_convert(const flgpu_mat *A, int prec) {
  flgpu_ctx *ctx = A->ctx;
  flgpu_mat *B = mat_new(ctx, A->nrows, A->ncols, A->nnz, prec);
  FLGPU_HIP(hipMemcpyAsync(B->rowptr, A->rowptr, sizeof(int) * (A->nrows + 1),
                           hipMemcpyDeviceToDevice, ctx->stream));
  if (A->nnz > 0) {
    FLGPU_HIP(hipMemcpyAsync(B->colidx, A->colidx, sizeof(int) * A->nnz,
                             hipMemcpyDeviceToDevice, ctx->stream));
    vcopy(ctx, A->nnz, A->prec, A->vals, prec, B->vals);
  }
  B->lat_dim = A->lat_dim;
  B->lat_order = A->lat_order;
  B->lat_n = A->lat_n;
  B->lat_f = A->lat_f;
  B->tp_kind = A->tp_kind;
  B->tp_nc = A->tp_nc;
  B->q2t = A->q2t;
  B->tp_geo = A->tp_geo;
  B->q2_nc = A->q2_nc;
  if (A->alpha) {
    long nc = (long)A->lat_n * A->lat_n * A->lat_n;
    B->alpha = dev_alloc(prec_bytes(prec) * nc);
    vcopy(ctx, nc, A->prec, A->alpha, prec, B->alpha);
    for (int j = 0; j < 8; j++) B->kt[j] = A->kt[j];
  }
  if (A->cell) {
    long nc = 1;
    for (int k = 0; k < A->lat_dim; k++) nc *= A->lat_n;
    B->cell = dev_alloc(prec_bytes(prec) * nc);
    vcopy(ctx, nc, A->prec, A->cell, prec, B->cell);
    lattice_set_kref(B);
  }
  mat_finish(B);
  if (A->transpose) B->transpose = mat_convert(A->transpose, prec);
  if (B->tp_kind && !(B->tp_kind == 1 && B->tp_geo)) tp_prepare(B);
  if (A->ncolours > 0) {
    // rebuild the colour subsets from A's row lists
    std::vector<int> colour(A->nrows, 0);
    for (int c = 0; c < A->ncolours; c++) {
      const Sell &s = A->colour_sell[c];
      std::vector<int> rows(s.nrows);
      if (s.nrows)
        FLGPU_HIP(hipMemcpy(rows.data(), s.rows, sizeof(int) * s.nrows, hipMemcpyDeviceToHost));
      for (int r : rows) colour[r] = c;
    }
    set_colouring(B, A->ncolours, colour.data());
  }
  return B;
}

void set_colouring(flgpu_mat *A, int ncolours, const int *colour) {
  FLGPU_REQUIRE(A->nrows == A->ncols, "colouring needs a square matrix");
  FLGPU_REQUIRE(ncolours >= 1, "ncolours must be >= 1");
  std::vector<std::vector<int>> rows(ncolours);
  for (int r = 0; r < A->nrows; r++) {
    FLGPU_REQUIRE(colour[r] >= 0 && colour[r] < ncolours, "colour out of range");
    rows[colour[r]].push_back(r);
  }
  // same-colour rows must not couple (otherwise the sweep would not be the
  // sequential <sor> sweep in (colour, index) order)
  std::vector<int> rp, ci;
  download_csr(A, rp, ci, nullptr);
  for (int r = 0; r < A->nrows; r++)
    for (int e = rp[r]; e < rp[r + 1]; e++)
      FLGPU_REQUIRE(ci[e] == r || colour[ci[e]] != colour[r],
                    "colouring couples two rows of one colour");
  for (auto &s : A->colour_sell) sell_free(s);
  A->colour_sell.clear();
  layout_changed(A);
  for (int c = 0; c < ncolours; c++) A->colour_sell.push_back(sell_build_rows(A, rows[c]));
  A->ncolours = ncolours;
}

// ---- kernels ----------------------------------------------------------------------

template <class T>
__device__ __forceinline__ T ld_stream(const T *p) {
  return __builtin_nontemporal_load(p);
}

// acc + sum_k (alpha x[col_k]) val_k over the w entries of one SELL row (stride 64), in
// order.  Chunks of 8: the 8 values and columns, then the 8 gathers, then the 8
// products, so a chunk costs two memory latencies rather than two per entry.
template <class T>
__device__ __forceinline__ T sell_row(const T *__restrict__ vp, const int *__restrict__ cp, int w,
                                      T alpha, const T *__restrict__ x, T acc) {
  constexpr int C = 8;
  int k = 0;
  for (; k + C <= w; k += C) {
    T a[C], xv[C];
    int c[C];
#pragma unroll
    for (int j = 0; j < C; j++) {
      a[j] = ld_stream(vp + (long)(k + j) * 64);
      c[j] = ld_stream(cp + (long)(k + j) * 64);
    }
#pragma unroll
    for (int j = 0; j < C; j++) xv[j] = x[c[j]];
#pragma unroll
    for (int j = 0; j < C; j++) acc += (alpha * xv[j]) * a[j];
  }
  int rem = w - k;  // uniform over the slice
  if (rem > 0) {
    T a[C], xv[C];
    int c[C];
#pragma unroll
    for (int j = 0; j < C; j++) {
      a[j] = j < rem ? ld_stream(vp + (long)(k + j) * 64) : (T)0;
      c[j] = j < rem ? ld_stream(cp + (long)(k + j) * 64) : 0;
    }
#pragma unroll
    for (int j = 0; j < C; j++) xv[j] = j < rem ? x[c[j]] : (T)0;
#pragma unroll
    for (int j = 0; j < C; j++)
      if (j < rem) acc += (alpha * xv[j]) * a[j];
  }
  return acc;
}

// out[row] = beta*z[row] + sum_k (alpha*x[col]) * val  over one SELL structure.  DOT (here and in
// the other products): also the block's share of sum_i out_i x_i to dpart (all rows, alpha 1,
// beta 0); a pass over both vectors and a launch less for the conjugate gradients
template <class T, bool DOT = false>
__global__ __launch_bounds__(256) void k_sell_spmv(int nsub, int nslices, const int *__restrict__ rows,
                                                   const long *__restrict__ slice_ptr,
                                                   const int *__restrict__ col,
                                                   const T *__restrict__ val, T alpha,
                                                   const T *__restrict__ x, T beta, const T *z,
                                                   T *out, double *dpart = nullptr) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  int s = (int)lb * 4 + (threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  int li = s * 64 + lane;
  double d = 0;
  if (s < nslices && li < nsub) {
    long base = slice_ptr[s];
    int w = (int)((slice_ptr[s + 1] - base) >> 6);
    int row = rows ? rows[li] : li;
    T acc = (beta == (T)0) ? (T)0 : beta * z[row];
    acc = sell_row<T>(val + base + lane, col + base + lane, w, alpha, x, acc);
    out[row] = acc;
    if (DOT) d = (double)acc * (double)x[row];
  }
  if (DOT) block_part(d, dpart);
}

// The sum over one CSR row [b, e) by the G lanes that share it (l: this lane's place): every lane
// takes each G-th entry, four of them loaded before the x values they name, and the lanes' sums
// are added by exchanges.  All G lanes return the row's sum of (alpha x_col) val.  FP32 sums
// are formed in FP64 too: adding lane by lane, not on top of beta z, would otherwise lose up to a
// fifth more to rounding than SELL's order where a residual cancels.
template <class T, int G>
__device__ __forceinline__ double csr_row(const int *__restrict__ col, const T *__restrict__ val, int b,
                                     int e, int l, T alpha, const T *x) {
  constexpr int U = 4;
  double acc = 0;
  for (int k = b + l; k < e; k += G * U) {
    T a[U], xv[U];
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kk = min(k + u * G, e - 1);
      a[u] = val[kk];
      c[u] = col[kk];
    }
#pragma unroll
    for (int u = 0; u < U; u++) xv[u] = x[c[u]];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u * G < e) acc += (double)(alpha * xv[u]) * (double)a[u];
  }
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  return acc;
}

// out[row] = beta z[row] + sum_k (alpha x[col]) val from the CSR rows, G lanes per row (csr_lanes).
// Nothing is read for padding and a row of w entries costs w / G steps of a lane instead of w:
// irregular matrices are bound by the longest row of every 64 in SELL.  300 007 rows of 18
// entries on average (55 at most), FP64: 23.1 us, 3.4 TB/s of entries, 40.3 us from SELL;
// Q2 12^3 (15 625 rows of 58): 4.1 against 16.7 us.
template <class T, int G, bool DOT = false>
__global__ __launch_bounds__(256) void k_csr_spmv(int nrows, const int *__restrict__ rowptr,
                                                  const int *__restrict__ col,
                                                  const T *__restrict__ val, T alpha,
                                                  const T *__restrict__ x, T beta, const T *z,
                                                  T *out, double *dpart = nullptr,
                                                  T *zero = nullptr) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int row = (int)lb * (256 / G) + threadIdx.x / G, l = threadIdx.x % G;
  double d = 0;
  if (row < nrows) {  // the lanes of a row together
    const double acc = csr_row<T, G>(col, val, rowptr[row], rowptr[row + 1], l, alpha, x);
    if (l == 0) {
      const T o = beta == (T)0 ? (T)acc : (T)((double)beta * (double)z[row] + acc);
      out[row] = o;
      if (zero) zero[row] = (T)0;
      if (DOT) d = (double)o * (double)x[row];
    }
  }
  if (DOT) block_part(d, dpart);
}

// long or irregular rows, where SELL pads: the sweeps' colours are read from the CSR (eight lanes a
// row, a colour's rows being few), the products if csr_lanes finds that faster.  The lattice
// forms' matrices (order 1, the trilinear transfers) stay with SELL, whose order their other
// storage forms sum in.
static bool csr_irregular(const flgpu_mat *A) {
  const double pad = A->nnz > 0 ? (double)A->sell.nstored / A->nnz : 1.0;
  return !(A->lat_order == 1 || A->tp_nc > 0 || A->sell.maxw <= 8 || pad <= 1.15 ||
           (pad <= 1.5 && A->nrows > 400000));
}

// Lanes per row of the products from the CSR, 0: SELL.  A lane takes four entries at a time, so
// four lanes cost the same up to 16 entries and eight up to 32; SELL's time goes with the entries
// it stores.  Up to 100 000 rows the longest row's chain decides, and the CSR is as fast or
// faster throughout.  Above, SELL against 4 / 8 lanes, us: 390 000 rows of 7 (11 entries stored a
// row) FP64 11.0 against 11.9 / 19.5, (13) 12.9 against 11.9 / 19.7; of 11 (15) 14.6 against 13.6 /
// 20.5, (18) 17.2 against 18.5 / 20.4; of 15 (18) 16.8 against 20.7 / 21.5; of 18 (29) 27.9 against
// 25.2 / 23.3; of 24 (29) 26.7 against 30.1 / 26.7, (43) 42.8 against 37.6 / 36.8; of 40 (48) 43.4
// against 52.1 / 49.0, (71) 77.6 against 66.2 / 59.6; FP32 0.7..0.8 of these.  Rows of 18 on average and 55 at most, 300 007 of
// them: 40.3 against 23.1 with eight.  Order 2: 2D, 314 721 rows of 16, FP32 11.3 against 10.8 /
// 12.9; 3D, rows of 61: 117 649 FP64 30.8 against 25.1 / 20.1, 456 533 96.7 against 113.9 / 93.9 and
// FP32 69.2 against 55.5 / 47.7, 912 673 (there SELL's loads fill the GPU) 196 against 231 / 191
// and 123 against 163 / 137.
static int csr_lanes(const flgpu_mat *A) {
  if (!csr_irregular(A)) return 0;
  const double len = (double)A->nnz / A->nrows, stored = (double)A->sell.nstored / A->nrows;
  if (A->nrows > 300000 && stored <= 1.25 * len) return 0;
  if (A->nrows > 100000 && stored < (len < 10 || A->sell.maxw <= 16 ? 11.5 : 19.5)) return 0;
  return len < 17 ? 4 : 8;
}

template <class T>
static void launch_csr_spmv(const flgpu_mat *A, T alpha, const void *x, T beta, const void *z,
                            void *out, double *dpart = nullptr, void *zero = nullptr) {
  const int G = A->lanes;
  const unsigned g = xcd_grid(grid_for((long)A->nrows * G, 256));
  auto launch = [&](auto kern) {
    kern<<<g, 256, 0, A->ctx->stream>>>(A->nrows, A->rowptr, A->colidx, (const T *)A->vals, alpha,
                                        (const T *)x, beta, (const T *)z, (T *)out, dpart,
                                        (T *)zero);
  };
  if (dpart) launch(G == 4 ? k_csr_spmv<T, 4, true> : k_csr_spmv<T, 8, true>);
  else launch(G == 4 ? k_csr_spmv<T, 4> : k_csr_spmv<T, 8>);
  FLGPU_HIP(hipGetLastError());
}

template <class T>
static void launch_spmv(flgpu_ctx *ctx, const Sell &s, double alpha, const void *x, double beta,
                        const void *z, void *out, double *dpart = nullptr) {
  if (s.nrows == 0) return;
  unsigned g = xcd_grid(grid_for(s.nslices, 4));
  if (dpart)
    k_sell_spmv<T, true><<<g, 256, 0, ctx->stream>>>(
        s.nrows, s.nslices, s.rows, s.slice_ptr, s.col, (const T *)s.val, (T)alpha, (const T *)x,
        (T)beta, (const T *)z, (T *)out, dpart);
  else
    k_sell_spmv<T><<<g, 256, 0, ctx->stream>>>(s.nrows, s.nslices, s.rows, s.slice_ptr, s.col,
                                               (const T *)s.val, (T)alpha, (const T *)x, (T)beta,
                                               (const T *)z, (T *)out);
  FLGPU_HIP(hipGetLastError());
}

// ---- 3D Q1 lattice with a per-cell coefficient: A applied from alpha ---------------

// The neighbours along one axis (one nonzero offset): the Q1 stiffness of a cube couples the
// nodes of a common edge with exactly 0, and kt holds the FP64 Gauss sum's residue, about
// 1e-17 of kt[0]: such an entry is 1e-17 of the row's diagonal, far below the FP32 resolution
// (6e-8), so the FP32 per-cell passes skip those 6 terms; FP64 keeps them, as the assembled
// values do.
template <class T>
__device__ __forceinline__ constexpr bool q1_axis(int dz, int dy, int dx) {
  return sizeof(T) == 4 && (dz != 0) + (dy != 0) + (dx != 0) == 1;
}

// ---- whole-lattice passes in the per-cell form, blocked along z ---------------------------
// A thread owns QZB consecutive rows along z at one (y, x).  It loads its own x column of the
// 3 lines y-1..y+1 over the QZB + 2 planes and its own cell-factor column of the lines y-1, y
// over QZB + 1 cell planes (18 + 10 loads for 4 rows), and takes the x-1 and x+1 columns from
// the neighbouring lanes of its wave (DPP whole-wave shifts).  Each wave computes 62
// consecutive positions; its two edge lanes only load the columns its first and last position
// need.  Dirichlet values are zeroed as they are loaded, which is what the explicit zeros of
// the eliminated columns contribute.  Row i is the sum over its neighbours j, ascending, of
// (coef x_j) A_ij with A_ij = kt[|dz| 4 + |dy| 2 + |dx|] (sum of alpha over the cells i and j
// share, ascending).
enum { Q1_SPMV = 0, Q1_JACOBI = 1 };

template <class T> struct Q1KT {
  T k[8];
};

// value of lane - 1 (DPP wave_shr:1) and of lane + 1 (DPP wave_shl:1); 0 on the end lanes
__device__ __forceinline__ int lane_up_i(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x138, 0xf, 0xf, true);
}
__device__ __forceinline__ int lane_down_i(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x130, 0xf, 0xf, true);
}
__device__ __forceinline__ float lane_up(float v) { return __int_as_float(lane_up_i(__float_as_int(v))); }
__device__ __forceinline__ float lane_down(float v) {
  return __int_as_float(lane_down_i(__float_as_int(v)));
}
__device__ __forceinline__ double lane_up(double v) {
  return __hiloint2double(lane_up_i(__double2hiint(v)), lane_up_i(__double2loint(v)));
}
__device__ __forceinline__ double lane_down(double v) {
  return __hiloint2double(lane_down_i(__double2hiint(v)), lane_down_i(__double2loint(v)));
}

template <class T, class I>
__device__ __forceinline__ T ld_at(const T *__restrict__ p, I byte_offset) {
  return *(const T *)((const char *)p + byte_offset);
}

// OP = Q1_SPMV:   out_i = beta z_i + sum_j (coef x_j) A_ij          (v = z)
// OP = Q1_JACOBI: out_i = x_i + coef (b_i - sum_j A_ij x_j) / A_ii  (v = b, coef = damp;
//                 A_ii from the factors, 1 on Dirichlet rows)
// I is the offset type: unsigned when the byte size of a lattice vector fits 32 bits and the
// position count 31 bits.  QZB rows per thread.
// W2: every result is also stored to out2 in FP64 (the last step of a cycle run in FP32 for
// an FP64 caller).
// DOT (Q1_SPMV): the block's share of sum_i out_i x_i goes to dpart[blockIdx.x] (each lane its
// rows in order, then the wave, then the block's waves in order).
template <class T, int OP, class I, int QZB, bool W2 = false, bool DOT = false>
__global__ __launch_bounds__(256) void k_q1_zblock(int M, int n, const T *__restrict__ alpha,
                                                   Q1KT<T> kt, T coef, T beta,
                                                   const T *__restrict__ v,
                                                   const T *__restrict__ x,
                                                   T *__restrict__ out,
                                                   double *__restrict__ out2 = nullptr,
                                                   double *__restrict__ dpart = nullptr) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x & 63;
  const I Mi = (I)M, M2 = Mi * Mi;
  const I total = M2 * (I)((M + QZB - 1) / QZB);
  const I tw = ((I)lb * (blockDim.x / 64) + (threadIdx.x >> 6)) * 62 + (I)lane;  // position + 1
  const bool compute = lane >= 1 && lane <= 62 && tw <= total;  // lanes 0 and 63 are halo
  const I t = tw == 0 ? (I)0 : (tw - 1 < total ? tw - 1 : total - 1);  // every lane loads
  const I line = t / Mi, zb = line / Mi;
  const int gx = (int)(t - line * Mi), gy = (int)(line - zb * Mi), z0 = (int)zb * QZB;
  const bool xbd = gx == 0 || gx == M - 1;
  // byte offsets (the narrow I keeps them in 32 bits: loads then take one VGPR offset from
  // the SGPR base)
  constexpr I B = (I)sizeof(T);
  const I M2B = M2 * B;
  I yo[3];
  bool ybd[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    int y = min(max(gy + d - 1, 0), M - 1);
    yo[d] = (I)(y * M + gx) * B;
    ybd[d] = y == 0 || y == M - 1;
  }
  // plane k (z = z0 - 1 + k, clamped to the lattice) starts at zpl[k]; the stride is uniform,
  // so only plane 0 needs a product (zbase wraps around for z0 = 0, where plane 0 clamps to 0)
  I zpl[QZB + 2];
  const I zbase = (I)z0 * M2B - M2B, ztop = (I)(M - 1) * M2B;
#pragma unroll
  for (int k = 0; k < QZB + 2; k++)
    zpl[k] = k == 0 ? (z0 == 0 ? (I)0 : zbase) : min(zbase + (I)k * M2B, ztop);
  const I nnB = (I)n * (I)n * B;
  I co[2];
#pragma unroll
  for (int q = 0; q < 2; q++) co[q] = (I)(min(max(gy - 1 + q, 0), n - 1) * n + min(gx, n - 1)) * B;
  const I cb = (I)z0 * nnB - nnB, ctop = (I)(n - 1) * nnB;

  // loads, issued in the order the rows consume them (row r needs x planes r..r+2, cell
  // planes r, r+1 and v at row r): the in-order memory counter then lets row r start while
  // the later planes are in flight
  T xv[QZB + 2][3][3], xi[QZB], av[QZB + 1][2][2], vr[QZB];
  auto load_x = [&](int k) {
#pragma unroll
    for (int dy = 0; dy < 3; dy++) xv[k][dy][1] = ld_at(x, zpl[k] + yo[dy]);
  };
  auto load_a = [&](int k) {
    I zo = k == 0 ? (z0 == 0 ? (I)0 : cb) : min(cb + (I)k * nnB, ctop);
#pragma unroll
    for (int q = 0; q < 2; q++) av[k][q][1] = ld_at(alpha, zo + co[q]);
  };
  load_x(0);
  load_x(1);
  load_a(0);
#pragma unroll
  for (int r = 0; r < QZB; r++) {
    load_x(r + 2);
    load_a(r + 1);
    if (OP == Q1_SPMV) vr[r] = (beta == (T)0) ? (T)0 : ld_at(v, zpl[r + 1] + yo[1]);
    else vr[r] = ld_at(v, zpl[r + 1] + yo[1]);
  }

  // Dirichlet values zeroed (the row's own value kept in xi); the x-1 / x+1 columns and the x-1
  // cell column from the neighbouring lanes: the same line and z-block for every interior row
  // (a line ends only at a Dirichlet row, which reads none).  Every lane runs to the end (the
  // shifts read all lanes); only computing lanes store.
  auto prep_x = [&](int k) {
    int z = min(max(z0 - 1 + k, 0), M - 1);
    bool zbd = z == 0 || z == M - 1;
#pragma unroll
    for (int dy = 0; dy < 3; dy++) {
      T val = xv[k][dy][1];
      if (dy == 1 && k >= 1 && k <= QZB) xi[k - 1] = val;
      val = (zbd || ybd[dy] || xbd) ? (T)0 : val;
      xv[k][dy][1] = val;
      xv[k][dy][0] = lane_up(val);
      xv[k][dy][2] = lane_down(val);
    }
  };
  // cs[k][dy][dx]: the ordered sum over cell plane k of the cells an entry with in-plane
  // offset (dy, dx) shares; pl = kt * cs is the entry itself when the offset crosses planes
  // (dz = -1 of row k, dz = +1 of row k - 1).  An entry within a plane (dz = 0) continues
  // row r's plane-r sum with the plane-(r + 1) cells.
  T cs[QZB + 1][3][3], pl[QZB + 1][3][3];
  auto prep_a = [&](int k) {
#pragma unroll
    for (int q = 0; q < 2; q++) av[k][q][0] = lane_up(av[k][q][1]);
#pragma unroll
    for (int e = 0; e < 9; e++) {
      int dy = e / 3 - 1, dx = e % 3 - 1;
      T sum = (T)-0.0;
#pragma unroll
      for (int q = (dy > 0); q <= (dy >= 0); q++)
#pragma unroll
        for (int c = (dx > 0); c <= (dx >= 0); c++) sum += av[k][q][c];
      cs[k][dy + 1][dx + 1] = sum;
      pl[k][dy + 1][dx + 1] = kt.k[4 + (dy != 0) * 2 + (dx != 0)] * sum;
    }
  };
  const bool side = xbd || gy == 0 || gy == M - 1;
  const T cf = (OP == Q1_SPMV) ? coef : (T)-1;
  double dsum = 0.0;
  prep_x(0);
  prep_x(1);
  prep_a(0);
#pragma unroll
  for (int r = 0; r < QZB; r++) {
    prep_x(r + 2);
    prep_a(r + 1);
    const int zz = z0 + r;
    const I i = zpl[r + 1] + yo[1];  // row zz, clamped to the lattice
    const T acc0 = vr[r];
    T acc = acc0, d = (T)1;
#pragma unroll
    for (int k = 0; k < 27; k++) {
      int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
      if (q1_axis<T>(dz, dy, dx)) continue;
      T aij;
      if (dz != 0) {
        aij = pl[r + (dz > 0)][dy + 1][dx + 1];
      } else {
        T sum = cs[r][dy + 1][dx + 1];
#pragma unroll
        for (int q = (dy > 0); q <= (dy >= 0); q++)
#pragma unroll
          for (int c = (dx > 0); c <= (dx >= 0); c++) sum += av[r + 1][q][c];
        aij = kt.k[(dy != 0) * 2 + (dx != 0)] * sum;
      }
      if (k == 13) d = aij;
      acc += (cf * xv[r + 1 + dz][dy + 1][dx + 1]) * aij;
    }
    const bool dir = side || zz == 0 || zz == M - 1;
    T res;
    if (OP == Q1_SPMV) {
      res = dir ? acc0 + (cf * xi[r]) * (T)1 : acc;
    } else {
      T accd = acc0 + (cf * xi[r]) * (T)1;
      res = xi[r] + coef * (dir ? accd / (T)1 : acc / d);
    }
    if (compute && zz < M) {
      *(T *)((char *)out + i) = res;
      if (W2) *(double *)((char *)out2 + i * (I)(sizeof(double) / sizeof(T))) = (double)res;
      if (DOT) dsum += (double)res * (double)xi[r];
    }
  }
  if (DOT) {  // every lane gets here: no lane leaves the kernel early
    __shared__ double ws[4];
    for (int off = 32; off > 0; off >>= 1) dsum += __shfl_down(dsum, off, 64);
    if (lane == 0) ws[threadIdx.x >> 6] = dsum;
    __syncthreads();
    if (threadIdx.x == 0) dpart[blockIdx.x] = ((ws[0] + ws[1]) + ws[2]) + ws[3];
  }
}

// rows per thread of the per-cell passes (measured on 129^3 lattices: FP32 5 rows; FP64 3 for
// the product, 4 for the <jacobi> step)
#ifndef FLGPU_QZB_F32
#define FLGPU_QZB_F32 5
#endif
#ifndef FLGPU_QZB_F64_SPMV
#define FLGPU_QZB_F64_SPMV 3
#endif
#ifndef FLGPU_QZB_F64_JACOBI
#define FLGPU_QZB_F64_JACOBI 4
#endif

template <class T, int OP>
static void launch_q1_pass(const flgpu_mat *A, T coef, T beta, const void *v, const void *x,
                           void *out, double *out2 = nullptr, double *dpart = nullptr) {
  constexpr int QZB = sizeof(T) == 4 ? FLGPU_QZB_F32
                      : (OP == Q1_SPMV ? FLGPU_QZB_F64_SPMV : FLGPU_QZB_F64_JACOBI);
  int M = A->lat_n + 1;
  long total = (long)M * M * ((M + QZB - 1) / QZB);
  long waves = (total + 61) / 62;
  unsigned g = xcd_grid(grid_for(waves * 64, 256));
  Q1KT<T> kt;
  for (int b = 0; b < 8; b++) kt.k[b] = (T)A->kt[b];
  bool narrow = (long)M * M * M * (long)sizeof(T) < (1L << 32) && (long)g * 256 < (1L << 31);
  if constexpr (OP == Q1_JACOBI && sizeof(T) == 4) {
    if (out2) {  // the FP64 byte offsets must fit too
      if (narrow && (long)M * M * M * (long)sizeof(double) < (1L << 32))
        k_q1_zblock<T, OP, unsigned, QZB, true><<<g, 256, 0, A->ctx->stream>>>(
            M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x,
            (T *)out, out2);
      else
        k_q1_zblock<T, OP, unsigned long, QZB, true><<<g, 256, 0, A->ctx->stream>>>(
            M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x,
            (T *)out, out2);
      FLGPU_HIP(hipGetLastError());
      return;
    }
  }
  FLGPU_REQUIRE(out2 == nullptr, "an FP64 copy is written only by the FP32 <jacobi> pass");
  if constexpr (OP == Q1_SPMV) {
    if (dpart) {  // the product and its dot with x; 4 waves per block, as launched below
      if (narrow)
        k_q1_zblock<T, OP, unsigned, QZB, false, true><<<g, 256, 0, A->ctx->stream>>>(
            M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x,
            (T *)out, nullptr, dpart);
      else
        k_q1_zblock<T, OP, unsigned long, QZB, false, true><<<g, 256, 0, A->ctx->stream>>>(
            M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x,
            (T *)out, nullptr, dpart);
      FLGPU_HIP(hipGetLastError());
      return;
    }
  }
  FLGPU_REQUIRE(dpart == nullptr, "the dot is formed only by the per-cell product");
  if (narrow)
    k_q1_zblock<T, OP, unsigned, QZB><<<g, 256, 0, A->ctx->stream>>>(
        M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x, (T *)out);
  else
    k_q1_zblock<T, OP, unsigned long, QZB><<<g, 256, 0, A->ctx->stream>>>(
        M, A->lat_n, (const T *)A->alpha, kt, coef, beta, (const T *)v, (const T *)x, (T *)out);
  FLGPU_HIP(hipGetLastError());
}

// ---- the per-cell <sor> sweep --------------------------------------------------------------
// The Q1 stiffness of a cube couples the nodes of a common edge with exactly 0 (kt's entries for
// one nonzero offset are the Gauss sum's residue, 1e-17 of kt[0], and are left out here), so a
// row couples only to rows that differ in at least two of the parities (z, y, x).  Of the eight
// colours c = 4 z + 2 y + x in their order, 2k and 2k + 1 then do not see each other: a sweep
// needs four steps, one for each (z, y) parity, and a step's rows are whole lines.  With the
// edge terms gone a row is, per cell it shares with its neighbours,
//   alpha_c (kt[6] x(z', y') + kt[5] x(z', x') + kt[7] x(z', y', x') + kt[3] x(y', x')),
// ' marking the neighbour on the cell's side: 4 products a cell plane instead of the 9 entries'
// sums and products.  A wave takes 62 consecutive positions of the lines (lanes 1..62, lanes 0
// and 63 only load); a lane loads the x and cell columns of its own position and takes the x - 1
// and x + 1 columns from its neighbouring lanes: a row's x - 1 and x + 1 are on its own line (a
// line ends only at a Dirichlet row, which reads none).
// Bound by the memory (x, the cells, b and the new x of a parity: 47 MB of FP64 a step at 129^3)
// and, up to 65^3, by the launches.  A sweep in place, FP64: 129^3 29 us, 97^3 12.7; two launches
// with eight in-plane colours in LDS, from a copy of the strips' edges, took 51 and 46.
template <class T> struct SorCols {
  T off[2][3];  // x at (z -+ 1, y - 1..y + 1)
  T in[2];      // x at (z, y -+ 1)
  T a[2][2];    // cells (z - 1.., y - 1..) of cell column x
  T xi, b;
};

// OFF0: x is zero on the planes z -+ 1, IN0: on the lines y -+ 1 (or not wanted), ZERO: the row's
// own x is zero; those are not read.  Indexes are clamped into the lattice.
template <class T, bool OFF0, bool IN0, bool ZERO>
__device__ __forceinline__ void sor_load(SorCols<T> &C, int M, int n, int z, int y, int xc,
                                         const T *__restrict__ alpha, const T *xoff,
                                         const T *xin, const T *b) {
  const unsigned uM = (unsigned)M, un = (unsigned)n, ux = (unsigned)xc;
  const int xcc = min(xc, n - 1);
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const unsigned zo = (unsigned)min(max(z - 1 + 2 * p, 0), M - 1) * uM;
    const unsigned zc = (unsigned)min(max(z - 1 + p, 0), n - 1) * un;
    if (!OFF0)
#pragma unroll
      for (int d = 0; d < 3; d++)
        C.off[p][d] = xoff[(zo + (unsigned)min(max(y + d - 1, 0), M - 1)) * uM + ux];
#pragma unroll
    for (int q = 0; q < 2; q++)
      C.a[p][q] = alpha[(zc + (unsigned)min(max(y - 1 + q, 0), n - 1)) * un + (unsigned)xcc];
  }
  if (!IN0)
#pragma unroll
    for (int q = 0; q < 2; q++)
      C.in[q] = xin[((unsigned)z * uM + (unsigned)min(max(y - 1 + 2 * q, 0), M - 1)) * uM + ux];
  const unsigned i = ((unsigned)z * uM + (unsigned)y) * uM + ux;
  C.xi = ZERO ? (T)0 : xin[i];
  C.b = b[i];
}

// b_i - (the terms of the planes z -+ 1), the cell columns' sums be over those planes.  Every
// lane of the wave calls it (the shifts read all lanes); Dirichlet values are zeroed, which is
// what their eliminated columns contribute.
template <class T, bool OFF0>
__device__ __forceinline__ T sor_off(const SorCols<T> &C, int M, int z, int y, bool xbd,
                                     const Q1KT<T> &kt, T (&be)[2][2]) {
  T acc = C.b;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    T xs[3][3], a[2][2];
    if (!OFF0) {
      const bool zbd = p ? z + 1 >= M - 1 : z - 1 <= 0;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const bool bd = zbd || xbd || (d == 0 ? y - 1 <= 0 : d == 2 && y + 1 >= M - 1);
        const T v = bd ? (T)0 : C.off[p][d];
        xs[d][1] = v;
        xs[d][0] = lane_up(v);
        xs[d][2] = lane_down(v);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
      a[q][1] = C.a[p][q];
      a[q][0] = lane_up(C.a[p][q]);
    }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        be[q][c] = p ? be[q][c] + a[q][c] : a[q][c];
        if (!OFF0) {
          const T s = kt.k[6] * xs[2 * q][1] + kt.k[5] * xs[1][2 * c] +
                      kt.k[7] * xs[2 * q][2 * c];
          acc -= a[q][c] * s;
        }
      }
  }
  return acc;
}

// the correction (b_i - sum_j A_ij x_j) / A_ii from sor_off's sum and the in-plane corners cn
template <class T>
__device__ __forceinline__ T sor_corr(T acc, T xi, const T (&be)[2][2], const T (&cn)[2][2],
                                      const Q1KT<T> &kt) {
  const T s = (be[0][0] * cn[0][0] + be[0][1] * cn[0][1]) +
              (be[1][0] * cn[1][0] + be[1][1] * cn[1][1]);
  const T d = kt.k[0] * ((be[0][0] + be[0][1]) + (be[1][0] + be[1][1]));
  return (acc - kt.k[3] * s - d * xi) / d;
}

// the corners' values from the line columns of sor_load
template <class T>
__device__ __forceinline__ void sor_corners(const SorCols<T> &C, int M, int y, bool xbd,
                                            T (&cn)[2][2]) {
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const T v = xbd || (q ? y + 1 >= M - 1 : y - 1 <= 0) ? (T)0 : C.in[q];
    cn[q][0] = lane_up(v);
    cn[q][1] = lane_down(v);
  }
}

// One step of a sweep in place: the rows of parity (cz, cy).  b may be r: a row's b is read
// before its r is written.  ZERO: the sweep starts from x = 0, which is not read (OFF0, IN0: as
// in sor_load, for the sweep's first two steps and its first and third).
template <class T, bool OFF0, bool IN0, bool ZERO>
__global__ __launch_bounds__(256) void k_q1_sor_lines(int M, int n, int cz, int cy, int nyl,
                                                      unsigned total, FastDiv fM, Div1 fny,
                                                      const T *__restrict__ alpha, Q1KT<T> kt,
                                                      T omega, T *x, const T *b, T *r) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x & 63;
  const unsigned tw = (lb * 4 + (threadIdx.x >> 6)) * 62 + (unsigned)lane;  // position + 1
  const unsigned t = tw == 0 ? 0u : min(tw - 1, total - 1);
  const unsigned line = fdiv(t, fM), zi = fdiv(line, fny);
  const int xc = (int)(t - line * (unsigned)M);
  const int z = cz + 2 * (int)zi, y = cy + 2 * (int)(line - zi * (unsigned)nyl);
  SorCols<T> C;
  sor_load<T, OFF0, IN0, ZERO>(C, M, n, z, y, xc, alpha, x, x, b);
  const bool xbd = xc == 0 || xc == M - 1;
  T be[2][2], cn[2][2] = {};
  const T acc = sor_off<T, OFF0>(C, M, z, y, xbd, kt, be);
  if (!IN0) sor_corners<T>(C, M, y, xbd, cn);
  if (lane < 1 || lane > 62 || tw > total) return;
  const bool bd = xbd || y == 0 || y == M - 1 || z == 0 || z == M - 1;
  const T corr = bd ? C.b - C.xi : sor_corr<T>(acc, C.xi, be, cn, kt);
  const unsigned i = ((unsigned)z * (unsigned)M + (unsigned)y) * (unsigned)M + (unsigned)xc;
  if (r) r[i] = corr;
  x[i] = C.xi + omega * corr;
}

// Two steps of a sweep in one launch, out of place: the planes of one z parity, first the lines
// of y parity ap, then the others.  xs is x before the sweep, xoff x on the other planes (xs in
// the first launch, xd in the second), xd gets the new values.  A block owns the lines
// [y0, y0 + H) of a plane; the first step is also done for the line on either side that the
// second step reads, from the same values with the same arithmetic as by the block that owns
// it, and reaches the second step through LDS.  b must not be r.
template <class T, bool OFF0, bool ZERO>
__global__ __launch_bounds__(256) void k_q1_sor_planes(int M, int n, int pz, int ap, int H,
                                                       int S, int planes, FastDiv fM,
                                                       const T *__restrict__ alpha, Q1KT<T> kt,
                                                       T omega, const T *__restrict__ xs,
                                                       const T *xoff, T *xd,
                                                       const T *__restrict__ b, T *r) {
  extern __shared__ char sor_lds[];
  T *la = (T *)sor_lds;  // the first step's lines, Dirichlet values 0
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int zi = (int)(lb / (unsigned)S), s = (int)(lb - (unsigned)(zi * S));
  if (zi >= planes) return;  // the grid's padding (whole blocks)
  const int z = pz + 2 * zi, y0 = s * H, y1 = min(M, y0 + H);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool zbd = z == 0 || z == M - 1;
  int a0 = max(0, y0 - 1);
  a0 += (a0 ^ ap) & 1;
  const int a1 = min(M - 1, y1), na = a1 >= a0 ? ((a1 - a0) / 2 + 1) * M : 0;
  const int b0 = y0 + ((y0 ^ ap ^ 1) & 1), nb = b0 < y1 ? ((y1 - 1 - b0) / 2 + 1) * M : 0;
  for (int c0 = wave * 62; c0 < na; c0 += 4 * 62) {
    const int e = c0 + lane - 1, ec = min(max(e, 0), na - 1);
    const int l = (int)fdiv((unsigned)ec, fM), xc = ec - l * M, y = a0 + 2 * l;
    SorCols<T> C;
    sor_load<T, OFF0, ZERO, ZERO>(C, M, n, z, y, xc, alpha, xoff, xs, b);
    const bool xbd = xc == 0 || xc == M - 1;
    T be[2][2], cn[2][2] = {};
    const T acc = sor_off<T, OFF0>(C, M, z, y, xbd, kt, be);
    if (!ZERO) sor_corners<T>(C, M, y, xbd, cn);
    const bool bd = zbd || xbd || y == 0 || y == M - 1;
    const T corr = bd ? C.b - C.xi : sor_corr<T>(acc, C.xi, be, cn, kt);
    const T xn = C.xi + omega * corr;
    if (lane >= 1 && lane <= 62 && e < na) {
      la[e] = bd ? (T)0 : xn;
      if (y >= y0 && y < y1) {
        const unsigned i = ((unsigned)z * (unsigned)M + (unsigned)y) * (unsigned)M + (unsigned)xc;
        xd[i] = xn;
        if (r) r[i] = corr;
      }
    }
  }
  // the second step's loads are issued before the wait for the first step's lines
  SorCols<T> C;
  int c0 = wave * 62, e, l, xc;
  auto place = [&] {
    e = c0 + lane - 1;
    const int ec = min(max(e, 0), nb - 1);
    l = (int)fdiv((unsigned)ec, fM);
    xc = ec - l * M;
    sor_load<T, OFF0, true, ZERO>(C, M, n, z, b0 + 2 * l, xc, alpha, xoff, xs, b);
  };
  if (c0 < nb) place();
  __syncthreads();
  for (; c0 < nb;) {
    const int y = b0 + 2 * l;
    const bool xbd = xc == 0 || xc == M - 1;
    T be[2][2];
    const T acc = sor_off<T, OFF0>(C, M, z, y, xbd, kt, be);
    if (lane >= 1 && lane <= 62 && e < nb) {
      T corr = C.b - C.xi;
      if (!(zbd || xbd || y == 0 || y == M - 1)) {
        const T *up = la + ((y - 1 - a0) >> 1) * M + xc;
        const T cn[2][2] = {{up[-1], up[1]}, {up[M - 1], up[M + 1]}};
        corr = sor_corr<T>(acc, C.xi, be, cn, kt);
      }
      const unsigned i = ((unsigned)z * (unsigned)M + (unsigned)y) * (unsigned)M + (unsigned)xc;
      xd[i] = C.xi + omega * corr;
      if (r) r[i] = corr;
    }
    c0 += 4 * 62;
    if (c0 < nb) place();
  }
}

// All sweeps of a smoothing step on a lattice of at most 10^3 nodes by one block, a row per
// thread (its cells, b and x in registers, x of the others in LDS).  Threads are laid out by the
// rows' (z, y) parity, each parity starting a wave.  rmode 1: r = the last corrections, 2: r =
// the residual after the sweeps, 0: r is not written.  Two sweeps of 9^3 nodes and the residual
// take 4.7 us, by launches they took 32: the steps' chains of LDS reads bound it, not the rows.
template <class T>
__global__ __launch_bounds__(1024) void k_q1_sor_small(int M, int n, int steps, int backwards,
                                                       int rmode, int zero,
                                                       const T *__restrict__ alpha, Q1KT<T> kt,
                                                       T omega, T *x, const T *b, T *r) {
  __shared__ T xs[1000];
  int cls = 0, t = (int)threadIdx.x, cnt = 0;
  for (; cls < 4; cls++) {
    cnt = ((M - (cls >> 1) + 1) / 2) * ((M - (cls & 1) + 1) / 2) * M;
    const int pad = (cnt + 63) & ~63;
    if (t < pad) break;
    t -= pad;
  }
  const bool row = cls < 4 && t < cnt;
  const int nyl = (M - (cls & 1) + 1) / 2;
  const int line = row ? t / M : 0, xc = row ? t - line * M : 0;
  const int zi = row ? line / nyl : 0;
  const int z = (cls >> 1) + 2 * zi, y = (cls & 1) + 2 * (line - zi * nyl);
  const int i = (z * M + y) * M + xc;
  const bool in = row && xc > 0 && xc < M - 1 && y > 0 && y < M - 1 && z > 0 && z < M - 1;
  T a[2][2][2] = {}, bi = (T)0, xi = (T)0, d = (T)1, corr = (T)0;
  if (row) {
    bi = b[i];
    if (!zero) xi = x[i];
    xs[i] = in ? xi : (T)0;  // the eliminated columns
  }
  if (in) {
    T s = (T)0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int p = k >> 2, q = (k >> 1) & 1, c = k & 1;
      a[p][q][c] = alpha[((z - 1 + p) * n + y - 1 + q) * n + xc - 1 + c];
      s += a[p][q][c];
    }
    d = kt.k[0] * s;
  }
  const int M2 = M * M;
  auto sum = [&] {  // b_i minus the neighbours' terms
    T acc = bi, s3 = (T)0;
#pragma unroll
    for (int p = 0; p < 2; p++) {
      const T *v = xs + i + (p ? M2 : -M2);
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const int dy = q ? M : -M, dx = c ? 1 : -1;
          acc -= a[p][q][c] * (kt.k[6] * v[dy] + kt.k[5] * v[dx] + kt.k[7] * v[dy + dx]);
        }
    }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 2; c++)
        s3 += (a[0][q][c] + a[1][q][c]) * xs[i + (q ? M : -M) + (c ? 1 : -1)];
    return acc - kt.k[3] * s3;
  };
  __syncthreads();
  for (int k = 0; k < 4 * steps; k++) {
    if (row && cls == (backwards ? 3 - (k & 3) : (k & 3))) {
      corr = in ? (sum() - d * xi) / d : bi - xi;
      xi += omega * corr;
      if (in) xs[i] = xi;
    }
    __syncthreads();
  }
  if (row) {
    x[i] = xi;
    if (rmode == 1) r[i] = corr;
    else if (rmode == 2) r[i] = in ? sum() - d * xi : bi - xi;
  }
}

// ---- 3D Q1 lattice matrices in 27-point stencil storage ------------------------------

// val27[k][i] = A(i, i + off_k) for the CSR entries of row i, 0 elsewhere
template <class T>
__global__ void k_st27_fill(int M, const int *__restrict__ rowptr, const int *__restrict__ colidx,
                            const T *__restrict__ vals, T *val27) {
  long N = (long)M * M * M;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  for (int k = 0; k < 27; k++) val27[k * N + i] = (T)0;
  int x = (int)(i % M), y = (int)((i / M) % M), z = (int)(i / ((long)M * M));
  for (int e = rowptr[i]; e < rowptr[i + 1]; e++) {
    long j = colidx[e];
    int jx = (int)(j % M), jy = (int)((j / M) % M), jz = (int)(j / ((long)M * M));
    int ax = jx - x + 1, ay = jy - y + 1, az = jz - z + 1;
    // lattice patterns only hold neighbours; anything else is never stored
    if ((unsigned)ax > 2u || (unsigned)ay > 2u || (unsigned)az > 2u) continue;
    val27[(long)(az * 9 + ay * 3 + ax) * N + i] = vals[e];
  }
}

// The same for rows of at most 27 entries on lattices of M >= 3: a block takes 128 rows, reads
// their CSR entries (contiguous) into LDS with coalesced loads, and every thread walks its row
// once along the 27 neighbour columns in ascending order (columns that are no lattice neighbour
// are passed over), writing every plane with coalesced stores.
constexpr int kSt27Rows = 128;

template <class T>
__global__ __launch_bounds__(kSt27Rows) void k_st27_fill_lds(int M,
                                                             const int *__restrict__ rowptr,
                                                             const int *__restrict__ colidx,
                                                             const T *__restrict__ vals,
                                                             T *val27) {
  __shared__ T sv[kSt27Rows * 27];
  __shared__ int sc[kSt27Rows * 27];
  const long N = (long)M * M * M;
  const long r0 = (long)blockIdx.x * kSt27Rows, i = r0 + threadIdx.x;
  const int e0 = rowptr[r0], e1 = rowptr[min(r0 + kSt27Rows, N)];
  for (int e = e0 + (int)threadIdx.x; e < e1; e += kSt27Rows) {
    sv[e - e0] = vals[e];
    sc[e - e0] = colidx[e];
  }
  __syncthreads();
  if (i >= N) return;
  const long M2 = (long)M * M;
  const int x = (int)(i % M), y = (int)((i / M) % M), z = (int)(i / M2);
  int e = rowptr[i] - e0;
  const int eend = rowptr[i + 1] - e0;
#pragma unroll
  for (int k = 0; k < 27; k++) {
    const int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
    T v = (T)0;
    if ((unsigned)(x + dx) < (unsigned)M && (unsigned)(y + dy) < (unsigned)M &&
        (unsigned)(z + dz) < (unsigned)M) {
      const long j = i + dz * M2 + dy * M + dx;
      while (e < eend && sc[e] < j) e++;
      if (e < eend && sc[e] == j) v = sv[e++];
    }
    val27[k * N + i] = v;
  }
}

// acc + sum over the lattice neighbours j of row i (ascending j) of
// (coef x_j) A_ij; the same entries in the same order as the CSR row.  The 27
// values and neighbour x are loaded first (a neighbour outside the lattice has
// a stored 0 and reads x_i), then summed in order: one memory latency per row.
// coefficient k of row i, whose neighbour i + off is in the lattice when live.  SYM: the values
// are exactly symmetric (A(i, i + d) == A(i + d, i), flgpu_mat::st_sym), so the lower half
// (k < 13) is read from the upper plane 26 - k of the neighbour row: 14 planes are streamed
// instead of 27, and the values read are the same
template <class T, bool SYM>
__device__ __forceinline__ T st27_coef(const T *__restrict__ val27, long N, int k, long i, long off,
                                       bool live) {
  if (SYM && k < 13) return live ? val27[(26 - k) * N + i + off] : (T)0;
  return val27[k * N + i];
}

template <class T, bool SYM = false>
__device__ __forceinline__ T st27_row(int M, long N, long i, int z, int y, int x,
                                      const T *__restrict__ val27, T acc, T coef,
                                      const T *__restrict__ xv, T *dii) {
  long M2 = (long)M * M;
  bool lz[3] = {z > 0, true, z < M - 1}, ly[3] = {y > 0, true, y < M - 1},
       lx[3] = {x > 0, true, x < M - 1};
  T av[27], xn[27];
#pragma unroll
  for (int k = 0; k < 27; k++) {
    int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
    bool live = lz[dz + 1] && ly[dy + 1] && lx[dx + 1];
    long off = dz * M2 + dy * M + dx;
    av[k] = st27_coef<T, SYM>(val27, N, k, i, off, live);
    xn[k] = xv[live ? i + off : i];
  }
  *dii = av[13];
#pragma unroll
  for (int k = 0; k < 27; k++) acc += (coef * xn[k]) * av[k];
  return acc;
}

template <class T, bool SYM, bool DOT = false>
__global__ __launch_bounds__(256) void k_st27_spmv(int M, const T *__restrict__ val27, T coef,
                                                   const T *__restrict__ x, T beta, const T *z,
                                                   T *out, double *dpart = nullptr) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  long i = (long)lb * blockDim.x + threadIdx.x;
  long N = (long)M * M * M;
  double dot = 0;
  if (i < N) {
    int xx = (int)(i % M), yy = (int)((i / M) % M), zz = (int)(i / ((long)M * M));
    T acc = (beta == (T)0) ? (T)0 : beta * z[i];
    T d;
    acc = st27_row<T, SYM>(M, N, i, zz, yy, xx, val27, acc, coef, x, &d);
    out[i] = acc;
    if (DOT) dot = (double)acc * (double)x[i];
  }
  if (DOT) block_part(dot, dpart);
}

// ---- the stencil-form <sor> sweep in tiles ---------------------------------------------------
// Colours 0-3 lie on the even z planes, 4-7 on the odd ones, and a row couples to the other z
// parity only through the planes z - 1 and z + 1, which no row of its own parity changes.  So one
// launch sweeps the four in-plane colours of one parity's planes, out of place (xs before the
// sweep, xoff x on the other planes: xs in the first launch, xd in the second).  A block owns H
// lines of W columns of one plane.  Colour j of the four needs the in-plane values of the
// colours before it one node away, so the block computes it on 3 - j lines and columns beyond
// its own on each side, from the same values with the same arithmetic as the block owning them,
// and keeps x of the plane in LDS.  A thread has at most one row of a colour and 4 / G rows (G
// groups of threads take every G-th colour): before the colour phases it loads their
// coefficients, sums b and the terms of the planes z - 1 and z + 1 and keeps the nine in-plane
// coefficients in registers, so that a phase waits for LDS only.  FP32 rows take
// the three planes' sums and the diagonal term together in FP64 (their terms one by one cost as
// much again as the loads).  b must not be r.
// The coefficients' bytes bound it from 65^3 on (27 a row and once more for the rows beyond the
// tile), their latency below.  A sweep in a cycle, FP64: 17^3 11, 33^3 12, 65^3 22 us; strips of
// whole lines that loaded each colour's coefficients in its phase, and copies of the strips'
// edges, took 19, 21 and 42.
constexpr int kTileCols = 65;
constexpr int kTileRows(int H) { return ((H + 7) / 2) * ((kTileCols + 7) / 2); }  // of a colour

// OFF0: x is zero on the planes z -+ 1, ZERO: on the plane itself; those are not read.
template <class T, bool SYM, bool OFF0, bool ZERO, int H, int G>
__global__ __launch_bounds__((kTileRows(H) + 63) / 64 * 64 * G) void k_st27_sor_tiles(
    int M, int pz, int W, int ntx, int nty, int planes, int backwards,
    const T *__restrict__ val27, T omega, const T *__restrict__ xs, const T *xoff, T *xd,
    const T *__restrict__ b, T *r) {
  constexpr int LW = kTileCols + 8, P = (kTileRows(H) + 63) / 64 * 64;
  __shared__ T lx[(H + 8) * LW];  // x of lines y0 - 4.., columns x0 - 4..; 0 outside the lattice
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int tx = (int)(lb % (unsigned)ntx), tyz = (int)(lb / (unsigned)ntx);
  const int ty = tyz % nty, zi = tyz / nty;
  if (zi >= planes) return;  // the grid's padding (whole blocks)
  const int z = pz + 2 * zi, y0 = ty * H, y1 = min(M, y0 + H), x0 = tx * W, x1 = min(M, x0 + W);
  const int M2 = M * M;
  const size_t N = (size_t)M2 * (size_t)M;
  const T *val = val27;  // plane k: val + k N, uniform
  constexpr int NE = ((H + 8) * LW + P * G - 1) / (P * G);
#pragma unroll
  for (int u = 0; u < NE; u++) {
    const int e = (int)threadIdx.x + u * P * G;
    const int l = e / LW, y = y0 - 4 + l, x = x0 - 4 + e - l * LW;
    if (e < (H + 8) * LW)
      lx[e] = !ZERO && y >= 0 && y < M && x >= 0 && x < M
                  ? xs[(unsigned)z * (unsigned)M2 + (unsigned)(y * M + x)] : (T)0;
  }
  constexpr int R = 4 / G;
  const int g = (int)threadIdx.x / P, t = (int)threadIdx.x - g * P;
  double acc[R];
  T cf[R][9];
  int li[R];          // the row's place in lx, -1: none
  unsigned gi[R];     // its index, 0xffffffff: another block's
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int j = g + q * G, c = backwards ? 3 - j : j, cy = c >> 1, cx = c & 1, e = 3 - j;
    int ya = max(0, y0 - e), xa = max(0, x0 - e);
    ya += (ya ^ cy) & 1;
    xa += (xa ^ cx) & 1;
    const int ny = (min(M, y1 + e) - ya + 1) >> 1, nx = (min(M, x1 + e) - xa + 1) >> 1;
    const int ey = nx > 0 ? t / nx : 0;
    const int y = ya + 2 * ey, x = xa + 2 * (t - ey * nx);
    li[q] = -1;
    gi[q] = 0xffffffffu;
    acc[q] = 0.0;
    if (nx <= 0 || ey >= ny) continue;
    li[q] = (y - y0 + 4) * LW + x - x0 + 4;
    const unsigned i = (unsigned)z * (unsigned)M2 + (unsigned)(y * M + x);
    if (y >= y0 && y < y1 && x >= x0 && x < x1) gi[q] = i;
    const bool lz[3] = {z > 0, true, z < M - 1}, ly[3] = {y > 0, true, y < M - 1},
               lxx[3] = {x > 0, true, x < M - 1};
    const T bi = b[i];
    T sd[2] = {};  // the planes' sums
#pragma unroll
    for (int k = 0; k < 27; k++) {
      const int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
      if (OFF0 && dz != 0) continue;
      const bool live = lz[dz + 1] && ly[dy + 1] && lxx[dx + 1];
      const unsigned in = live ? i + (unsigned)(dz * M2 + dy * M + dx) : i;
      T v = SYM && k < 13 ? (val + (size_t)(26 - k) * N)[in] : (val + (size_t)k * N)[i];
      if (SYM && k < 13) v = live ? v : (T)0;
      if (dz == 0) cf[q][k - 9] = v;
      else sd[dz > 0] += (live ? xoff[in] : (T)0) * v;
    }
    acc[q] = ((double)bi - (double)sd[0]) - (double)sd[1];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int q = j / G;
    if (j % G == g && li[q] >= 0) {
      const T *v = lx + li[q];
      T sp = (T)0;
#pragma unroll
      for (int k = 0; k < 9; k++)
        if (k != 4) sp += v[(k / 3 - 1) * LW + k % 3 - 1] * cf[q][k];
      const double a = (acc[q] - (double)sp) - (double)v[0] * (double)cf[q][4];
      const T corr = (T)a / cf[q][4];
      const T xn = v[0] + omega * corr;
      lx[li[q]] = xn;
      if (gi[q] != 0xffffffffu) {
        xd[gi[q]] = xn;
        if (r) r[gi[q]] = corr;
      }
    }
    __syncthreads();
  }
}

bool is_q1_lattice(const flgpu_mat *A) {
  return A->lat_dim == 3 && A->lat_order == 1 &&
         (long)A->nrows == (long)(A->lat_n + 1) * (A->lat_n + 1) * (A->lat_n + 1) &&
         A->nrows == A->ncols;
}

// asym[0] = 1 unless every stored A(i, i + d), d in the lower half, equals A(i + d, i) and the
// coefficients of neighbours outside the lattice are zero
template <class T>
__global__ void k_st27_symcheck(int M, const T *__restrict__ val27, int *asym) {
  const long N = (long)M * M * M, M2 = (long)M * M;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int x = (int)(i % M), y = (int)((i / M) % M), z = (int)(i / M2);
  const bool lz[3] = {z > 0, true, z < M - 1}, ly[3] = {y > 0, true, y < M - 1},
             lx[3] = {x > 0, true, x < M - 1};
  bool bad = false;
  for (int k = 0; k < 13; k++) {
    int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
    T a = val27[k * N + i];
    if (lz[dz + 1] && ly[dy + 1] && lx[dx + 1])
      bad |= !(a == val27[(26 - k) * N + i + dz * M2 + dy * M + dx]);
    else
      bad |= !(a == (T)0);
  }
  if (bad) asym[0] = 1;
}

void stencil_refresh(flgpu_mat *A) {
  if (!A->val27) return;
  int M = A->lat_n + 1;
  long N = A->nrows;
  Scratch<int> flag(A->ctx, 1);
  int *asym = flag.p;
  FLGPU_HIP(hipMemsetAsync(asym, 0, sizeof(int), A->ctx->stream));
  const bool lds = M >= 3 && A->sell.maxw <= 27;
  const unsigned gl = (unsigned)((N + kSt27Rows - 1) / kSt27Rows);
  if (A->prec == FLGPU_F64) {
    if (lds)
      k_st27_fill_lds<double><<<gl, kSt27Rows, 0, A->ctx->stream>>>(
          M, A->rowptr, A->colidx, (const double *)A->vals, (double *)A->val27);
    else
      k_st27_fill<double><<<grid_for(N, 256), 256, 0, A->ctx->stream>>>(
          M, A->rowptr, A->colidx, (const double *)A->vals, (double *)A->val27);
    k_st27_symcheck<double><<<grid_for(N, 256), 256, 0, A->ctx->stream>>>(
        M, (const double *)A->val27, asym);
  } else {
    if (lds)
      k_st27_fill_lds<float><<<gl, kSt27Rows, 0, A->ctx->stream>>>(
          M, A->rowptr, A->colidx, (const float *)A->vals, (float *)A->val27);
    else
      k_st27_fill<float><<<grid_for(N, 256), 256, 0, A->ctx->stream>>>(
          M, A->rowptr, A->colidx, (const float *)A->vals, (float *)A->val27);
    k_st27_symcheck<float><<<grid_for(N, 256), 256, 0, A->ctx->stream>>>(
        M, (const float *)A->val27, asym);
  }
  FLGPU_HIP(hipGetLastError());
  int h = 1;
  FLGPU_HIP(hipMemcpyAsync(&h, asym, sizeof(int), hipMemcpyDeviceToHost, A->ctx->stream));
  FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
  if (A->st_sym != (h == 0)) layout_changed(A);
  A->st_sym = (h == 0);
}

void drop_stencil(flgpu_mat *A) {
  if (A->val27) layout_changed(A);
  dev_free(A->val27);
  A->val27 = nullptr;
  A->st_sym = false;
  dev_free(A->sor_work);
  A->sor_work = nullptr;
}

// ---- 3D order-1 lattice interpolation with the pattern implied ------------------------------
// 1-D: fine node i (0..2nc) has the coarse neighbours i/2 (even i) or (i-1)/2, (i+1)/2 (odd
// i), c(i) = 1 + (i & 1) of them, and its entries start at o(i) = i + i/2 of the S = 3nc + 1
// entries of the 1-D table.  Coarse node c has the fine neighbours 2c-1 (c > 0), 2c, 2c+1
// (c < nc), ct(c) of them, starting at ot(c) = 3c - 1 (c > 0), 0.  A 3-D row (z, y, x) of the
// tensor product starts at o(z) S^2 + c(z) (o(y) S + c(y) o(x)) and lists its entries in
// ascending column order, z-major.  The products below form every row exactly as the SELL
// product does: acc = beta z_i, then acc += (alpha x_j) a_ij in ascending j.

// start of fine row (fz, fy, fx) in the interpolation's values
__device__ __forceinline__ long tp_row_start(int nc, int fz, int fy, int fx) {
  const long S = 3L * nc + 1;
  return (long)(fz + fz / 2) * S * S +
         (long)(1 + (fz & 1)) * ((long)(fy + fy / 2) * S + (long)(1 + (fy & 1)) * (fx + fx / 2));
}

// (z, y, x) of lattice index i < M^3 < 2^31, M = dM.d
__device__ __forceinline__ void lat_decode(unsigned i, FastDiv dM, int &z, int &y, int &x) {
  const unsigned line = fdiv(i, dM), zz = fdiv(line, dM);
  x = (int)(i - line * dM.d);
  y = (int)(line - zz * dM.d);
  z = (int)zz;
}

// The interpolation's values as 27 planes over the coarse nodes c, for the fine nodes
// 2c + (a, b, e) of c's block, a, b, e in {0, 1} (parity classes in lexicographic order): class
// (a, b, e) owns 2^(a+b+e) planes from tp_class_base, one per coarse corner c + (pz, py, px),
// pz <= a, py <= b, px <= e, in the row's own (ascending column) order.  Classes whose fine
// node lies past the lattice (a = 1 at cz = nc, ...) hold zeros there.
__host__ __device__ constexpr int tp_class_base(int cls) {
  return cls == 0 ? 0 : cls == 1 ? 1 : cls == 2 ? 3 : cls == 3 ? 5 : cls == 4 ? 9
       : cls == 5 ? 11 : cls == 6 ? 15 : 19;
}

template <class T>
__global__ void k_tp8_fill(int nc, const T *__restrict__ vals, T *__restrict__ p27) {
  const int Mc = nc + 1, Mf = 2 * nc + 1;
  const long Nc = (long)Mc * Mc * Mc;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= Nc) return;
  const int cx = (int)(c % Mc), cy = (int)((c / Mc) % Mc), cz = (int)(c / ((long)Mc * Mc));
  for (int cls = 0; cls < 8; cls++) {
    const int a = cls >> 2, b = (cls >> 1) & 1, e = cls & 1;
    const int fz = 2 * cz + a, fy = 2 * cy + b, fx = 2 * cx + e;
    const bool in = fz < Mf && fy < Mf && fx < Mf;
    const long rs = in ? tp_row_start(nc, fz, fy, fx) : 0;
    for (int k = 0; k < (1 << (a + b + e)); k++)
      p27[(long)(tp_class_base(cls) + k) * Nc + c] = in ? vals[rs + k] : (T)0;
  }
}

// out = beta z + alpha P x: one thread per coarse node c writes the fine nodes of c's block
// from the 8 coarse values of the cell [c, c + 1]^3 and the 27 planes
// GEO: the weights of the trilinear interpolation, powers of 1/2 per odd axis and 0 in the rows and
// columns on the boundary, the same bits as the stored ones: 129^3 FP64 8.8 us, 18.0 with them
template <class T, bool GEO>
__global__ __launch_bounds__(256) void k_tp_prolong(int nc, FastDiv dMc,
                                                    const T *__restrict__ p27, T alpha,
                                                    const T *__restrict__ x, T beta,
                                                    const T *__restrict__ z, T *__restrict__ out) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const unsigned Mc = dMc.d, Mf = 2 * nc + 1, Nc = Mc * Mc * Mc;
  const unsigned c = lb * blockDim.x + threadIdx.x;
  if (c >= Nc) return;
  int cz, cy, cx;
  lat_decode(c, dMc, cz, cy, cx);
  const bool uz = cz < nc, uy = cy < nc, ux = cx < nc;  // the upper neighbours exist
  T xc[8], w[27], zf[8];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int pz = q >> 2, py = (q >> 1) & 1, px = q & 1;
    if ((!pz || uz) && (!py || uy) && (!px || ux))
      xc[q] = x[c + ((unsigned)pz * Mc + (unsigned)py) * Mc + (unsigned)px];
  }
  if (GEO) {
    const int cc[3] = {cz, cy, cx};
    T wa[3][3];  // per axis: even node; odd node's lower and upper neighbour
#pragma unroll
    for (int k = 0; k < 3; k++) {
      wa[k][0] = cc[k] == 0 || cc[k] == nc ? (T)0 : (T)1;
      wa[k][1] = cc[k] == 0 ? (T)0 : (T)0.5;
      wa[k][2] = cc[k] + 1 == nc ? (T)0 : (T)0.5;
    }
#pragma unroll
    for (int cls = 0; cls < 8; cls++) {
      const int a = cls >> 2, b = (cls >> 1) & 1, e = cls & 1;
#pragma unroll
      for (int pz = 0; pz <= a; pz++)
#pragma unroll
        for (int py = 0; py <= b; py++)
#pragma unroll
          for (int px = 0; px <= e; px++)
            w[tp_class_base(cls) + (pz * (b + 1) + py) * (e + 1) + px] =
                wa[0][a + pz] * wa[1][b + py] * wa[2][e + px];
    }
  } else {
#pragma unroll
    for (int k = 0; k < 27; k++) w[k] = p27[(unsigned long)k * Nc + c];
  }
  const unsigned f0 = ((unsigned)(2 * cz) * Mf + (unsigned)(2 * cy)) * Mf + (unsigned)(2 * cx);
#pragma unroll
  for (int cls = 0; cls < 8; cls++) {
    const int a = cls >> 2, b = (cls >> 1) & 1, e = cls & 1;
    if ((!a || uz) && (!b || uy) && (!e || ux) && beta != (T)0)
      zf[cls] = z[f0 + ((unsigned)a * Mf + (unsigned)b) * Mf + (unsigned)e];
  }
#pragma unroll
  for (int cls = 0; cls < 8; cls++) {
    const int a = cls >> 2, b = (cls >> 1) & 1, e = cls & 1;
    if ((!a || uz) && (!b || uy) && (!e || ux)) {
      T acc = (beta == (T)0) ? (T)0 : beta * zf[cls];
#pragma unroll
      for (int pz = 0; pz <= a; pz++)
#pragma unroll
        for (int py = 0; py <= b; py++)
#pragma unroll
          for (int px = 0; px <= e; px++)
            acc += (alpha * xc[(pz * 2 + py) * 2 + px]) *
                   w[tp_class_base(cls) + (pz * (b + 1) + py) * (e + 1) + px];
      out[f0 + ((unsigned)a * Mf + (unsigned)b) * Mf + (unsigned)e] = acc;
    }
  }
}

// coarse row c of the transpose: its fine neighbours per axis and where offset 0 sits
struct TpRow {
  int tz, ty, tx, lz, ly, lx;
  long off;
};
__device__ __forceinline__ TpRow tp_trow(int nc, int cz, int cy, int cx) {
  const long S = 3L * nc + 1;
  auto cnt = [&](int q) { return 3 - (q == 0) - (q == nc); };
  auto ot = [&](int q) { return q == 0 ? 0 : 3 * q - 1; };
  TpRow t;
  t.tz = cnt(cz);
  t.ty = cnt(cy);
  t.tx = cnt(cx);
  t.lz = cz > 0;
  t.ly = cy > 0;
  t.lx = cx > 0;
  t.off = (long)ot(cz) * S * S + (long)t.tz * ((long)ot(cy) * S + (long)t.ty * ot(cx));
  return t;
}

// tp27[k][c] from the transpose's CSR values
template <class T>
__global__ void k_tp27_fill(int nc, const T *__restrict__ tvals, T *__restrict__ t27) {
  const unsigned Mc = nc + 1;
  const unsigned Nc = Mc * Mc * Mc;
  const unsigned c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= Nc) return;
  const unsigned line = c / Mc;
  const int cx = (int)(c - line * Mc), cy = (int)(line % Mc), cz = (int)(line / Mc);
  const TpRow t = tp_trow(nc, cz, cy, cx);
  for (int e = 0; e < 27; e++) {
    const int iz = e / 9 - 1 + t.lz, iy = (e / 3) % 3 - 1 + t.ly, ix = e % 3 - 1 + t.lx;
    const bool live = iz >= 0 && iz < t.tz && iy >= 0 && iy < t.ty && ix >= 0 && ix < t.tx;
    t27[(long)e * Nc + c] = live ? tvals[t.off + (iz * t.ty + iy) * t.tx + ix] : (T)0;
  }
}

// out = beta z + alpha P^T r (coarse rows; t27 = the transpose's values as 27 planes).  FIRST:
// also the first <jacobi> step from zero on the coarse level, xo = damp (out / diag), as
// k_jacobi_zero forms it
template <class T, bool GEO, bool FIRST = false>
__global__ __launch_bounds__(256) void k_tp_restrict(int nc, FastDiv dMc,
                                                     const T *__restrict__ t27, T alpha,
                                                     const T *__restrict__ r, T beta,
                                                     const T *__restrict__ z,
                                                     T *__restrict__ out,
                                                     const T *__restrict__ diag = nullptr,
                                                     T damp = (T)0, T *__restrict__ xo = nullptr) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const unsigned Mf = 2 * nc + 1, Mc = dMc.d;
  const unsigned Nc = Mc * Mc * Mc;
  const unsigned c = lb * blockDim.x + threadIdx.x;
  if (c >= Nc) return;
  int cz, cy, cx;
  lat_decode(c, dMc, cz, cy, cx);
  const bool vz[3] = {cz > 0, true, cz < nc}, vy[3] = {cy > 0, true, cy < nc},
             vx[3] = {cx > 0, true, cx < nc};
  const unsigned f0 = ((unsigned)(2 * cz) * Mf + (unsigned)(2 * cy)) * Mf + (unsigned)(2 * cx);
  // GEO: as in k_tp_prolong (129^3 FP64 7.0 us, 15.0 with the values)
  const T inner = cz > 0 && cy > 0 && cx > 0 && cz < nc && cy < nc && cx < nc ? (T)1 : (T)0;
  T a[27], rv[27];
#pragma unroll
  for (int e = 0; e < 27; e++) {
    const int dz = e / 9 - 1, dy = (e / 3) % 3 - 1, dx = e % 3 - 1;
    const bool live = vz[dz + 1] && vy[dy + 1] && vx[dx + 1];
    a[e] = GEO ? inner * (dz ? (T)0.5 : (T)1) * (dy ? (T)0.5 : (T)1) * (dx ? (T)0.5 : (T)1)
               : t27[(long)e * Nc + c];
    if (live) rv[e] = r[f0 + (unsigned)((dz * (int)Mf + dy) * (int)Mf + dx)];
  }
  T acc = (beta == (T)0) ? (T)0 : beta * z[c];
#pragma unroll
  for (int e = 0; e < 27; e++) {
    const int dz = e / 9 - 1, dy = (e / 3) % 3 - 1, dx = e % 3 - 1;
    if (vz[dz + 1] && vy[dy + 1] && vx[dx + 1]) acc += (alpha * rv[e]) * a[e];
  }
  out[c] = acc;
  if (FIRST) xo[c] = damp * (acc / diag[c]);
}

void tp_prepare(flgpu_mat *T) {
  if (T->tp_kind == 0) return;
  const int nc = T->tp_nc;
  const long Nc = (long)(nc + 1) * (nc + 1) * (nc + 1);
  if (!T->tp27) {
    T->tp27 = dev_alloc(27 * Nc * prec_bytes(T->prec));
    layout_changed(T);
  }
  const unsigned g = grid_for(Nc, 256);
  if (T->tp_kind == 1) {
    if (T->prec == FLGPU_F64)
      k_tp8_fill<double><<<g, 256, 0, T->ctx->stream>>>(nc, (const double *)T->vals,
                                                        (double *)T->tp27);
    else
      k_tp8_fill<float><<<g, 256, 0, T->ctx->stream>>>(nc, (const float *)T->vals,
                                                       (float *)T->tp27);
  } else {
    if (T->prec == FLGPU_F64)
      k_tp27_fill<double><<<g, 256, 0, T->ctx->stream>>>(nc, (const double *)T->vals,
                                                         (double *)T->tp27);
    else
      k_tp27_fill<float><<<g, 256, 0, T->ctx->stream>>>(nc, (const float *)T->vals,
                                                        (float *)T->tp27);
  }
  FLGPU_HIP(hipGetLastError());
}

void tp_drop(flgpu_mat *A) {
  if (A->tp_kind == 1 && A->transpose) tp_drop(A->transpose);
  if (A->tp_kind || A->tp27) layout_changed(A);
  dev_free(A->tp27);
  A->tp27 = nullptr;
  A->tp_kind = 0;
}

// the same for order 2: products of A and its transpose from their stored values
static void q2t_drop(flgpu_mat *A) {
  if (A->q2t == 1 && A->transpose) q2t_drop(A->transpose);
  if (A->q2t) layout_changed(A);
  A->q2t = 0;
}

template <class T>
static void launch_tp(const flgpu_mat *A, T alpha, const void *x, T beta, const void *z,
                      void *out) {
  const int nc = A->tp_nc;
  const long Nc = (long)(nc + 1) * (nc + 1) * (nc + 1);
  unsigned g = xcd_grid(grid_for(Nc, 256));
  auto launch = [&](auto kern) {
    kern<<<g, 256, 0, A->ctx->stream>>>(nc, fast_div(nc + 1), (const T *)A->tp27, alpha,
                                        (const T *)x, beta, (const T *)z, (T *)out);
  };
  auto restricts = [&](auto kern) {
    kern<<<g, 256, 0, A->ctx->stream>>>(nc, fast_div(nc + 1), (const T *)A->tp27, alpha,
                                        (const T *)x, beta, (const T *)z, (T *)out, nullptr, (T)0,
                                        nullptr);
  };
  if (A->tp_kind == 1) launch(A->tp_geo ? k_tp_prolong<T, true> : k_tp_prolong<T, false>);
  else restricts(A->tp_geo ? k_tp_restrict<T, true> : k_tp_restrict<T, false>);
  FLGPU_HIP(hipGetLastError());
}

template <class T>
static void launch_st27_spmv(const flgpu_mat *A, T alpha, const T *x, T beta, const T *z, T *out,
                             double *dpart = nullptr) {
  auto launch = [&](auto kern) {
    kern<<<xcd_grid(grid_for(A->nrows, 256)), 256, 0, A->ctx->stream>>>(
        A->lat_n + 1, (const T *)A->val27, alpha, x, beta, z, out, dpart);
  };
  if (A->st_sym) launch(dpart ? k_st27_spmv<T, true, true> : k_st27_spmv<T, true>);
  else launch(dpart ? k_st27_spmv<T, false, true> : k_st27_spmv<T, false>);
  FLGPU_HIP(hipGetLastError());
}

bool restrict_first_step(const flgpu_mat *PT, const void *r, void *rhs, const flgpu_mat *Ac,
                         double damp, void *xo) {
  if (PT->tp_kind != 2 || !Ac->diag || Ac->nrows != PT->nrows) return false;
  const int nc = PT->tp_nc;
  const long Nc = (long)(nc + 1) * (nc + 1) * (nc + 1);
  unsigned g = xcd_grid(grid_for(Nc, 256));
  auto run = [&](auto t) {
    using T = decltype(t);
    auto launch = [&](auto kern) {
      kern<<<g, 256, 0, PT->ctx->stream>>>(nc, fast_div(nc + 1), (const T *)PT->tp27, (T)1,
                                           (const T *)r, (T)0, (const T *)rhs, (T *)rhs,
                                           (const T *)Ac->diag, (T)damp, (T *)xo);
    };
    launch(PT->tp_geo ? k_tp_restrict<T, true, true> : k_tp_restrict<T, false, true>);
  };
  if (PT->prec == FLGPU_F64) run(0.0);
  else run(0.0f);
  FLGPU_HIP(hipGetLastError());
  return true;
}

template <class S, class T>
__global__ void k_stage_first(long n, const S *__restrict__ r, T *__restrict__ b,
                              const T *__restrict__ diag, T damp, T *__restrict__ xo) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T bi = (T)r[i];
  b[i] = bi;
  xo[i] = damp * (bi / diag[i]);
}

void stage_first_step(const flgpu_mat *A, int rprec, const void *r, void *b, double damp,
                      void *xo) {
  long n = A->nrows;
  unsigned g = grid_for(n, 256);
  if (rprec == FLGPU_F64 && A->prec == FLGPU_F32)
    k_stage_first<double, float><<<g, 256, 0, A->ctx->stream>>>(
        n, (const double *)r, (float *)b, (const float *)A->diag, (float)damp, (float *)xo);
  else if (rprec == FLGPU_F32 && A->prec == FLGPU_F64)
    k_stage_first<float, double><<<g, 256, 0, A->ctx->stream>>>(
        n, (const float *)r, (double *)b, (const double *)A->diag, damp, (double *)xo);
  else if (A->prec == FLGPU_F64)
    k_stage_first<double, double><<<g, 256, 0, A->ctx->stream>>>(
        n, (const double *)r, (double *)b, (const double *)A->diag, damp, (double *)xo);
  else
    k_stage_first<float, float><<<g, 256, 0, A->ctx->stream>>>(
        n, (const float *)r, (float *)b, (const float *)A->diag, (float)damp, (float *)xo);
  FLGPU_HIP(hipGetLastError());
}

// ---- order-2 lattices with a coefficient constant per cell: products without the matrix ------
// out = beta z + alpha A x with A = sum over the cells of cell[c] Kref.  A workgroup owns the
// DOFs 2c, 2c + 1 (per axis) of a box of cells; its 256 lanes take the box's cells and those one
// below it per axis, which share DOFs with it.  Every lane applies the reference matrix to its
// cell's 3^DIM values of x from an LDS patch (zero at Dirichlet points, as the eliminated columns
// are) and leaves the scaled result in LDS; then every lane of the box adds up its 2^DIM rows,
// cells in ascending order.  Dirichlet rows are identity rows.
//
// Kref is the sum of the tensor products of one 1-D stiffness matrix K and 1-D mass matrices M of
// the reference interval.  Both are symmetric under reflection, so on (u0 + u2, u1, u0 - u2) they
// are a 2 x 2 block and a scalar: 315 multiply-adds and 108 additions per 3D cell instead of the
// 729 of the 27 x 27 matrix, with ten constants in scalar registers (the matrix itself, fetched by
// scalar loads, took 21.5 us at Q2 48^3, FP64).
// Bytes: 8 (FP32) or 16 per row instead of 62 matrix entries with their columns.  The latency of
// the three phases bounds small lattices, the waves in flight (LDS) large ones.
// Q2 48^3: FP64 15.2 us, FP32 14.2 us; 193 and 128 us from SELL.
template <class T>
struct Ref1D {  // a 1-D reference matrix on (sum, middle, difference): a, b; b, c; d
  T a, b, c, d;
};
template <class T>
__device__ __forceinline__ Ref1D<T> ref_mass() {  // 1/30 [4 2 -1; 2 16 2; -1 2 4]
  return {(T)(1.5 / 30), (T)(2.0 / 30), (T)(16.0 / 30), (T)(2.5 / 30)};
}
template <class T>
__device__ __forceinline__ Ref1D<T> ref_stiff() {  // 1/3 [7 -8 1; -8 16 -8; 1 -8 7]
  return {(T)(4.0 / 3), (T)(-8.0 / 3), (T)(16.0 / 3), (T)1};
}
// (e, m, o) of the line through u with stride S -> the matrix's product, plus `add` if given
template <class T>
__device__ __forceinline__ void ref_apply(const Ref1D<T> &R, T e, T m, T o, T &p, T &q, T &r) {
  p = R.a * e + R.b * m;
  q = R.b * e + R.c * m;
  r = R.d * o;
}
template <class T>
__device__ __forceinline__ void ref_add(const Ref1D<T> &R, T e, T m, T o, T &p, T &q, T &r) {
  p += R.a * e + R.b * m;
  q += R.b * e + R.c * m;
  r += R.d * o;
}

// v <- Kref v for the 3^DIM values of one cell, last axis fastest
template <class T, int DIM>
__device__ __forceinline__ void cell_matrix(T *v) {
  constexpr int NL = DIM == 3 ? 27 : 9;
  const Ref1D<T> Mm = ref_mass<T>(), Km = ref_stiff<T>();
  // to (sum, middle, difference) along every axis
#pragma unroll
  for (int st = 1; st < NL; st *= 3)
#pragma unroll
    for (int i = 0; i < NL; i++)
      if ((i / st) % 3 == 0) {
        const T u0 = v[i], u2 = v[i + 2 * st];
        v[i] = u0 + u2;
        v[i + 2 * st] = u0 - u2;
      }
  // last axis: a = M v, b = K v
  T a[NL], b[NL];
#pragma unroll
  for (int i = 0; i < NL; i += 3) {
    ref_apply(Mm, v[i], v[i + 1], v[i + 2], a[i], a[i + 1], a[i + 2]);
    ref_apply(Km, v[i], v[i + 1], v[i + 2], b[i], b[i + 1], b[i + 2]);
  }
  // middle axis (the first in 2D): a <- M a, b <- K a + M b
#pragma unroll
  for (int i = 0; i < NL; i++)
    if ((i / 3) % 3 == 0) {
      T m0, m1, m2, k0, k1, k2;
      if (DIM == 3) ref_apply(Mm, a[i], a[i + 3], a[i + 6], m0, m1, m2);
      ref_apply(Km, a[i], a[i + 3], a[i + 6], k0, k1, k2);
      ref_add(Mm, b[i], b[i + 3], b[i + 6], k0, k1, k2);
      if (DIM == 3) {
        a[i] = m0;
        a[i + 3] = m1;
        a[i + 6] = m2;
      }
      b[i] = k0;
      b[i + 3] = k1;
      b[i + 6] = k2;
    }
  // first axis: K a + M b
  if (DIM == 3) {
#pragma unroll
    for (int i = 0; i < 9; i++) {
      T k0, k1, k2;
      ref_apply(Km, a[i], a[i + 9], a[i + 18], k0, k1, k2);
      ref_add(Mm, b[i], b[i + 9], b[i + 18], k0, k1, k2);
      b[i] = k0;
      b[i + 9] = k1;
      b[i + 18] = k2;
    }
  }
  // back: first and last node from (half sum, middle, half difference)
#pragma unroll
  for (int st = 1; st < NL; st *= 3)
#pragma unroll
    for (int i = 0; i < NL; i++)
      if ((i / st) % 3 == 0) {
        const T p = b[i], q = b[i + 2 * st];
        b[i] = p + q;
        b[i + 2 * st] = p - q;
      }
#pragma unroll
  for (int i = 0; i < NL; i++) v[i] = b[i];
}

// Below this many rows the CSR product is faster: 15 625 rows (3D) 4.1 against 6.4 us, 9 409 (2D)
// 3.6 against 3.8; above, 35 937 (3D) 7.5 against 6.5, 37 249 (2D) 3.6 against 3.7, 103 041 (2D)
// 6.7 against 3.9, 117 649 (3D) 20.3 against 6.6 us (FP64).
constexpr int kCellApplyRows = 30000;

template <int DIM>
struct CellBox;
template <>
struct CellBox<3> {
  static constexpr int B[3] = {3, 7, 7};  // cells of the box: 4 x 8 x 8 lanes
};
template <>
struct CellBox<2> {
  static constexpr int B[3] = {0, 15, 15};  // 16 x 16 lanes
};

template <class T, int DIM, bool DOT = false>
__global__ __launch_bounds__(256) void k_cell_apply(int n, Div1 dby, Div1 dbx,
                                                    const T *__restrict__ cell, T alpha,
                                                    const T *__restrict__ x, T beta, const T *z,
                                                    T *out, unsigned nblk,
                                                    double *dpart = nullptr) {
  constexpr int NL = DIM == 3 ? 27 : 9;
  constexpr int PZ = DIM == 3 ? 2 * (CellBox<DIM>::B[0] + 1) + 1 : 1,
                PY = 2 * (CellBox<DIM>::B[1] + 1) + 1, PX = 2 * (CellBox<DIM>::B[2] + 1) + 1;
  constexpr int LX = CellBox<DIM>::B[2] + 1, LY = CellBox<DIM>::B[1] + 1;
  __shared__ T px[PZ * PY * PX];
  __shared__ T ye[NL * 256];
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  if (lb >= nblk) {
    if (DOT && threadIdx.x == 0) dpart[blockIdx.x] = 0.0;
    return;
  }
  const int tid = threadIdx.x, M = 2 * n + 1;
  unsigned u = lb, q = fdiv(u, dbx);
  const int cx0 = (int)(u - q * dbx.f.d) * CellBox<DIM>::B[2];
  u = q;
  q = fdiv(u, dby);
  const int cy0 = (int)(u - q * dby.f.d) * CellBox<DIM>::B[1];
  const int cz0 = DIM == 3 ? (int)q * CellBox<DIM>::B[0] : 0;
  // the x patch [2 c0 - 2, 2 (c0 + B)] per axis
  constexpr int NP = PZ * PY * PX, NS = (NP + 255) / 256;
  T pv[NS];
#pragma unroll
  for (int k = 0; k < NS; k++) {
    const int e = min(tid + k * 256, NP - 1);
    const int qx = 2 * cx0 - 2 + e % PX, qy = 2 * cy0 - 2 + (e / PX) % PY,
              qz = DIM == 3 ? 2 * cz0 - 2 + e / (PX * PY) : 1;
    const bool in = qx > 0 && qx < M - 1 && qy > 0 && qy < M - 1 &&
                    (DIM == 2 || (qz > 0 && qz < M - 1));
    const long idx = DIM == 3 ? ((long)qz * M + qy) * M + qx : (long)qy * M + qx;
    const T t = x[in ? idx : 0];
    pv[k] = in ? t : (T)0;
  }
#pragma unroll
  for (int k = 0; k < NS; k++)
    if (tid + k * 256 < NP) px[tid + k * 256] = pv[k];
  const int lx = tid % LX, ly = (tid / LX) % LY, lz = tid / (LX * LY);
  const int cx = cx0 - 1 + lx, cy = cy0 - 1 + ly, cz = DIM == 3 ? cz0 - 1 + lz : 0;
  const bool live = cx >= 0 && cx < n && cy >= 0 && cy < n && cz >= 0 && cz < n;
  const T fac = cell[live ? ((long)cz * n + cy) * n + cx : 0];
  // the rows 2c, 2c + 1 of this lane's cell; what they need besides the sums is loaded ahead
  const bool own = lx > 0 && ly > 0 && (DIM == 2 || lz > 0) && cx <= n && cy <= n && cz <= n;
  const long row0 = ((DIM == 3 ? (long)2 * cz * M : 0) + 2 * cy) * M + 2 * cx;
  T zv[1 << DIM];
#pragma unroll
  for (int t = 0; t < (1 << DIM); t++) {
    const int tx = t & 1, ty = (t >> 1) & 1, tz = DIM == 3 ? t >> 2 : 0;
    const bool in = own && (cx < n || !tx) && (cy < n || !ty) && (DIM == 2 || cz < n || !tz);
    if (beta != (T)0) zv[t] = z[in ? row0 + ((long)tz * M + ty) * M + tx : 0];
  }
  __syncthreads();
  double xv[NL];  // FP64 for FP32 too: the same rate, and no rounding before the cells' sums
  const int pb = ((DIM == 3 ? 2 * lz : 0) * PY + 2 * ly) * PX + 2 * lx;
#pragma unroll
  for (int j = 0; j < NL; j++) {
    const int o = DIM == 3 ? ((j / 9) * PY + (j / 3) % 3) * PX + j % 3 : (j / 3) * PX + j % 3;
    xv[j] = px[pb + o];
  }
  cell_matrix<double, DIM>(xv);
#pragma unroll
  for (int l = 0; l < NL; l++) ye[l * 256 + tid] = live ? (T)((double)fac * xv[l]) : (T)0;
  __syncthreads();
  double d = 0;
#pragma unroll
  for (int t = 0; t < (1 << DIM); t++) {
    const int tx = t & 1, ty = (t >> 1) & 1, tz = DIM == 3 ? t >> 2 : 0;
    const int qx = 2 * cx + tx, qy = 2 * cy + ty, qz = 2 * cz + tz;
    if (!own || qx >= M || qy >= M || qz >= M) continue;
    double s = 0;
#pragma unroll
    for (int c = 0; c < (1 << DIM); c++) {  // bit set: this lane's cell, else the one below
      const int ux = c & 1, uy = (c >> 1) & 1, uz = DIM == 3 ? c >> 2 : 1;
      if ((tx && !ux) || (ty && !uy) || (tz && !uz)) continue;  // interior node of this cell
      const int jx = ux ? tx : 2, jy = uy ? ty : 2, jz = uz ? tz : 2;
      const int l = DIM == 3 ? (jz * 3 + jy) * 3 + jx : jy * 3 + jx;
      const int src = tid - (ux ? 0 : 1) - (uy ? 0 : LX) - (uz ? 0 : LX * LY);
      s += (double)ye[l * 256 + src];
    }
    const long idx = row0 + ((long)tz * M + ty) * M + tx;
    const bool dir = qx == 0 || qx == M - 1 || qy == 0 || qy == M - 1 ||
                     (DIM == 3 && (qz == 0 || qz == M - 1));
    if (dir) s = (double)x[idx];
    s *= (double)alpha;
    const T o = beta == (T)0 ? (T)s : (T)((double)beta * (double)zv[t] + s);
    out[idx] = o;
    if (DOT) d += (double)o * (double)x[idx];
  }
  if (DOT) block_part(d, dpart);
}

// the boxes of an A; per axis into by, bx
static unsigned cell_boxes(const flgpu_mat *A, unsigned &by, unsigned &bx) {
  const int n = A->lat_n;
  auto boxes = [&](int B) { return (unsigned)((n + 1 + B - 1) / B); };
  if (A->lat_dim == 3) {
    by = boxes(CellBox<3>::B[1]);
    bx = boxes(CellBox<3>::B[2]);
    return boxes(CellBox<3>::B[0]) * by * bx;
  }
  by = boxes(CellBox<2>::B[1]);
  bx = boxes(CellBox<2>::B[2]);
  return by * bx;
}

template <class T>
static void launch_cell_apply(const flgpu_mat *A, T alpha, const void *x, T beta, const void *z,
                              void *out, double *dpart = nullptr) {
  unsigned by, bx;
  const unsigned nb = cell_boxes(A, by, bx);
  auto launch = [&](auto kern) {
    kern<<<xcd_grid(nb), 256, 0, A->ctx->stream>>>(A->lat_n, div1(by), div1(bx),
                                                   (const T *)A->cell, alpha, (const T *)x, beta,
                                                   (const T *)z, (T *)out, nb, dpart);
  };
  if (A->lat_dim == 3) launch(dpart ? k_cell_apply<T, 3, true> : k_cell_apply<T, 3>);
  else launch(dpart ? k_cell_apply<T, 2, true> : k_cell_apply<T, 2>);
  FLGPU_HIP(hipGetLastError());
}

// ---- 3D order-2 lattice interpolation without its matrix -------------------------------------
// A coarse Q2 node j lies on the fine node 2j.  Per axis a fine node i takes, for even i, the
// coarse node i / 2 and, for odd i, the three nodes of its coarse cell i / 4 with the quadratic
// shape functions at 1/4 or 3/4: 3/8, 3/4, -1/8 or the reverse.  Transposed, a coarse vertex j
// (even) takes the fine nodes 2j - 3, 2j - 1, 2j, 2j + 1, 2j + 3 with -1/8, 3/8, 1, 3/8, -1/8 and a
// mid node 2j - 1, 2j, 2j + 1 with 3/4, 1, 3/4.  Rows and columns on the boundary are zero
// (constrained interpolation).  FP32 sums are formed in FP64, as the CSR products form them.
// Bound by the vectors' bytes and, for the restriction, by a vertex's 125 reads.  48^3 cells, FP32:
// 9.2 and 17.2 us; from the CSR 26.7 and 22.8, its 7.5 million entries.
__device__ __forceinline__ double q2_weight(int r, int t) {  // r = i mod 4 in {1, 3}, tap t of 3
  const double w[3] = {0.375, 0.75, -0.125};
  return t == 1 ? w[1] : (r == 1) == (t == 0) ? w[0] : w[2];
}

template <class T>
__global__ __launch_bounds__(256) void k_q2_prolong(int M, int Mc, FastDiv fM, T alpha,
                                                    const T *__restrict__ x, T beta, const T *z,
                                                    T *out) {
  const unsigned i = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (i >= (unsigned)M * (unsigned)M * (unsigned)M) return;
  int q[3];
  lat_decode(i, fM, q[0], q[1], q[2]);
  const T zi = beta == (T)0 ? (T)0 : z[i];
  // the taps of an axis: coarse nodes j0 + t with weights w[t]; 0 for those on the boundary
  int j0[3];
  double w[3][3];
  bool in = true;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const bool odd = q[a] & 1;
    j0[a] = odd ? 2 * (q[a] >> 2) : min(max((q[a] >> 1) - 1, 0), Mc - 3);
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const int j = j0[a] + t;
      const double v = odd ? q2_weight(q[a] & 3, t) : j == q[a] >> 1 ? 1.0 : 0.0;
      w[a][t] = j == 0 || j == Mc - 1 ? 0.0 : v;
    }
    in &= q[a] > 0 && q[a] < M - 1;
  }
  double s = 0;
  if (in)
#pragma unroll
    for (int tz = 0; tz < 3; tz++) {
      if (w[0][tz] == 0.0) continue;  // a plane's nodes alike
      T v[3][3];
#pragma unroll
      for (int ty = 0; ty < 3; ty++) {
        const T *p = x + ((unsigned)(j0[0] + tz) * (unsigned)Mc + (unsigned)(j0[1] + ty)) *
                             (unsigned)Mc + (unsigned)j0[2];
#pragma unroll
        for (int u = 0; u < 3; u++) v[ty][u] = p[u];
      }
#pragma unroll
      for (int ty = 0; ty < 3; ty++) {
        double line = 0;
#pragma unroll
        for (int u = 0; u < 3; u++)
          line += w[2][u] * (double)(w[1][ty] != 0.0 && w[2][u] != 0.0 ? v[ty][u] : (T)0);
        s += w[0][tz] * w[1][ty] * line;
      }
    }
  out[i] = (T)((double)beta * (double)zi + (double)alpha * s);
}

// tap t of 5 of the coarse coordinate q: its weight, 0 where there is none, and its fine coordinate
// f (2q where there is none)
__device__ __forceinline__ double q2_tap(int q, int t, int M, int &f) {
  const int d = t == 2 ? 0 : t < 2 ? 2 * t - 3 : 2 * t - 5;  // -3, -1, 0, 1, 3
  f = 2 * q + d;
  const bool near = t == 1 || t == 3, ok = f > 0 && f < M - 1 && t < 5;
  const double v = t == 2 ? 1.0 : q & 1 ? (near ? 0.75 : 0.0) : near ? 0.375 : -0.125;
  if (!ok) f = 2 * q;
  return ok ? v : 0.0;
}

// Eight lanes share a coarse row, each every eighth of its 25 lines of fine nodes: all of a lane's
// loads are in flight together (one lane a row: 11 us on small lattices too).
template <class T>
__global__ __launch_bounds__(256) void k_q2_restrict(int M, int Mc, FastDiv fMc, T alpha,
                                                     const T *__restrict__ x, T beta, const T *z,
                                                     T *out, T *zero) {
  const unsigned t0 = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const unsigned Nc = (unsigned)Mc * (unsigned)Mc * (unsigned)Mc;
  const unsigned c = min(t0 >> 3, Nc - 1);
  const int l = (int)(t0 & 7u);
  int q[3];
  lat_decode(c, fMc, q[0], q[1], q[2]);
  bool in = true;
#pragma unroll
  for (int a = 0; a < 3; a++) in &= q[a] > 0 && q[a] < Mc - 1;
  int fx[5];
  double wx[5];
#pragma unroll
  for (int u = 0; u < 5; u++) wx[u] = q2_tap(q[2], u, M, fx[u]);
  double w[4];
  T v[4][5];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int t = l + 8 * k, tz = (t * 13) >> 6;  // t / 5 for t < 32
    int fz, fy;
    w[k] = q2_tap(q[0], tz, M, fz) * q2_tap(q[1], t - 5 * tz, M, fy);
    const T *p = x + ((unsigned)fz * (unsigned)M + (unsigned)fy) * (unsigned)M;
#pragma unroll
    for (int u = 0; u < 5; u++) v[k][u] = p[fx[u]];
  }
  double s = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    double line = 0;
#pragma unroll
    for (int u = 0; u < 5; u++)
      line += wx[u] * (double)(w[k] != 0.0 && wx[u] != 0.0 ? v[k][u] : (T)0);
    s += w[k] * line;
  }
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (l != 0 || t0 >> 3 >= Nc) return;
  if (!in) s = 0;
  const T zi = beta == (T)0 ? (T)0 : z[c];
  out[c] = (T)((double)beta * (double)zi + (double)alpha * s);
  if (zero) zero[c] = (T)0;
}

template <class T>
static void launch_q2t(const flgpu_mat *A, T alpha, const void *x, T beta, const void *z,
                       void *out, void *zero = nullptr) {
  const int M = 4 * A->q2_nc + 1, Mc = 2 * A->q2_nc + 1;
  const unsigned g = xcd_grid(grid_for((long)A->nrows * (A->q2t == 1 ? 1 : 8), 256));
  if (A->q2t == 1)
    k_q2_prolong<T><<<g, 256, 0, A->ctx->stream>>>(M, Mc, fast_div((unsigned)M), alpha,
                                                   (const T *)x, beta, (const T *)z, (T *)out);
  else
    k_q2_restrict<T><<<g, 256, 0, A->ctx->stream>>>(M, Mc, fast_div((unsigned)Mc), alpha,
                                                    (const T *)x, beta, (const T *)z, (T *)out,
                                                    (T *)zero);
  FLGPU_HIP(hipGetLastError());
}

void spmv_zero(const flgpu_mat *A, const void *x, void *out, void *zero) {
  const bool f64 = A->prec == FLGPU_F64;
  if (A->q2t == 2) {
    if (f64) launch_q2t<double>(A, 1.0, x, 0.0, out, out, zero);
    else launch_q2t<float>(A, 1.0f, x, 0.0f, out, out, zero);
  } else if (!A->tp_kind && !A->alpha && !A->val27 && !A->cell && A->lanes) {
    if (f64) launch_csr_spmv<double>(A, 1.0, x, 0.0, out, out, nullptr, zero);
    else launch_csr_spmv<float>(A, 1.0f, x, 0.0f, out, out, nullptr, zero);
  } else {
    spmv(A, 1.0, x, 0.0, out, out);
    vfill(A->ctx, A->nrows, A->prec, zero, 0.0);
  }
}

void spmv(const flgpu_mat *A, double alpha, const void *x, double beta, const void *z,
          void *out) {
  if (A->q2t) {
    if (A->prec == FLGPU_F64) launch_q2t<double>(A, alpha, x, beta, z, out);
    else launch_q2t<float>(A, (float)alpha, x, (float)beta, z, out);
    return;
  }
  if (A->cell && A->lat_dim >= 2 && A->nrows >= kCellApplyRows) {
    if (A->prec == FLGPU_F64) launch_cell_apply<double>(A, alpha, x, beta, z, out);
    else launch_cell_apply<float>(A, (float)alpha, x, (float)beta, z, out);
    return;
  }
  if (A->tp_kind) {
    if (A->prec == FLGPU_F64) launch_tp<double>(A, alpha, x, beta, z, out);
    else launch_tp<float>(A, (float)alpha, x, (float)beta, z, out);
    return;
  }
  if (A->alpha) {
    if (A->prec == FLGPU_F64) launch_q1_pass<double, Q1_SPMV>(A, alpha, beta, z, x, out);
    else launch_q1_pass<float, Q1_SPMV>(A, (float)alpha, (float)beta, z, x, out);
    return;
  }
  if (A->val27) {
    if (A->prec == FLGPU_F64)
      launch_st27_spmv<double>(A, alpha, (const double *)x, beta, (const double *)z,
                               (double *)out);
    else
      launch_st27_spmv<float>(A, (float)alpha, (const float *)x, (float)beta, (const float *)z,
                              (float *)out);
    return;
  }
  if (A->lanes) {
    if (A->prec == FLGPU_F64) launch_csr_spmv<double>(A, alpha, x, beta, z, out);
    else launch_csr_spmv<float>(A, (float)alpha, x, (float)beta, z, out);
    return;
  }
  if (A->prec == FLGPU_F64) launch_spmv<double>(A->ctx, A->sell, alpha, x, beta, z, out);
  else launch_spmv<float>(A->ctx, A->sell, alpha, x, beta, z, out);
}

// blocks of a per-cell pass over A (launch_q1_pass's grid)
static long q1_blocks(const flgpu_mat *A, int qzb) {
  long M = A->lat_n + 1;
  long total = M * M * ((M + qzb - 1) / qzb);
  return (long)xcd_grid(grid_for((total + 61) / 62 * 64, 256));
}

template <class T>
static DotParts spmv_dot_t(const flgpu_mat *A, const void *x, void *out, int slot) {
  // the blocks of the form that spmv would take, 0: the dot is read from the vectors
  long nb = 0;
  unsigned by, bx;
  const bool cell = A->cell && A->lat_dim >= 2 && A->nrows >= kCellApplyRows;
  if (cell) nb = (long)xcd_grid(cell_boxes(A, by, bx));
  else if (A->tp_kind || A->q2t) nb = 0;
  else if (A->alpha) nb = q1_blocks(A, sizeof(T) == 8 ? FLGPU_QZB_F64_SPMV : FLGPU_QZB_F32);
  else if (A->val27) nb = (long)xcd_grid(grid_for(A->nrows, 256));
  else if (A->lanes) nb = (long)xcd_grid(grid_for((long)A->nrows * A->lanes, 256));
  else if (A->sell.nrows == A->nrows) nb = (long)xcd_grid(grid_for(A->sell.nslices, 4));
  // a CSR product with more blocks than the consumer adds up needs a launch for the sum as well,
  // and then a pass over the vectors costs no more: 300 007 rows 23 + 4.7 against 24 + 4.5 us
  if (!cell && A->lanes && nb > kPartsMax) nb = 0;
  if (nb == 0) {
    spmv(A, 1.0, x, 0.0, out, out);
    return dot_parts(A->ctx, A->nrows, A->prec, out, x);
  }
  flgpu_mat *M = const_cast<flgpu_mat *>(A);
  if (M->dot_np < nb) {
    dev_free(M->dot_part);
    M->dot_part = nullptr;
    M->dot_np = 0;
    M->dot_part = (double *)dev_alloc(sizeof(double) * nb);
    M->dot_np = nb;
  }
  double *dp = M->dot_part;
  if (cell) launch_cell_apply<T>(A, (T)1, x, (T)0, out, out, dp);
  else if (A->alpha) launch_q1_pass<T, Q1_SPMV>(A, (T)1, (T)0, out, x, out, nullptr, dp);
  else if (A->val27)
    launch_st27_spmv<T>(A, (T)1, (const T *)x, (T)0, (const T *)out, (T *)out, dp);
  else if (A->lanes) launch_csr_spmv<T>(A, (T)1, x, (T)0, out, out, dp);
  else launch_spmv<T>(A->ctx, A->sell, 1.0, x, 0.0, out, out, dp);
  return dot_parts_bound(A->ctx, dp, nb, slot);
}

DotParts spmv_dot(const flgpu_mat *A, const void *x, void *out, int slot) {
  return A->prec == FLGPU_F64 ? spmv_dot_t<double>(A, x, out, slot)
                              : spmv_dot_t<float>(A, x, out, slot);
}

void spmv_t(const flgpu_mat *A, double alpha, const void *x, double beta, void *out) {
  mat_build_transpose(A);
  spmv(A->transpose, alpha, x, beta, out, out);
}

template <class T>
__global__ void k_jacobi(int n, T damp, const T *__restrict__ diag, T *x, T *r) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T ri = r[i] / diag[i];
  r[i] = ri;
  x[i] += damp * ri;
}

// One <jacobi> step of a product-iterator (linit.lisp:94-120,220-250) with the residual it
// needs recomputed in the same pass, out of place: r_i = b_i - (A x)_i (the sum of spmv with
// alpha = -1, beta = 1), r_i /= A_ii, xo_i = x_i + damp r_i.  The per-cell form runs
// k_q1_zblock (A_ii from the cell factors); the stencil and SELL forms read A_ii from diag:
template <class T, bool SYM>
__global__ __launch_bounds__(256) void k_st27_jacobi(int M, const T *__restrict__ val27,
                                                     const T *__restrict__ diag, T damp,
                                                     const T *__restrict__ x,
                                                     const T *__restrict__ b, T *__restrict__ xo) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  long i = (long)lb * blockDim.x + threadIdx.x;
  long N = (long)M * M * M;
  if (i >= N) return;
  int xx = (int)(i % M), yy = (int)((i / M) % M), zz = (int)(i / ((long)M * M));
  T d;
  T acc = st27_row<T, SYM>(M, N, i, zz, yy, xx, val27, b[i], (T)-1, x, &d);
  xo[i] = x[i] + damp * (acc / diag[i]);
}

template <class T>
__global__ __launch_bounds__(256) void k_sell_jacobi(int nsub, int nslices,
                                                     const long *__restrict__ slice_ptr,
                                                     const int *__restrict__ col,
                                                     const T *__restrict__ val,
                                                     const T *__restrict__ diag, T damp,
                                                     const T *__restrict__ x,
                                                     const T *__restrict__ b, T *__restrict__ xo) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  int s = (int)lb * 4 + (threadIdx.x >> 6);
  if (s >= nslices) return;
  int lane = threadIdx.x & 63;
  int row = s * 64 + lane;
  long base = slice_ptr[s];
  int w = (int)((slice_ptr[s + 1] - base) >> 6);
  if (row >= nsub) return;
  T acc = sell_row<T>(val + base + lane, col + base + lane, w, (T)-1, x, b[row]);
  xo[row] = x[row] + damp * (acc / diag[row]);
}

// S <jacobi> steps of a small stencil-form level in one pass.  A block owns a region of R^3
// rows: a tile of TE^3 rows with a halo of S - 1 (R = TE + 2 (S - 1)).  x is staged in LDS over
// the region and one more layer; step s (0-based) updates the rows of the region shrunk by s,
// from the previous step's values in LDS, so the last step has exact values on the tile, which
// alone is stored.  Each row keeps its 27 coefficients in registers across the steps and is
// formed as k_st27_jacobi forms it (st27_row's order; a neighbour outside the lattice reads the
// row's own value against its zero coefficient).  All global loads of a thread are issued
// before its first LDS store.  Halo rows are recomputed by neighbouring blocks; this pays only
// where a level is small enough that a launch costs more than its work.
constexpr int MJ_MAXLOAD = 8;  // x values a thread stages: (R + 2)^3 <= MJ_MAXLOAD * block

template <class T, int S, bool SYM>
__global__ __launch_bounds__(1024) void k_st27_jacobi_multi(int M, int TE, const T *__restrict__ val27,
                                                           const T *__restrict__ diag, T damp,
                                                           const T *__restrict__ x,
                                                           const T *__restrict__ b,
                                                           T *__restrict__ xo) {
  extern __shared__ unsigned char mj_lds[];
  const int R = TE + 2 * (S - 1), L = R + 2, L3 = L * L * L;
  T *xs0 = (T *)mj_lds, *xs1 = xs0 + L3;
  const int nt = (M + TE - 1) / TE;
  const int tb = blockIdx.x;
  const int oz = (tb / (nt * nt)) * TE - (S - 1), oy = ((tb / nt) % nt) * TE - (S - 1),
            ox = (tb % nt) * TE - (S - 1);  // region origin
  const long M2 = (long)M * M, N = M2 * M;
  const int t = threadIdx.x;
  const int rz = t / (R * R), ry = (t / R) % R, rx = t % R;
  const int gz = oz + rz, gy = oy + ry, gx = ox + rx;
  const bool row = t < R * R * R && gz >= 0 && gz < M && gy >= 0 && gy < M && gx >= 0 && gx < M;
  const long i = row ? gz * M2 + (long)gy * M + gx : 0;
  const bool lz[3] = {gz > 0, true, gz < M - 1}, ly[3] = {gy > 0, true, gy < M - 1},
             lx[3] = {gx > 0, true, gx < M - 1};
  T av[27], bi = (T)0, di = (T)1;
  if (row) {
#pragma unroll
    for (int k = 0; k < 27; k++) {
      int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
      av[k] = st27_coef<T, SYM>(val27, N, k, i, dz * M2 + dy * M + dx,
                                lz[dz + 1] && ly[dy + 1] && lx[dx + 1]);
    }
    bi = b[i];
    di = diag[i];
  }
  // x over the region and one more layer (lattice values only; the rest is never read)
  T xl[MJ_MAXLOAD];
#pragma unroll
  for (int j = 0; j < MJ_MAXLOAD; j++) {
    const int k = t + j * blockDim.x;
    const int gz2 = oz - 1 + k / (L * L), gy2 = oy - 1 + (k / L) % L, gx2 = ox - 1 + k % L;
    const bool in = k < L3 && gz2 >= 0 && gz2 < M && gy2 >= 0 && gy2 < M && gx2 >= 0 && gx2 < M;
    xl[j] = in ? x[gz2 * M2 + (long)gy2 * M + gx2] : (T)0;
  }
#pragma unroll
  for (int j = 0; j < MJ_MAXLOAD; j++) {
    const int k = t + j * blockDim.x;
    if (k < L3) xs0[k] = xl[j];
  }
  const int own = ((rz + 1) * L + (ry + 1)) * L + (rx + 1);
  __syncthreads();
#pragma unroll
  for (int st = 0; st < S; st++) {
    const T *cur = (st & 1) ? xs1 : xs0;
    T *nxt = (st & 1) ? xs0 : xs1;
    const bool act = row && rz >= st && rz < R - st && ry >= st && ry < R - st && rx >= st &&
                     rx < R - st;
    if (act) {
      T acc = bi;
#pragma unroll
      for (int k = 0; k < 27; k++) {
        int dz = k / 9 - 1, dy = (k / 3) % 3 - 1, dx = k % 3 - 1;
        bool live = lz[dz + 1] && ly[dy + 1] && lx[dx + 1];
        T xn = cur[live ? own + (dz * L + dy) * L + dx : own];
        acc += ((T)-1 * xn) * av[k];
      }
      T xn = cur[own] + damp * (acc / di);
      if (st == S - 1) xo[i] = xn;  // the tile (the region shrunk by S - 1)
      else nxt[own] = xn;
    }
    if (st < S - 1) __syncthreads();
  }
}

// tile edge of a multi-step pass over a lattice of size M: about 200 blocks, a region of at
// most 1024 rows and an x box a block can stage; 0 when S steps do not fit
static int mj_tile(int M, int S) {
  int te = std::max(2, (M + 5) / 6);
  for (; te >= 2; te--) {
    int R = te + 2 * (S - 1), L = R + 2;
    int threads = (R * R * R + 63) / 64 * 64;
    if (threads <= 1024 && L * L * L <= MJ_MAXLOAD * threads) return te;
  }
  return 0;
}

template <class T>
static void launch_jacobi_multi(const flgpu_mat *A, int S, int te, T damp, const T *x,
                                const T *b, T *xo) {
  const int M = A->lat_n + 1;
  const int nt = (M + te - 1) / te, R = te + 2 * (S - 1), L = R + 2;
  const unsigned g = (unsigned)nt * nt * nt;
  const unsigned threads = (R * R * R + 63) / 64 * 64;
  const size_t lds = 2 * sizeof(T) * (size_t)L * L * L;
  hipStream_t st = A->ctx->stream;
  const T *v = (const T *)A->val27, *d = (const T *)A->diag;
  FLGPU_REQUIRE(S >= 2 && S <= 4, "2 to 4 steps per pass");
  if (A->st_sym) {
    if (S == 2) k_st27_jacobi_multi<T, 2, true><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
    if (S == 3) k_st27_jacobi_multi<T, 3, true><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
    if (S == 4) k_st27_jacobi_multi<T, 4, true><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
  } else {
    if (S == 2) k_st27_jacobi_multi<T, 2, false><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
    if (S == 3) k_st27_jacobi_multi<T, 3, false><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
    if (S == 4) k_st27_jacobi_multi<T, 4, false><<<g, threads, lds, st>>>(M, te, v, d, damp, x, b, xo);
  }
  FLGPU_HIP(hipGetLastError());
}

// stencil-form levels up to this lattice size take several <jacobi> steps per launch
// (measured, FP32: 17^3 lattice, 3 steps 7.7 us against 3 x 3.7 us; 33^3, 3 steps 13.6 us
// against 3 x 3.85 us, where the recomputed halos cost more than the launches)
#ifndef FLGPU_MULTI_MAX_M
#define FLGPU_MULTI_MAX_M 20
#endif

template <class T>
static void jacobi_step(const flgpu_mat *A, T damp, const T *x, const T *b, T *xo) {
  hipStream_t st = A->ctx->stream;
  if (A->alpha) {
    launch_q1_pass<T, Q1_JACOBI>(A, damp, (T)0, b, x, xo);
    return;
  } else if (A->val27) {
    unsigned g = xcd_grid(grid_for(A->nrows, 256));
    if (A->st_sym)
      k_st27_jacobi<T, true><<<g, 256, 0, st>>>(A->lat_n + 1, (const T *)A->val27,
                                                (const T *)A->diag, damp, x, b, xo);
    else
      k_st27_jacobi<T, false><<<g, 256, 0, st>>>(A->lat_n + 1, (const T *)A->val27,
                                                 (const T *)A->diag, damp, x, b, xo);
  } else {
    const Sell &s = A->sell;
    if (s.nrows == 0) return;
    unsigned g = xcd_grid(grid_for(s.nslices, 4));
    k_sell_jacobi<T><<<g, 256, 0, st>>>(s.nrows, s.nslices, s.slice_ptr, s.col, (const T *)s.val,
                                        (const T *)A->diag, damp, x, b, xo);
  }
  FLGPU_HIP(hipGetLastError());
}

// the first step from x = 0: b - A 0 = b exactly, so xo = damp b / A_ii without reading A
template <class T>
__global__ void k_jacobi_zero(long n, const T *__restrict__ diag, T damp, const T *__restrict__ b,
                              T *__restrict__ xo) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xo[i] = damp * (b[i] / diag[i]);
}

// `steps` <jacobi> steps, each from a freshly computed residual, x ping-ponged through tmp
// (n values); the residual vector of the iteration is not touched (left stale).  x_zero:
// x holds no values yet and stands for zero.  done = 1: the first step from zero has been
// taken already and its result is in tmp.
bool jacobi_steps(const flgpu_mat *A, double damp, int steps, void *x, const void *b, void *tmp,
                  bool x_zero, int done, double *x64) {
  if (steps <= 0 || A->nrows == 0) return false;
  FLGPU_REQUIRE(A->nrows == A->ncols, "<jacobi> needs a square matrix");
  FLGPU_REQUIRE(done == 0 || (done == 1 && x_zero), "only the first step from zero comes done");
  // x64: the last step also stores x in FP64 when it is a per-cell FP32 pass that ends in x
  const bool w2 = x64 && A->alpha && A->prec == FLGPU_F32 && steps % 2 == 0 && steps - 1 >= done;
  // small stencil-form levels: several steps per launch (each launch writes the buffer it
  // does not read, so the remaining steps are split to end in x)
  const bool multi = A->val27 && !A->alpha && A->lat_n + 1 <= FLGPU_MULTI_MAX_M;
  void *cur = done ? tmp : x;  // where the iterate is (x stands for zero when x_zero, !done)
  int k = done;
  while (k < steps) {
    void *dst = (cur == x) ? tmp : x;
    const int rem = steps - k;
    if (k == 0 && x_zero) {
      unsigned g = grid_for(A->nrows, 256);
      if (A->prec == FLGPU_F64)
        k_jacobi_zero<double><<<g, 256, 0, A->ctx->stream>>>(
            A->nrows, (const double *)A->diag, damp, (const double *)b, (double *)dst);
      else
        k_jacobi_zero<float><<<g, 256, 0, A->ctx->stream>>>(
            A->nrows, (const float *)A->diag, (float)damp, (const float *)b, (float *)dst);
      FLGPU_HIP(hipGetLastError());
      k++;
    } else if (multi && rem >= 2) {
      // from tmp one launch lands in x; from x two are needed
      int S = (cur == tmp) ? rem : rem - rem / 2;
      S = S < 4 ? S : 4;
      int te = 0;
      while (S >= 2 && (te = mj_tile(A->lat_n + 1, S)) == 0) S--;
      if (S >= 2) {
        if (A->prec == FLGPU_F64)
          launch_jacobi_multi<double>(A, S, te, damp, (const double *)cur, (const double *)b,
                                      (double *)dst);
        else
          launch_jacobi_multi<float>(A, S, te, (float)damp, (const float *)cur,
                                     (const float *)b, (float *)dst);
      } else {
        S = 1;
        if (A->prec == FLGPU_F64)
          jacobi_step<double>(A, damp, (const double *)cur, (const double *)b, (double *)dst);
        else
          jacobi_step<float>(A, (float)damp, (const float *)cur, (const float *)b, (float *)dst);
      }
      k += S;
    } else if (w2 && k == steps - 1) {
      launch_q1_pass<float, Q1_JACOBI>(A, (float)damp, 0.0f, b, cur, dst, x64);
      k++;
    } else {
      if (A->prec == FLGPU_F64)
        jacobi_step<double>(A, damp, (const double *)cur, (const double *)b, (double *)dst);
      else
        jacobi_step<float>(A, (float)damp, (const float *)cur, (const float *)b, (float *)dst);
      k++;
    }
    cur = dst;
  }
  if (cur != x) vcopy(A->ctx, A->nrows, A->prec, cur, A->prec, x);
  return w2 && cur == x;
}

void jacobi_iterate(const flgpu_mat *A, double damp, void *x, void *r) {
  int n = A->nrows;
  if (n == 0) return;
  if (A->prec == FLGPU_F64)
    k_jacobi<double><<<grid_for(n, 256), 256, 0, A->ctx->stream>>>(
        n, damp, (const double *)A->diag, (double *)x, (double *)r);
  else
    k_jacobi<float><<<grid_for(n, 256), 256, 0, A->ctx->stream>>>(
        n, (float)damp, (const float *)A->diag, (float *)x, (float *)r);
  FLGPU_HIP(hipGetLastError());
}

// One colour of a <sor> sweep: rows of one colour do not couple, so the
// sequential sweep over them equals this parallel update.
template <class T>
__global__ __launch_bounds__(256) void k_sor_colour(int nsub, int nslices, const int *__restrict__ rows,
                                                    const long *__restrict__ slice_ptr,
                                                    const int *__restrict__ col,
                                                    const T *__restrict__ val,
                                                    const T *__restrict__ diag, T omega, T *x,
                                                    const T *b, T *r) {
  unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  int s = (int)lb * 4 + (threadIdx.x >> 6);
  if (s >= nslices) return;
  int lane = threadIdx.x & 63;
  int li = s * 64 + lane;
  long base = slice_ptr[s];
  int w = (int)((slice_ptr[s + 1] - base) >> 6);
  if (li >= nsub) return;
  int row = rows[li];
  T corr = sell_row<T>(val + base + lane, col + base + lane, w, (T)-1, x, b[row]);
  corr = corr / diag[row];
  r[row] = corr;
  x[row] += omega * corr;
}

// The same from the CSR rows, eight lanes per row.  A colour's rows are few, so the length of a
// row's chain of loads sets the time: 60 001 rows of 12 entries in nine colours, FP32: 3.1 us per
// colour, 8.1 us from SELL.
template <class T>
__global__ __launch_bounds__(256) void k_sor_colour_csr(int nsub, const int *__restrict__ rows,
                                                        const int2 *__restrict__ span,
                                                        const int *__restrict__ col,
                                                        const T *__restrict__ val,
                                                        const T *__restrict__ diag, T omega, T *x,
                                                        const T *b, T *r) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int li = (int)lb * 32 + threadIdx.x / 8, l = threadIdx.x % 8;
  if (li >= nsub) return;  // the lanes of a row leave together
  const int row = rows[li];
  const int2 be = span[li];
  const T bi = b[row], di = diag[row], xi = x[row];
  T corr = (T)((double)bi + csr_row<T, 8>(col, val, be.x, be.y, l, (T)-1, x));
  corr = corr / di;
  if (l == 0) {
    r[row] = corr;
    x[row] = xi + omega * corr;
  }
}

// the CSR bounds of a colour's rows
__global__ void k_row_span(int nsub, const int *__restrict__ rows, const int *__restrict__ rowptr,
                           int2 *__restrict__ span) {
  const int li = blockIdx.x * blockDim.x + threadIdx.x;
  if (li < nsub) span[li] = make_int2(rowptr[rows[li]], rowptr[rows[li] + 1]);
}

// lines of a block of k_q1_sor_planes
constexpr int kSorLines = 8;
// lattices of at most 65^3 nodes sweep out of place where a spare vector is there: a launch costs
// 2.3 us at least, so two of 3.8 us beat four at 17^3 and 33^3 (7.6 against 11 us FP64), they are
// equal at 65^3, and at 129^3 the halo lines and LDS cost more than the launches (33 against 29)
constexpr int kSorOutplaceM = 65;

bool sor_outplace(const flgpu_mat *A) { return A->alpha && A->lat_n < kSorOutplaceM; }

template <class T>
static Q1KT<T> q1kt(const flgpu_mat *A) {
  Q1KT<T> k;
  for (int j = 0; j < 8; j++) k.k[j] = (T)A->kt[j];
  return k;
}

// a sweep in place, four launches
template <class T>
static void q1_sor_inplace(const flgpu_mat *A, T omega, int backwards, T *x, const T *b, T *r,
                           bool zero) {
  const int M = A->lat_n + 1;
  const Q1KT<T> kt = q1kt<T>(A);
  for (int k = 0; k < 4; k++) {
    const int cz = backwards ? 1 - (k >> 1) : k >> 1, cy = backwards ? 1 - (k & 1) : k & 1;
    const int nzl = (M - cz + 1) / 2, nyl = (M - cy + 1) / 2;
    const unsigned total = (unsigned)nzl * (unsigned)nyl * (unsigned)M;
    const unsigned g = xcd_grid((total + 4 * 62 - 1) / (4 * 62));
    auto launch = [&](auto kern) {
      kern<<<g, 256, 0, A->ctx->stream>>>(M, A->lat_n, cz, cy, nyl, total, fast_div((unsigned)M),
                                          div1((unsigned)nyl), (const T *)A->alpha, kt, omega, x,
                                          b, r);
      FLGPU_HIP(hipGetLastError());
    };
    if (!zero) launch(k_q1_sor_lines<T, false, false, false>);
    else if (k == 0) launch(k_q1_sor_lines<T, true, true, true>);
    else if (k == 1) launch(k_q1_sor_lines<T, true, false, true>);
    else if (k == 2) launch(k_q1_sor_lines<T, false, true, true>);
    else launch(k_q1_sor_lines<T, false, false, true>);
  }
}

// a sweep from xs into xd, two launches
template <class T>
static void q1_sor_outplace(const flgpu_mat *A, T omega, int backwards, const T *xs, T *xd,
                            const T *b, T *r, bool zero) {
  const int M = A->lat_n + 1, H = kSorLines, S = (M + H - 1) / H;
  const Q1KT<T> kt = q1kt<T>(A);
  const size_t lds = sizeof(T) * (size_t)(H / 2 + 1) * M;
  for (int k = 0; k < 2; k++) {
    const int pz = backwards ? 1 - k : k, planes = (M - 1 - pz) / 2 + 1;
    const unsigned g = xcd_grid((unsigned)planes * (unsigned)S);
    auto launch = [&](auto kern) {
      kern<<<g, 256, lds, A->ctx->stream>>>(M, A->lat_n, pz, backwards ? 1 : 0, H, S, planes,
                                            fast_div((unsigned)M), (const T *)A->alpha, kt,
                                            omega, xs, k == 0 ? xs : xd, xd, b, r);
      FLGPU_HIP(hipGetLastError());
    };
    if (!zero) launch(k_q1_sor_planes<T, false, false>);
    else if (k == 0) launch(k_q1_sor_planes<T, true, true>);
    else launch(k_q1_sor_planes<T, false, true>);
  }
}

// `steps` sweeps of the per-cell form; true when r holds the residual (rmode 2)
template <class T>
static bool q1_sor(const flgpu_mat *A, T omega, int steps, int backwards, T *x, const T *b, T *r,
                   T *tmp, bool zero, int rmode) {
  const int M = A->lat_n + 1;
  if (b == r) rmode = 1;
  if (M <= 10) {
    const int per = b == r ? 1 : steps;  // each sweep reads the last one's r
    for (int k = 0; k < steps; k += per, zero = false) {
      k_q1_sor_small<T><<<1, 1024, 0, A->ctx->stream>>>(M, A->lat_n, per, backwards, rmode, zero,
                                                        (const T *)A->alpha, q1kt<T>(A), omega,
                                                        x, b, r);
      FLGPU_HIP(hipGetLastError());
    }
    return rmode == 2;
  }
  int k = 0;
  if (tmp && b != r && sor_outplace(A))
    for (; k + 2 <= steps; k += 2, zero = false) {
      q1_sor_outplace<T>(A, omega, backwards, x, tmp, b, nullptr, zero);
      q1_sor_outplace<T>(A, omega, backwards, tmp, x, b, k + 2 == steps && rmode == 1 ? r : nullptr,
                         false);
    }
  for (; k < steps; k++, zero = false)
    q1_sor_inplace<T>(A, omega, backwards, x, b,
                      b == r || (k + 1 == steps && rmode == 1) ? r : nullptr, zero);
  return false;
}

// A sweep of the stencil form from xs into xd.  Small lattices leave the GPU idle and wait for
// one row's loads: one row a thread.  On larger ones taller tiles recompute less (1.45 times the
// rows with 8 lines, 1.3 with 12, 1.25 with 16, 1.2 with 20).  Measured, us an iterate, 8 lines
// and 1 row a thread / 12 and 2 / 20 and 4: 49^3 FP64 16.0 / 18.7 / 24.9; 65^3 28.6 / 24.2 / 33.8;
// 129^3 158 / 151 / 165, FP32 114 / 86 / 91.  Above, 12 and 2 / 16 and 2 / 20 and 4, FP64: 137^3
// 223 / 204 / 198, 153^3 313 / 296 / 310, 177^3 457 / 464 / 467, 201^3 699 / 654 / 700; FP32, where
// the last tile's idle lines decide, 12 and 2 / 16 and 4 / 20 and 4: 137^3 108 / 106 / 100, 153^3
// 153 / 148 / 153, 177^3 258 / 259 / 253, 185^3 299 / 286 / 295, 193^3 340 / 335 / 327, 201^3 405 /
// 386 / 399.
template <class T>
static void st27_sor(const flgpu_mat *A, T omega, int backwards, const T *xs, T *xd, const T *b,
                     T *r, bool zero) {
  const int M = A->lat_n + 1;
  const int ntx = (M + kTileCols - 1) / kTileCols, W = (M + ntx - 1) / ntx;
  for (int k = 0; k < 2; k++) {
    const int pz = backwards ? 1 - k : k, planes = (M - 1 - pz) / 2 + 1;
    auto launch = [&](auto sym, auto lines, auto grp) {
      constexpr bool SYM = decltype(sym)::value;
      constexpr int H = decltype(lines)::value, G = decltype(grp)::value;
      constexpr int threads = (kTileRows(H) + 63) / 64 * 64 * G;
      const int nty = (M + H - 1) / H;
      const unsigned g = xcd_grid((unsigned)planes * (unsigned)(ntx * nty));
      auto run = [&](auto kern) {
        kern<<<g, threads, 0, A->ctx->stream>>>(M, pz, W, ntx, nty, planes, backwards,
                                                (const T *)A->val27, omega, xs,
                                                k == 0 ? xs : xd, xd, b, r);
        FLGPU_HIP(hipGetLastError());
      };
      if (!zero) run(k_st27_sor_tiles<T, SYM, false, false, H, G>);
      else if (k == 0) run(k_st27_sor_tiles<T, SYM, true, true, H, G>);
      else run(k_st27_sor_tiles<T, SYM, false, true, H, G>);
    };
    auto shape = [&](auto sym) {
      using std::integral_constant;
      constexpr int G = sizeof(T) == 8 ? 2 : 1;
      auto idle = [&](int H) { return (M + H - 1) / H * H - M; };
      if (M <= 56) launch(sym, integral_constant<int, 8>(), integral_constant<int, 4>());
      else if (M <= 132) launch(sym, integral_constant<int, 12>(), integral_constant<int, 2>());
      else if (G == 2 || idle(16) <= idle(20))
        launch(sym, integral_constant<int, 16>(), integral_constant<int, G>());
      else launch(sym, integral_constant<int, 20>(), integral_constant<int, 1>());
    };
    if (A->st_sym) shape(std::true_type());
    else shape(std::false_type());
  }
}

template <class T>
static void st27_sor_sweeps(const flgpu_mat *A, T omega, int steps, int backwards, T *x,
                            const T *b, T *r, bool zero, int rmode) {
  FLGPU_REQUIRE(A->sor_work, "stencil <sor> sweeps need sor_prepare");
  const long N = A->nrows;
  T *w = (T *)A->sor_work, *cur = x, *other = w;
  for (int k = 0; k < steps; k++, zero = false) {
    const T *bk = b;
    if (b == r) {  // the sweep reads b beyond the rows whose r it writes
      vcopy(A->ctx, N, A->prec, b, A->prec, w + N);
      bk = w + N;
    }
    const bool wr = b == r || (rmode == 1 && k + 1 == steps);
    st27_sor<T>(A, omega, backwards, cur, other, bk, wr ? r : nullptr, zero);
    std::swap(cur, other);
  }
  if (cur != x) vcopy(A->ctx, N, A->prec, cur, A->prec, x);
}

void sor_prepare(const flgpu_mat *A) {
  if (A->alpha || !A->val27 || A->sor_work) return;
  const_cast<flgpu_mat *>(A)->sor_work = dev_alloc(prec_bytes(A->prec) * 2 * (size_t)A->nrows);
}

static void sor_sweep(const flgpu_mat *A, double omega, int backwards, void *x, const void *b,
                      void *r) {
  FLGPU_REQUIRE(A->ncolours > 0, "<sor> needs a colouring of the matrix");
  for (int k = 0; k < A->ncolours; k++) {
    const Sell &s = A->colour_sell[backwards ? A->ncolours - 1 - k : k];
    if (s.nrows == 0) continue;
    if (s.span) {
      const unsigned gc = xcd_grid(grid_for(s.nrows, 32));
      if (A->prec == FLGPU_F64)
        k_sor_colour_csr<double><<<gc, 256, 0, A->ctx->stream>>>(
            s.nrows, s.rows, (const int2 *)s.span, A->colidx, (const double *)A->vals,
            (const double *)A->diag, omega, (double *)x, (const double *)b, (double *)r);
      else
        k_sor_colour_csr<float><<<gc, 256, 0, A->ctx->stream>>>(
            s.nrows, s.rows, (const int2 *)s.span, A->colidx, (const float *)A->vals,
            (const float *)A->diag, (float)omega, (float *)x, (const float *)b, (float *)r);
      FLGPU_HIP(hipGetLastError());
      continue;
    }
    unsigned g = xcd_grid(grid_for(s.nslices, 4));
    if (A->prec == FLGPU_F64)
      k_sor_colour<double><<<g, 256, 0, A->ctx->stream>>>(
          s.nrows, s.nslices, s.rows, s.slice_ptr, s.col, (const double *)s.val,
          (const double *)A->diag, omega, (double *)x, (const double *)b, (double *)r);
    else
      k_sor_colour<float><<<g, 256, 0, A->ctx->stream>>>(
          s.nrows, s.nslices, s.rows, s.slice_ptr, s.col, (const float *)s.val,
          (const float *)A->diag, (float)omega, (float *)x, (const float *)b, (float *)r);
    FLGPU_HIP(hipGetLastError());
  }
}

// `steps` <sor> sweeps (the product-iterator of a smoother, linit.lisp:94-120)
bool sor_sweeps(const flgpu_mat *A, double omega, int steps, int backwards, void *x, const void *b,
                void *r, void *tmp, bool x_zero, int rmode) {
  if (A->alpha) {
    if (A->prec == FLGPU_F64)
      return q1_sor<double>(A, omega, steps, backwards, (double *)x, (const double *)b,
                            (double *)r, (double *)tmp, x_zero, rmode);
    return q1_sor<float>(A, (float)omega, steps, backwards, (float *)x, (const float *)b,
                         (float *)r, (float *)tmp, x_zero, rmode);
  }
  if (A->val27) {
    if (A->prec == FLGPU_F64)
      st27_sor_sweeps<double>(A, omega, steps, backwards, (double *)x, (const double *)b,
                              (double *)r, x_zero, rmode);
    else
      st27_sor_sweeps<float>(A, (float)omega, steps, backwards, (float *)x, (const float *)b,
                             (float *)r, x_zero, rmode);
    return false;
  }
  if (x_zero) vfill(A->ctx, A->nrows, A->prec, x, 0.0);
  for (int k = 0; k < steps; k++) sor_sweep(A, omega, backwards, x, b, r);
  return false;
}

// ---- Galerkin product P^T A P (src/iteration/amg.lisp:247-280) ---------------------

// One thread per coarse row k: for fine l in column k of P (row k of P^T,
// ascending), entries A_lm of row l, and P's row m: acc[k][n] += (P_lk A_lm)
// P_mn, accumulated in FP64 into the caller's coarse pattern.  For a fixed
// coarse entry the contributions arrive in (l, m) order, as in femlisp's
// loop nest.  A product entry outside the pattern sets *bad.
template <class T>
__global__ void k_rap(int nc, const int *__restrict__ ptrp, const int *__restrict__ ptci,
                      const T *__restrict__ ptv, const int *__restrict__ arp,
                      const int *__restrict__ aci, const T *__restrict__ av,
                      const int *__restrict__ prp, const int *__restrict__ pci,
                      const T *__restrict__ pv, const int *__restrict__ crp,
                      const int *__restrict__ cci, double *acc, int *bad, int upper) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nc) return;
  int c0 = crp[k], c1 = crp[k + 1];
  for (int e = c0; e < c1; e++) acc[e] = 0.0;
  for (int a = ptrp[k]; a < ptrp[k + 1]; a++) {
    int l = ptci[a];
    double plk = (double)ptv[a];
    for (int b = arp[l]; b < arp[l + 1]; b++) {
      int m = aci[b];
      double w = plk * (double)av[b];
      for (int c = prp[m]; c < prp[m + 1]; c++) {
        int n = pci[c];
        if (upper && n < k) continue;  // the lower triangle is mirrored afterwards
        int lo = c0, hi = c1 - 1;
        while (lo < hi) {
          int mid = (lo + hi) >> 1;
          if (cci[mid] < n) lo = mid + 1;
          else hi = mid;
        }
        if (lo >= c1 || cci[lo] != n) {
          *bad = 1;
          continue;
        }
        acc[lo] += w * (double)pv[c];
      }
    }
  }
}

// The same with the coarse row's columns and accumulators in LDS (coarse rows of at most
// kRapW entries): the column searches and the FP64 sums stay on the CU instead of reaching
// device memory for every contribution.  Same loops, same order, same results.
constexpr int kRapW = 27, kRapB = 128;

template <class T>
__global__ __launch_bounds__(kRapB) void k_rap_lds(
    int nc, const int *__restrict__ ptrp, const int *__restrict__ ptci, const T *__restrict__ ptv,
    const int *__restrict__ arp, const int *__restrict__ aci, const T *__restrict__ av,
    const int *__restrict__ prp, const int *__restrict__ pci, const T *__restrict__ pv,
    const int *__restrict__ crp, const int *__restrict__ cci, double *acc, int *bad, int upper) {
  __shared__ double sacc[kRapW * kRapB];  // entry j of this thread's row at j * kRapB + tid
  __shared__ int scol[kRapW * kRapB];
  const int tid = threadIdx.x;
  const int k = blockIdx.x * kRapB + tid;
  if (k >= nc) return;
  const int c0 = crp[k], w = crp[k + 1] - c0;
  for (int j = 0; j < w; j++) {
    scol[j * kRapB + tid] = cci[c0 + j];
    sacc[j * kRapB + tid] = 0.0;
  }
  for (int a = ptrp[k]; a < ptrp[k + 1]; a++) {
    const int l = ptci[a];
    const double plk = (double)ptv[a];
    for (int b = arp[l]; b < arp[l + 1]; b++) {
      const int m = aci[b];
      const double wv = plk * (double)av[b];
      for (int c = prp[m]; c < prp[m + 1]; c++) {
        const int n = pci[c];
        if (upper && n < k) continue;  // the lower triangle is mirrored afterwards
        int lo = 0, hi = w - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (scol[mid * kRapB + tid] < n) lo = mid + 1;
          else hi = mid;
        }
        if (lo >= w || scol[lo * kRapB + tid] != n) {
          *bad = 1;
          continue;
        }
        sacc[lo * kRapB + tid] += wv * (double)pv[c];
      }
    }
  }
  for (int j = 0; j < w; j++) acc[c0 + j] = sacc[j * kRapB + tid];
}

// the contributions of one l (offset LE of the 27), entry by entry of A's row: which of its
// entries, which entry c of the coarse row, which plane of t27
struct RapList {
  int n = 0;
  signed char e[125] = {}, d[125] = {}, p[125] = {};
};
// The coarse entries (k, n), n >= k, are shared out to three threads of 343 to 486 contributions:
// the diagonal, the faces' and the edges' and corners' neighbours
constexpr int rap_group(int d) {
  const int far = (d / 9 != 1) + ((d / 3) % 3 != 1) + (d % 3 != 1);
  return far < 2 ? far : 2;
}
constexpr RapList rap_list(int le, int g) {
  RapList q;
  const int L[3] = {le / 9 - 1, (le / 3) % 3 - 1, le % 3 - 1};
  for (int e = 0; e < 27; e++) {
    const int E[3] = {e / 9 - 1, (e / 3) % 3 - 1, e % 3 - 1};
    for (int d = 13; d < 27; d++) {
      if (rap_group(d) != g) continue;
      const int D[3] = {d / 9 - 1, (d / 3) % 3 - 1, d % 3 - 1};
      bool near = true;
      int plane = 0;
      for (int a = 0; a < 3; a++) {
        const int o = L[a] + E[a] - 2 * D[a];
        near = near && o >= -1 && o <= 1;
        plane = plane * 3 + o + 1;
      }
      if (!near) continue;
      q.e[q.n] = (signed char)e;
      q.d[q.n] = (signed char)d;
      q.p[q.n] = (signed char)plane;
      q.n++;
    }
  }
  return q;
}

// l = 2k + offset LE: its loads, then its contributions in order
template <class T, int G, int LE, int... C>
__device__ __forceinline__ void rap_step(int M, const int (&K)[3], unsigned k, unsigned i0,
                                         size_t N, unsigned Nc, const T *a27, const T *t27,
                                         const unsigned (&nn)[27], double (&s)[27],
                                         std::integer_sequence<int, C...>) {
  if constexpr (sizeof...(C) == 0) return;  // l reaches none of the group's entries
  else {
    constexpr RapList Q = rap_list(LE, G);
    constexpr int L[3] = {LE / 9 - 1, (LE / 3) % 3 - 1, LE % 3 - 1};
    bool in = true;
#pragma unroll
    for (int a = 0; a < 3; a++) in &= 2 * K[a] + L[a] >= 0 && 2 * K[a] + L[a] < M;
    const unsigned l = in ? i0 + (unsigned)((L[0] * M + L[1]) * M + L[2]) : i0;
    asm volatile("" ::: "memory");  // P's values are loaded for every l: kept, they'd spill
    const double plk = in ? (double)t27[(size_t)LE * Nc + k] : 0.0;
    T av[27];
#pragma unroll
    for (int e = 0; e < 27; e++) av[e] = a27[(size_t)e * N + l];
    T pv[sizeof...(C)];
    ((pv[C] = t27[(size_t)Q.p[C] * Nc + nn[(int)Q.d[C]]]), ...);
    asm volatile("" ::: "memory");
    ((s[(int)Q.d[C]] += (plk * (double)av[(int)Q.e[C]]) * (double)pv[C]), ...);
    // the sums stay here: sunk to the stores, which are conditional, they'd keep every load alive
#pragma unroll
    for (int d = 13; d < 27; d++)
      if (rap_group(d) == G) asm volatile("" : "+v"(s[d]));
  }
}

// The same product on 3D Q1 lattices, a few threads per coarse node k: the fine matrix holds the
// lattice pattern and its values as 27 planes (a27), P the pattern of the lattice interpolation
// (fine node m takes the coarse nodes floor(m / 2) and ceil(m / 2) per axis) and its transpose's
// values as 27 planes (t27: plane of offset e holds P(2c + e, c)), the coarse matrix the coarse
// lattice pattern.  With l = 2k + a, m = l + b and n = k + c every offset is a constant of the
// unrolled loops, so a contribution (P_lk A_lm) P_mn is two multiplications and its loads, which
// neighbouring threads make side by side.  An entry sums its contributions in ascending l, then
// m: the order that k_rap's loops bring them in, so the sums are equal bit for bit.  A and P are 0
// where l or m is outside the lattice.  A is exactly symmetric: only entries n >= k are formed, and
// written to (n, k) too.  Bound by the loads of P's values, one per contribution (1270 a row), and
// the conversions to FP64; on small lattices by the 27 l's load latencies.  49^3 coarse nodes, FP32
// 257 us, 7^3 21: a thread per entry that computed every position, the mirrored triangle and the
// values took three launches, 1168 + 79 + 13 and 78 + 9 + 2.
template <class T, int G, int... LE>
__device__ __forceinline__ void rap_row(int Mc, unsigned k, const int (&K)[3], const T *a27,
                                        const T *t27, const int *__restrict__ crp, T *cv,
                                        std::integer_sequence<int, LE...>) {
  const int M = 2 * Mc - 1;
  const unsigned Nc = (unsigned)Mc * (unsigned)Mc * (unsigned)Mc;
  const size_t N = (size_t)M * M * M;
  const unsigned i0 = ((unsigned)(2 * K[0]) * (unsigned)M + (unsigned)(2 * K[1])) * (unsigned)M +
                      (unsigned)(2 * K[2]);
  unsigned nn[27];  // the coarse neighbours, k itself for those outside
#pragma unroll
  for (int d = 0; d < 27; d++) {
    const int D[3] = {d / 9 - 1, (d / 3) % 3 - 1, d % 3 - 1};
    bool in = true;
#pragma unroll
    for (int a = 0; a < 3; a++) in &= K[a] + D[a] >= 0 && K[a] + D[a] < Mc;
    nn[d] = in ? k + (unsigned)((D[0] * Mc + D[1]) * Mc + D[2]) : k;
  }
  double s[27] = {};
  (rap_step<T, G, LE>(M, K, k, i0, N, Nc, a27, t27, nn, s,
                          std::make_integer_sequence<int, rap_list(LE, G).n>()),
   ...);
  // a coarse row's entries: the neighbours within the lattice, ascending
  int cnt[3], lo[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    lo[a] = K[a] > 0 ? -1 : 0;
    cnt[a] = (K[a] < Mc - 1 ? 1 : 0) - lo[a] + 1;
  }
  const int row = crp[k];
#pragma unroll
  for (int d = 13; d < 27; d++) {
    if (rap_group(d) != G) continue;
    const int D[3] = {d / 9 - 1, (d / 3) % 3 - 1, d % 3 - 1};
    bool in = true;
    int pos = 0, back = 0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int n = K[a] + D[a];
      in &= n >= 0 && n < Mc;
      pos = pos * cnt[a] + D[a] - lo[a];
      const int nlo = n > 0 ? -1 : 0;  // k's place in row n
      back = back * ((n < Mc - 1 ? 1 : 0) - nlo + 1) - D[a] - nlo;
    }
    if (!in) continue;
    cv[row + pos] = (T)s[d];
    if (d > 13) cv[crp[nn[d]] + back] = (T)s[d];
  }
}

template <class T>
__global__ __launch_bounds__(64, sizeof(T) == 4 ? 2 : 1) void k_rap_q1(
    int Mc, FastDiv dMc, const T *a27, const T *t27, const int *__restrict__ crp, T *cv) {
  const unsigned k = blockIdx.x * 64 + threadIdx.x;
  if (k >= (unsigned)Mc * (unsigned)Mc * (unsigned)Mc) return;
  int K[3];
  lat_decode(k, dMc, K[0], K[1], K[2]);
  const auto all = std::make_integer_sequence<int, 27>();
  if (blockIdx.y == 0) rap_row<T, 0>(Mc, k, K, a27, t27, crp, cv, all);
  else if (blockIdx.y == 1) rap_row<T, 1>(Mc, k, K, a27, t27, crp, cv, all);
  else rap_row<T, 2>(Mc, k, K, a27, t27, crp, cv, all);
}

// The same from the CSRs, one thread per coarse entry (k, n), for matrices that hold no 27 planes
// (capped to SELL) or are not exactly symmetric and for interpolations without planes: every
// position is computed, the row starts included.  Same contributions in the same order.  Bound by
// the position arithmetic (49^3 coarse nodes FP32 1168 us).  A black-box hierarchy of six levels
// to 96^3 cells, FP32, capped to SELL, reassembles in 5.6 ms, 16.5 with k_rap_lds, which searches
// the positions; of five levels to 32^3 cells in 1.7, 9.3.
__device__ __forceinline__ int lat_pos3(const int lo[3], const int cnt[3], int a, int b, int c) {
  return ((a - lo[0]) * cnt[1] + (b - lo[1])) * cnt[2] + (c - lo[2]);
}

// the first entry of row (z, y, x) of a tensor product of 1-D patterns: pre[a] entries precede
// the row's coordinate on axis a, which has cnt[a] entries; nnz1 per 1-D pattern
__device__ __forceinline__ long pat_row_start(const long pre[3], const int cnt[3], long nnz1) {
  return (pre[0] * nnz1 + cnt[0] * pre[1]) * nnz1 + (long)cnt[0] * cnt[1] * pre[2];
}

template <class T>
__global__ __launch_bounds__(256) void k_rap_entry(int Mc, int M, const T *__restrict__ av,
                                                   const T *__restrict__ pv,
                                                   const int *__restrict__ crp, double *acc,
                                                   int upper) {
  // the 1-D patterns: A's row i holds i - 1, i, i + 1 within the lattice (3 M - 2 entries,
  // 3 i - 1 of them before row i > 0); P's row i holds i / 2 and, for odd i, i / 2 + 1
  // (3 Mc - 2 entries, i + i / 2 before row i)
  const long nA = 3L * M - 2, nP = 3L * Mc - 2;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long Nc = (long)Mc * Mc * Mc;
  if (t >= Nc * 27) return;
  const int k = (int)(t / 27), d = (int)(t - (long)k * 27);
  const int K[3] = {k / (Mc * Mc), (k / Mc) % Mc, k % Mc};
  const int D[3] = {d / 9 - 1, (d / 3) % 3 - 1, d % 3 - 1};
  int Nn[3], clo[3], ccnt[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    Nn[a] = K[a] + D[a];
    if (Nn[a] < 0 || Nn[a] >= Mc) return;
    clo[a] = K[a] > 0 ? -1 : 0;
    ccnt[a] = (K[a] < Mc - 1 ? 1 : 0) - clo[a] + 1;
  }
  const int n = (Nn[0] * Mc + Nn[1]) * Mc + Nn[2];
  if (upper && n < k) return;  // the lower triangle is mirrored afterwards
  double s = 0.0;
  const int l0[3] = {max(2 * K[0] - 1, 0), max(2 * K[1] - 1, 0), max(2 * K[2] - 1, 0)};
  const int l1[3] = {min(2 * K[0] + 1, M - 1), min(2 * K[1] + 1, M - 1), min(2 * K[2] + 1, M - 1)};
  for (int lz = l0[0]; lz <= l1[0]; lz++)
    for (int ly = l0[1]; ly <= l1[1]; ly++)
      for (int lx = l0[2]; lx <= l1[2]; lx++) {
        const int L[3] = {lz, ly, lx};
        // P_lk: row l holds floor(l / 2) (and ceil(l / 2) on odd coordinates) per axis
        int plo[3], pcnt[3], alo[3], acnt[3], m0[3], m1[3];
        long ppre[3], apre[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
          plo[a] = L[a] >> 1;
          pcnt[a] = (L[a] & 1) + 1;
          ppre[a] = L[a] + (L[a] >> 1);
          alo[a] = L[a] > 0 ? L[a] - 1 : 0;
          acnt[a] = min(L[a] + 1, M - 1) - alo[a] + 1;
          apre[a] = L[a] > 0 ? 3L * L[a] - 1 : 0;
          m0[a] = max(max(L[a] - 1, 2 * Nn[a] - 1), 0);
          m1[a] = min(min(L[a] + 1, 2 * Nn[a] + 1), M - 1);
        }
        const double plk =
            (double)pv[pat_row_start(ppre, pcnt, nP) + lat_pos3(plo, pcnt, K[0], K[1], K[2])];
        const long ab = pat_row_start(apre, acnt, nA);
        for (int mz = m0[0]; mz <= m1[0]; mz++)
          for (int my = m0[1]; my <= m1[1]; my++)
            for (int mx = m0[2]; mx <= m1[2]; mx++) {
              const double w = plk * (double)av[ab + lat_pos3(alo, acnt, mz, my, mx)];
              const int qlo[3] = {mz >> 1, my >> 1, mx >> 1};
              const int qcnt[3] = {(mz & 1) + 1, (my & 1) + 1, (mx & 1) + 1};
              const long qpre[3] = {mz + (mz >> 1), my + (my >> 1), mx + (mx >> 1)};
              s += w * (double)pv[pat_row_start(qpre, qcnt, nP) +
                                  lat_pos3(qlo, qcnt, Nn[0], Nn[1], Nn[2])];
            }
      }
  acc[crp[k] + lat_pos3(clo, ccnt, D[0], D[1], D[2])] = s;
}

// the longest row: a grid of at most 1024 blocks strides over the rows, each block reduces its
// maximum in LDS and issues one atomic (atomics to one address are serialised)
constexpr int kMaxRowBlocks = 1024;

__global__ __launch_bounds__(256) void k_max_row(int n, const int *__restrict__ rp, int *mx) {
  __shared__ int wm[4];
  int len = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    len = max(len, rp[i + 1] - rp[i]);
  for (int off = 32; off > 0; off >>= 1) len = max(len, __shfl_xor(len, off, 64));
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = len;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int m = max(max(wm[0], wm[1]), max(wm[2], wm[3]));
    if (m > 0) atomicMax(mx, m);
  }
}

// the longest row of A's CSR (A's SELL may not be built yet)
static int max_row_length(const flgpu_mat *A) {
  if (A->nrows == 0) return 0;
  int *dm = (int *)dev_alloc(sizeof(int));
  FLGPU_HIP(hipMemsetAsync(dm, 0, sizeof(int), A->ctx->stream));
  const unsigned g = std::min<unsigned>(grid_for(A->nrows, 256), kMaxRowBlocks);
  k_max_row<<<g, 256, 0, A->ctx->stream>>>(A->nrows, A->rowptr, dm);
  FLGPU_HIP(hipGetLastError());
  int h = 0;
  FLGPU_HIP(hipMemcpyAsync(&h, dm, sizeof(int), hipMemcpyDeviceToHost, A->ctx->stream));
  FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
  dev_free(dm);
  return h;
}

template <class T>
__global__ void k_store(long n, const double *acc, T *v) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = (T)acc[i];
}

// asym[0] = 1 unless A's values are exactly symmetric (every A(i, j) has an equal A(j, i))
template <class T>
__global__ void k_csr_symcheck(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                               const T *__restrict__ v, int *asym) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bool bad = false;
  for (int e = rp[i]; e < rp[i + 1]; e++) {
    int j = ci[e];
    if (j == i) continue;
    int lo = rp[j], hi = rp[j + 1] - 1;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (ci[mid] < i) lo = mid + 1;
      else hi = mid;
    }
    bad |= lo > hi || ci[lo] != i || !(v[lo] == v[e]);
  }
  if (bad) asym[0] = 1;
}

// The same with one lane per entry (32 lanes per row, rows of at most 32 entries): the binary
// searches of a row run side by side instead of one after another.
template <class T>
__global__ __launch_bounds__(256) void k_csr_symcheck32(int n, const int *__restrict__ rp,
                                                        const int *__restrict__ ci,
                                                        const T *__restrict__ v, int *asym) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int i = (int)(t >> 5), k = (int)(t & 31);
  if (i >= n) return;
  const int e = rp[i] + k;
  if (e >= rp[i + 1]) return;
  const int j = ci[e];
  if (j == i) return;
  int lo = rp[j], hi = rp[j + 1] - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (ci[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  if (lo > hi || ci[lo] != i || !(v[lo] == v[e])) asym[0] = 1;
}

// the lower triangle of the coarse accumulators from the upper one (missing[0] = 1 when the
// pattern has no transposed position)
__global__ void k_mirror(int nc, const int *__restrict__ crp, const int *__restrict__ cci,
                         double *acc, int *missing) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nc) return;
  for (int e = crp[k]; e < crp[k + 1]; e++) {
    int m = cci[e];
    if (m >= k) break;
    int lo = crp[m], hi = crp[m + 1] - 1;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (cci[mid] < k) lo = mid + 1;
      else hi = mid;
    }
    if (lo > hi || cci[lo] != k) missing[0] = 1;
    else acc[e] = acc[lo];
  }
}

static bool csr_symmetric(const flgpu_mat *A) {
  if (A->nrows != A->ncols || A->nrows == 0) return false;
  flgpu_ctx *ctx = A->ctx;
  int *asym = (int *)dev_alloc(sizeof(int));
  FLGPU_HIP(hipMemsetAsync(asym, 0, sizeof(int), ctx->stream));
  const bool lanes = max_row_length(A) <= 32;
  const unsigned g32 = grid_for(32L * A->nrows, 256);
  if (A->prec == FLGPU_F64) {
    if (lanes)
      k_csr_symcheck32<double><<<g32, 256, 0, ctx->stream>>>(A->nrows, A->rowptr, A->colidx,
                                                              (const double *)A->vals, asym);
    else
      k_csr_symcheck<double><<<grid_for(A->nrows, 256), 256, 0, ctx->stream>>>(
          A->nrows, A->rowptr, A->colidx, (const double *)A->vals, asym);
  } else {
    if (lanes)
      k_csr_symcheck32<float><<<g32, 256, 0, ctx->stream>>>(A->nrows, A->rowptr, A->colidx,
                                                             (const float *)A->vals, asym);
    else
      k_csr_symcheck<float><<<grid_for(A->nrows, 256), 256, 0, ctx->stream>>>(
          A->nrows, A->rowptr, A->colidx, (const float *)A->vals, asym);
  }
  FLGPU_HIP(hipGetLastError());
  int h = 1;
  FLGPU_HIP(hipMemcpyAsync(&h, asym, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  FLGPU_HIP(hipStreamSynchronize(ctx->stream));
  dev_free(asym);
  return h == 0;
}

// Ac's values <- P^T A P (pattern of Ac given); all three share one precision.  When A is
// exactly symmetric, only the upper triangle is accumulated and mirrored, so Ac is exactly
// symmetric too (the two triangles of P^T A P otherwise round differently), which lets the
// stencil kernels stream half the coefficients.
void galerkin_product(const flgpu_mat *P, const flgpu_mat *A, flgpu_mat *Ac, bool lattice) {
  FLGPU_REQUIRE(P->nrows == A->nrows && A->nrows == A->ncols, "galerkin: P and A do not match");
  FLGPU_REQUIRE(Ac->nrows == P->ncols && Ac->ncols == P->ncols, "galerkin: Ac does not match P");
  FLGPU_REQUIRE(P->prec == A->prec && A->prec == Ac->prec, "galerkin: precisions differ");
  flgpu_ctx *ctx = A->ctx;
  const int nc = Ac->nrows;
  // the structured products: 3D Q1, the fine lattice of an even n, the patterns' sizes as the
  // lattices give them
  const long nf = A->lat_n, ncl = nf / 2;
  const bool q1 = lattice && is_q1_lattice(A) && nf % 2 == 0 &&
                  A->nnz == (3 * nf + 1) * (3 * nf + 1) * (3 * nf + 1) &&
                  Ac->nrows == (ncl + 1) * (ncl + 1) * (ncl + 1) &&
                  Ac->nnz == (3 * ncl + 1) * (3 * ncl + 1) * (3 * ncl + 1) &&
                  P->nnz == (3 * ncl + 1) * (3 * ncl + 1) * (3 * ncl + 1);
  const flgpu_mat *PT = P->transpose;
  // from the planes: A exactly symmetric
  if (q1 && A->val27 && A->st_sym && PT && PT->tp_kind == 2 && PT->tp27 && PT->tp_nc == ncl) {
    auto run = [&](auto t) {
      using T = decltype(t);
      k_rap_q1<T><<<dim3(grid_for(nc, 64), 3), 64, 0, ctx->stream>>>(
          (int)ncl + 1, fast_div((unsigned)ncl + 1), (const T *)A->val27, (const T *)PT->tp27,
          Ac->rowptr, (T *)Ac->vals);
    };
    if (A->prec == FLGPU_F64) run(0.0);
    else run(0.0f);
    FLGPU_HIP(hipGetLastError());
    return;
  }
  double *acc = (double *)dev_alloc(sizeof(double) * std::max<long>(Ac->nnz, 1));
  int *bad = (int *)dev_alloc(sizeof(int));
  FLGPU_HIP(hipMemsetAsync(bad, 0, sizeof(int), ctx->stream));
  int *missing = (int *)dev_alloc(sizeof(int));
  if (!q1) mat_build_transpose(P);  // the general product walks the rows of P^T
  PT = P->transpose;
  const bool lds = !q1 && max_row_length(Ac) <= kRapW;
  auto rap = [&](int upper) {
    const unsigned gl = (unsigned)((nc + kRapB - 1) / kRapB);
    if (q1 && A->prec == FLGPU_F64)
      k_rap_entry<double><<<grid_for(27L * nc, 256), 256, 0, ctx->stream>>>(
          (int)ncl + 1, (int)nf + 1, (const double *)A->vals, (const double *)P->vals,
          Ac->rowptr, acc, upper);
    else if (q1)
      k_rap_entry<float><<<grid_for(27L * nc, 256), 256, 0, ctx->stream>>>(
          (int)ncl + 1, (int)nf + 1, (const float *)A->vals, (const float *)P->vals, Ac->rowptr,
          acc, upper);
    else if (lds && A->prec == FLGPU_F64)
      k_rap_lds<double><<<gl, kRapB, 0, ctx->stream>>>(
          nc, PT->rowptr, PT->colidx, (const double *)PT->vals, A->rowptr, A->colidx,
          (const double *)A->vals, P->rowptr, P->colidx, (const double *)P->vals, Ac->rowptr,
          Ac->colidx, acc, bad, upper);
    else if (lds)
      k_rap_lds<float><<<gl, kRapB, 0, ctx->stream>>>(
          nc, PT->rowptr, PT->colidx, (const float *)PT->vals, A->rowptr, A->colidx,
          (const float *)A->vals, P->rowptr, P->colidx, (const float *)P->vals, Ac->rowptr,
          Ac->colidx, acc, bad, upper);
    else if (A->prec == FLGPU_F64)
      k_rap<double><<<grid_for(nc, 128), 128, 0, ctx->stream>>>(
          nc, PT->rowptr, PT->colidx, (const double *)PT->vals, A->rowptr, A->colidx,
          (const double *)A->vals, P->rowptr, P->colidx, (const double *)P->vals, Ac->rowptr,
          Ac->colidx, acc, bad, upper);
    else
      k_rap<float><<<grid_for(nc, 128), 128, 0, ctx->stream>>>(
          nc, PT->rowptr, PT->colidx, (const float *)PT->vals, A->rowptr, A->colidx,
          (const float *)A->vals, P->rowptr, P->colidx, (const float *)P->vals, Ac->rowptr,
          Ac->colidx, acc, bad, upper);
    FLGPU_HIP(hipGetLastError());
  };
  int hmiss = 1;
  // a lattice matrix's stencil form records whether its values are exactly symmetric
  if (q1 && A->val27 ? A->st_sym : csr_symmetric(A)) {
    FLGPU_HIP(hipMemsetAsync(missing, 0, sizeof(int), ctx->stream));
    rap(1);
    k_mirror<<<grid_for(nc, 128), 128, 0, ctx->stream>>>(nc, Ac->rowptr, Ac->colidx, acc,
                                                          missing);
    FLGPU_HIP(hipGetLastError());
    FLGPU_HIP(hipMemcpyAsync(&hmiss, missing, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    FLGPU_HIP(hipStreamSynchronize(ctx->stream));
  }
  if (hmiss) rap(0);  // not symmetric, or the coarse pattern is not: the full product
  if (A->prec == FLGPU_F64)
    k_store<double><<<grid_for(Ac->nnz, 256), 256, 0, ctx->stream>>>(Ac->nnz, acc,
                                                                     (double *)Ac->vals);
  else
    k_store<float><<<grid_for(Ac->nnz, 256), 256, 0, ctx->stream>>>(Ac->nnz, acc,
                                                                    (float *)Ac->vals);
  FLGPU_HIP(hipGetLastError());
  int hbad = 0;
  FLGPU_HIP(hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  FLGPU_HIP(hipStreamSynchronize(ctx->stream));
  dev_free(acc);
  dev_free(bad);
  dev_free(missing);
  FLGPU_REQUIRE(!hbad, "galerkin: P^T A P has entries outside the coarse pattern");
}

}  // namespace flgpu

using namespace flgpu;

// ---- C-ABI ---------------------------------------------------------------------------

extern "C" int flgpu_galerkin_product(const flgpu_mat *P, const flgpu_mat *A, flgpu_mat *Ac) {
  return guard([&] {
    FLGPU_REQUIRE(P && A && Ac, "arguments must not be NULL");
    FLGPU_REQUIRE(P->ctx == A->ctx && A->ctx == Ac->ctx, "matrices of different contexts");
    CTX_LOCK(A->ctx);
    galerkin_product(P, A, Ac);
    drop_alpha(Ac);  // Ac's forms that are sums over cells do not hold the new values
    drop_cells(Ac);
    mat_refresh_values(Ac);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    return 0;
  });
}

extern "C" int flgpu_csr_upload(flgpu_ctx *ctx, int nrows, int ncols, long nnz, const int *rowptr,
                                const int *colidx, const double *vals, int prec,
                                flgpu_mat **out) {
  return guard([&] {
    FLGPU_REQUIRE(ctx && out && rowptr, "ctx, rowptr and out must not be NULL");
    FLGPU_REQUIRE(nnz == 0 || (colidx && vals), "colidx and vals must not be NULL");
    FLGPU_REQUIRE(nrows >= 0 && ncols >= 0, "negative dimension");
    FLGPU_REQUIRE(rowptr[0] == 0 && rowptr[nrows] == nnz, "rowptr must run from 0 to nnz");
    for (int r = 0; r < nrows; r++) {
      FLGPU_REQUIRE(rowptr[r + 1] >= rowptr[r], "rowptr must be non-decreasing");
      for (int e = rowptr[r]; e < rowptr[r + 1]; e++) {
        FLGPU_REQUIRE(colidx[e] >= 0 && colidx[e] < ncols, "column index out of range");
        FLGPU_REQUIRE(e == rowptr[r] || colidx[e] > colidx[e - 1],
                      "column indices must ascend strictly within a row");
      }
    }
    CTX_LOCK(ctx);
    flgpu_mat *A = mat_new(ctx, nrows, ncols, nnz, prec);
    try {
      FLGPU_HIP(hipMemcpyAsync(A->rowptr, rowptr, sizeof(int) * (nrows + 1), hipMemcpyHostToDevice,
                               ctx->stream));
      if (nnz)
        FLGPU_HIP(hipMemcpyAsync(A->colidx, colidx, sizeof(int) * nnz, hipMemcpyHostToDevice,
                                 ctx->stream));
      upload_vals(A, vals);
      mat_finish(A);
      FLGPU_HIP(hipStreamSynchronize(ctx->stream));
    } catch (...) {
      mat_free(A);
      throw;
    }
    *out = A;
    return 0;
  });
}

extern "C" int flgpu_csr_update_values(flgpu_mat *A, const double *vals) {
  return guard([&] {
    FLGPU_REQUIRE(A && (vals || A->nnz == 0), "arguments must not be NULL");
    CTX_LOCK(A->ctx);
    drop_alpha(A);
    drop_cells(A);
    upload_vals(A, vals);
    mat_refresh_values(A);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    return 0;
  });
}

extern "C" int flgpu_csr_download(const flgpu_mat *A, int *rowptr, int *colidx, double *vals) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    CTX_LOCK(A->ctx);
    std::vector<int> rp, ci;
    std::vector<double> v;
    download_csr(A, rp, ci, vals ? &v : nullptr);
    if (rowptr) std::memcpy(rowptr, rp.data(), sizeof(int) * rp.size());
    if (colidx) std::memcpy(colidx, ci.data(), sizeof(int) * ci.size());
    if (vals) std::memcpy(vals, v.data(), sizeof(double) * v.size());
    return 0;
  });
}

extern "C" int flgpu_mat_info(const flgpu_mat *A, int *nrows, int *ncols, long *nnz, int *prec) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    if (nrows) *nrows = A->nrows;
    if (ncols) *ncols = A->ncols;
    if (nnz) *nnz = A->nnz;
    if (prec) *prec = A->prec;
    return 0;
  });
}

extern "C" int flgpu_mat_convert(const flgpu_mat *A, int prec, flgpu_mat **out) {
  return guard([&] {
    FLGPU_REQUIRE(A && out, "arguments must not be NULL");
    CTX_LOCK(A->ctx);
    *out = mat_convert(A, prec);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    return 0;
  });
}

extern "C" int flgpu_mat_storage(flgpu_mat *A, int max_form, int *form) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    CTX_LOCK(A->ctx);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    if (max_form < FLGPU_STORAGE_CELL) {
      drop_alpha(A);
      drop_cells(A);
    }
    if (max_form < FLGPU_STORAGE_STENCIL) {
      drop_stencil(A);
      tp_drop(A);
      q2t_drop(A);
    }
    long lat_rows = 1;
    for (int k = 0; k < A->lat_dim; k++) lat_rows *= (long)A->lat_order * A->lat_n + 1;
    if (!A->alpha && !A->val27 && A->lat_dim > 0 && A->ncolours == 0 && A->nrows == lat_rows)
      lattice_colouring(A, A->lat_dim, A->lat_order, A->lat_n);
    if (form)
      *form = A->alpha                   ? FLGPU_STORAGE_CELL
              : (A->val27 || A->tp_kind) ? FLGPU_STORAGE_STENCIL
                                         : FLGPU_STORAGE_SELL;
    return 0;
  });
}

extern "C" int flgpu_mat_stencil_planes(const flgpu_mat *A, int *planes) {
  return guard([&] {
    FLGPU_REQUIRE(A && planes, "arguments must not be NULL");
    *planes = (A->alpha || !A->val27) ? 0 : (A->st_sym ? 14 : 27);
    return 0;
  });
}

extern "C" int flgpu_mat_destroy(flgpu_mat *A) {
  return guard([&] {
    if (!A) return 0;
    CTX_LOCK(A->ctx);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    mat_free(A);
    return 0;
  });
}

static void check_vec(const flgpu_mat *A, const flgpu_vec *v, long n, const char *what) {
  FLGPU_REQUIRE(v != nullptr, std::string(what) + " must not be NULL");
  FLGPU_REQUIRE(v->ctx == A->ctx, std::string(what) + " belongs to another context");
  FLGPU_REQUIRE(v->n == n, std::string(what) + ": length mismatch");
  FLGPU_REQUIRE(v->prec == A->prec, std::string(what) + ": precision differs from the matrix");
}

extern "C" int flgpu_gemm_nn(double alpha, const flgpu_mat *A, const flgpu_vec *y, double beta,
                             flgpu_vec *x) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    check_vec(A, y, A->ncols, "y");
    check_vec(A, x, A->nrows, "x");
    FLGPU_REQUIRE(x->d != y->d, "gemm!: x and y must be different vectors");
    CTX_LOCK(A->ctx);
    spmv(A, alpha, y->d, beta, x->d, x->d);
    return 0;
  });
}

extern "C" int flgpu_gemm_tn(double alpha, const flgpu_mat *A, const flgpu_vec *y, double beta,
                             flgpu_vec *x) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    check_vec(A, y, A->nrows, "y");
    check_vec(A, x, A->ncols, "x");
    FLGPU_REQUIRE(x->d != y->d, "gemm!: x and y must be different vectors");
    CTX_LOCK(A->ctx);
    mat_build_transpose(A);
    spmv(A->transpose, alpha, y->d, beta, x->d, x->d);
    return 0;
  });
}

extern "C" int flgpu_compute_residual(const flgpu_mat *A, const flgpu_vec *x, const flgpu_vec *b,
                                      flgpu_vec *r) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    FLGPU_REQUIRE(A->nrows == A->ncols, "compute-residual needs a square matrix");
    check_vec(A, x, A->ncols, "x");
    check_vec(A, b, A->nrows, "b");
    check_vec(A, r, A->nrows, "r");
    FLGPU_REQUIRE(x->d != r->d, "compute-residual: x and r must be different vectors");
    CTX_LOCK(A->ctx);
    spmv(A, -1.0, x->d, 1.0, b->d, r->d);
    return 0;
  });
}

extern "C" int flgpu_mat_set_colouring(flgpu_mat *A, int ncolours, const int *colour) {
  return guard([&] {
    FLGPU_REQUIRE(A && colour, "arguments must not be NULL");
    CTX_LOCK(A->ctx);
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    drop_alpha(A);  // sweeps follow the caller's colours from now on
    drop_stencil(A);
    set_colouring(A, ncolours, colour);
    return 0;
  });
}

extern "C" int flgpu_mat_colour_greedy(flgpu_mat *A, int *ncolours) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    FLGPU_REQUIRE(A->nrows == A->ncols, "colouring needs a square matrix");
    CTX_LOCK(A->ctx);
    std::vector<int> rp, ci;
    download_csr(A, rp, ci, nullptr);
    std::vector<int> colour(A->nrows, -1);
    int nc = 0;
    std::vector<int> used;
    for (int r = 0; r < A->nrows; r++) {
      used.assign(nc + 1, 0);
      for (int e = rp[r]; e < rp[r + 1]; e++) {
        int c = ci[e];
        if (c != r && colour[c] >= 0) used[colour[c]] = 1;
      }
      // symmetric pattern assumed for the reverse couplings; check columns
      int k = 0;
      while (k < nc && used[k]) k++;
      colour[r] = k;
      if (k == nc) nc++;
    }
    FLGPU_HIP(hipStreamSynchronize(A->ctx->stream));
    drop_alpha(A);
    drop_stencil(A);
    set_colouring(A, nc, colour.data());
    if (ncolours) *ncolours = nc;
    return 0;
  });
}

extern "C" int flgpu_jacobi_steps(const flgpu_mat *A, double damp, int steps, flgpu_vec *x,
                                  const flgpu_vec *b, flgpu_vec *tmp) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    FLGPU_REQUIRE(A->nrows == A->ncols, "<jacobi> needs a square matrix");
    FLGPU_REQUIRE(steps >= 0, "negative number of steps");
    check_vec(A, x, A->nrows, "x");
    check_vec(A, b, A->nrows, "b");
    check_vec(A, tmp, A->nrows, "tmp");
    FLGPU_REQUIRE(x != tmp && b != tmp && x != b, "x, b and tmp must be distinct vectors");
    CTX_LOCK(A->ctx);
    jacobi_steps(A, damp, steps, x->d, b->d, tmp->d);
    return 0;
  });
}

extern "C" int flgpu_jacobi_iterate(const flgpu_mat *A, double damp, flgpu_vec *x, flgpu_vec *r) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    FLGPU_REQUIRE(A->nrows == A->ncols, "<jacobi> needs a square matrix");
    check_vec(A, x, A->nrows, "x");
    check_vec(A, r, A->nrows, "r");
    CTX_LOCK(A->ctx);
    jacobi_iterate(A, damp, x->d, r->d);
    return 0;
  });
}

extern "C" int flgpu_sor_iterate(const flgpu_mat *A, double omega, int backwards, flgpu_vec *x,
                                 const flgpu_vec *b, flgpu_vec *r) {
  return guard([&] {
    FLGPU_REQUIRE(A, "matrix must not be NULL");
    check_vec(A, x, A->nrows, "x");
    check_vec(A, b, A->nrows, "b");
    check_vec(A, r, A->nrows, "r");
    CTX_LOCK(A->ctx);
    sor_prepare(A);
    sor_sweeps(A, omega, 1, backwards, x->d, b->d, r->d);
    return 0;
  });
}
