// Krylov kernels on the reduced system in SELL-64 layout: SpMV, Jacobi-PCG
// with fused vector updates and deterministic reductions, and the
// reliable-update hook used by mixed-precision CG.
//
// Replaces the matrix-free jvp + jax.scipy.sparse.linalg.cg of
// linear_solve_jax (solver.py:1044-1116) and the host spsolve of
// linear_solve_scipy (:1493-1539) for the 'hip' backend.
//
// One PCG iteration = two streaming kernels, each followed by a one-block
// finalize kernel:
//   k_pcg_spmv  : p = z + beta p_old fused into the gather, q = A p, block
//                 partials of p.q;  k_pcg_alpha_fin forms alpha = gamma / p.q.
//   k_pcg_update: x += alpha p, r -= alpha q, z = D^-1 r, partials of r.z and
//                 r.r;  k_pcg_beta_fin forms beta, gamma, the stop flag and
//                 the reliable-update request.
// On symmetric 9-point matrices k_pcg_lines stands in for k_pcg_spmv and also updates x (below); systems
// that fit on the compute units run all iterations in one launch (resident.hip).
// Scalars live on the device.  Kernels exit at entry once a flag is set, so
// the host enqueues iterations in batches and reads the flags one batch late.
// The two direction buffers alternate by the device iteration counter.
// Reductions: fixed grid, per-block shuffle tree, the finalize kernel sums
// the partials in index order -> bitwise reproducible.  (A last-block-done
// reduction inside the streaming kernel would need a device-scope fence per
// block, which writes back the L2 of every XCD and cost more than the extra
// launch.)
//
// Bandwidth: every thread issues kUnroll independent element loads per pass
// (vector kernels) and one wavefront owns one 64-row SELL chunk with its
// value / column loads unrolled by 4, so enough requests are in flight to
// cover HBM latency; grids are sized to about one pass per thread.
#include <chrono>
#include <cstring>
#include <type_traits>

#include "assembly.hpp"

namespace apx {

constexpr int kBS = 256;        // vector kernels
constexpr int kSpmvBS = 512;    // SpMV kernels: 8 wavefronts = 8 chunks per block
constexpr int kUnroll = 4;
constexpr int kMaxBlocks = 8192;

ScopedTimer::ScopedTimer(Plan& p, const char* n, hipStream_t s, int64_t b) : P(p), name(n), st(s), bytes(b) {
  if (P.timing) (void)hipEventRecord(P.ev0, st);
}
ScopedTimer::~ScopedTimer() {
  if (!P.timing) return;
  (void)hipEventRecord(P.ev1, st);
  (void)hipEventSynchronize(P.ev1);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, P.ev0, P.ev1);
  auto& t = P.timers[name];
  t.total_ms += ms;
  t.count += 1;
  t.bytes = bytes;
}

static inline int grid_for(int64_t n) {
  const int64_t per_block = (int64_t)kBS * kUnroll;
  return (int)std::max<int64_t>(1, std::min<int64_t>((n + per_block - 1) / per_block, kMaxBlocks));
}
static inline int grid_chunks(int64_t n_chunks) {
  constexpr int wpb = kSpmvBS / 64;
  return (int)std::min<int64_t>(round_xcd(std::max<int64_t>(1, (n_chunks + wpb - 1) / wpb)), kMaxBlocks);
}

static_assert(kKrylovPartials == 4 * kMaxBlocks, "partials layout: 4 rows of kMaxBlocks");

void ensure_krylov_scratch(Plan& P, hipStream_t st) {
  if (P.partials.n < (size_t)(4 * kMaxBlocks)) P.partials.alloc(4 * kMaxBlocks);
  if (P.kstate.n < 64) {
    P.kstate.alloc(64);
    APX_HIP(hipMemsetAsync(P.kstate.p, 0, P.kstate.bytes(), st));
  }
}

// Cross-block reductions are split in two launches on the same stream: every
// block writes its partial sums (plain stores), then a one-block finalize
// kernel adds them in index order and updates the device scalars.  The kernel
// boundary makes the partials visible across the XCDs' separate L2 caches; an
// in-kernel last-block scheme would need an agent-scope release per block,
// which writes back the whole L2 each time.
template <int BS, int NV>
__device__ inline void block_partials_at(double (&v)[NV], double* partials, int64_t block) {
  __shared__ double lds[BS / 64];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const double s = block_sum<BS>(v[j], lds);
    if (threadIdx.x == 0) partials[j * kMaxBlocks + block] = s;
  }
}
template <int BS, int NV>
__device__ inline void block_partials(double (&v)[NV], double* partials) {
  block_partials_at<BS, NV>(v, partials, blockIdx.x);
}

constexpr int kFinBS = 1024;

// Sum NV rows of nb partials (fixed order) -> valid in all threads.
template <int NV>
__device__ inline void finalize_sums(const double* partials, int nb, double (&sums)[NV]) {
  __shared__ double lds[kFinBS / 64];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    double s = 0.0;
#pragma unroll 8
    for (int i = threadIdx.x; i < nb; i += kFinBS) s += partials[j * kMaxBlocks + i];
    sums[j] = block_sum<kFinBS>(s, lds);
  }
}

// Column of a stored entry: an int32 column as stored, or an int16 offset from the row (base)
__device__ __forceinline__ int32_t sell_col(int32_t c, int32_t) { return c; }
__device__ __forceinline__ int32_t sell_col(int16_t d, int32_t base) { return base + (int32_t)d; }
// The row an int16 offset is taken from: the lane's row, or the last row for lanes past n
__device__ __forceinline__ int32_t sell_base(int64_t row, int64_t n) { return (int32_t)(row < n ? row : n - 1); }

// Row gather of one SELL chunk: sum_k vals[k] * f(col[k]) for this lane's row,
// values of type M, accumulated in V (FP32 values with FP64 vectors: each
// value is widened exactly and the products and sums are FP64).
// U entries per step: all their column and value loads are issued before the gathers (U = 8
// for the wide rows of 3-DOF elasticity, 4 otherwise); the sum order is k = 0, 1, 2, ... either way.
template <class M, class V = M, int U = 4, class C, class F>
__device__ __forceinline__ V sell_row(const M* __restrict__ v, const C* __restrict__ ci, int w, int32_t base, F f) {
  V s = 0;
  int k = 0;
  for (; k + U <= w; k += U) {
    // values and columns are read once per SpMV: non-temporal, so L2 keeps the gathered vector
    C c[U];
    M vv[U];
#pragma unroll
    for (int j = 0; j < U; ++j) c[j] = __builtin_nontemporal_load(ci + (k + j) * 64);
#pragma unroll
    for (int j = 0; j < U; ++j) vv[j] = __builtin_nontemporal_load(v + (k + j) * 64);
#pragma unroll
    for (int j = 0; j < U; ++j) s += (V)vv[j] * f(sell_col(c[j], base));
  }
  for (; k < w; ++k)
    s += (V)__builtin_nontemporal_load(v + k * 64) * f(sell_col(__builtin_nontemporal_load(ci + k * 64), base));
  return s;
}

// ---- SpMV (SELL-64: one wavefront per chunk, lane = row) --------------------------
template <class T, class C>
__global__ __launch_bounds__(kSpmvBS) void k_spmv_sell(int64_t n, int64_t n_chunks, const int32_t* __restrict__ sptr,
                                                       const C* __restrict__ cols, const T* __restrict__ vals,
                                                       const T* __restrict__ x, T* __restrict__ y) {
  constexpr int wpb = kSpmvBS / 64;
  const int lane = threadIdx.x & 63;
  for (int64_t c = blockIdx.x * (int64_t)wpb + (threadIdx.x >> 6); c < n_chunks; c += (int64_t)gridDim.x * wpb) {
    const int32_t off = sptr[c], w = (sptr[c + 1] - off) >> 6;
    const int64_t row = c * 64 + lane;
    const T s = sell_row<T>(vals + off + lane, cols + off + lane, w, sell_base(row, n),
                            [&](int32_t col) { return x[col]; });
    if (row < n) y[row] = s;
  }
}

void spmv(Plan& P, const void* vals, const void* x, void* y, int precision, hipStream_t st) {
  const int g = grid_chunks(P.n_chunks);
  auto run = [&](auto cols) {
    using C = std::remove_const_t<std::remove_pointer_t<decltype(cols)>>;
    if (precision == APX_FP64)
      hipLaunchKernelGGL((k_spmv_sell<double, C>), dim3(g), dim3(kSpmvBS), 0, st, P.n_free, P.n_chunks, P.sell_ptr.p,
                         cols, (const double*)vals, (const double*)x, (double*)y);
    else
      hipLaunchKernelGGL((k_spmv_sell<float, C>), dim3(g), dim3(kSpmvBS), 0, st, P.n_free, P.n_chunks, P.sell_ptr.p,
                         cols, (const float*)vals, (const float*)x, (float*)y);
  };
  if (P.sell_dcol.p)
    run((const int16_t*)P.sell_dcol.p);
  else
    run((const int32_t*)P.sell_cols.p);
  APX_LAUNCH_CHECK();
}

// ---- layout conversion --------------------------------------------------------------
template <class T>
__global__ void k_sell_to_csr(int64_t nnz, const int32_t* csr2sell, const T* sell, T* csr) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nnz; k += (int64_t)gridDim.x * blockDim.x)
    csr[k] = sell[csr2sell[k]];
}
template <class T>
__global__ void k_csr_to_sell(int64_t nnz, const int32_t* csr2sell, const T* csr, T* sell) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nnz; k += (int64_t)gridDim.x * blockDim.x)
    sell[csr2sell[k]] = csr[k];
}

void sell_to_csr(Plan& P, const void* sell, void* csr, int precision, hipStream_t st) {
  const int g = (int)std::max<int64_t>(1, std::min<int64_t>((P.nnz + 255) / 256, 65536));
  if (precision == APX_FP64)
    hipLaunchKernelGGL(k_sell_to_csr<double>, dim3(g), dim3(256), 0, st, P.nnz, P.csr2sell.p, (const double*)sell,
                       (double*)csr);
  else
    hipLaunchKernelGGL(k_sell_to_csr<float>, dim3(g), dim3(256), 0, st, P.nnz, P.csr2sell.p, (const float*)sell,
                       (float*)csr);
  APX_LAUNCH_CHECK();
}

void csr_to_sell(Plan& P, const void* csr, void* sell, int precision, hipStream_t st) {
  const int g = (int)std::max<int64_t>(1, std::min<int64_t>((P.nnz + 255) / 256, 65536));
  if (precision == APX_FP64) {
    fill<double>((double*)sell, P.sell_total, 0.0, st);
    hipLaunchKernelGGL(k_csr_to_sell<double>, dim3(g), dim3(256), 0, st, P.nnz, P.csr2sell.p, (const double*)csr,
                       (double*)sell);
  } else {
    fill<float>((float*)sell, P.sell_total, 0.0f, st);
    hipLaunchKernelGGL(k_csr_to_sell<float>, dim3(g), dim3(256), 0, st, P.nnz, P.csr2sell.p, (const float*)csr,
                       (float*)sell);
  }
  APX_LAUNCH_CHECK();
}

// ---- Jacobi ------------------------------------------------------------------------
template <class M, class V = M>
__global__ void k_inv_diag(int64_t n, const int32_t* diag_slot, const M* vals, V* inv) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    inv[i] = V(1) / (V)vals[diag_slot[i]];
}

void jacobi_inverse(Plan& P, const void* vals, void* inv, int precision, hipStream_t st) {
  const int g = std::max(1, (int)std::min<int64_t>((P.n_free + 255) / 256, 65536));
  if (precision == APX_FP64)
    hipLaunchKernelGGL(k_inv_diag<double>, dim3(g), dim3(256), 0, st, P.n_free, P.diag_slot.p, (const double*)vals,
                       (double*)inv);
  else
    hipLaunchKernelGGL(k_inv_diag<float>, dim3(g), dim3(256), 0, st, P.n_free, P.diag_slot.p, (const float*)vals,
                       (float*)inv);
  APX_LAUNCH_CHECK();
}

void jacobi_inverse_f32_to_f64(Plan& P, const float* vals, double* inv, hipStream_t st) {
  const int g = std::max(1, (int)std::min<int64_t>((P.n_free + 255) / 256, 65536));
  hipLaunchKernelGGL((k_inv_diag<float, double>), dim3(g), dim3(256), 0, st, P.n_free, P.diag_slot.p, vals, inv);
  APX_LAUNCH_CHECK();
}

// ---- PCG kernels --------------------------------------------------------------------
__device__ __forceinline__ bool halted(const KState* S) { return S->done | S->reliable; }

// Elementwise pass with kUnroll independent elements per thread and pass.
#define APX_FOR_ELEMENTS(n, BODY_LOAD, BODY_STORE)                                         \
  for (int64_t base = blockIdx.x * (int64_t)kBS * kUnroll + threadIdx.x; base < (n);        \
       base += (int64_t)gridDim.x * kBS * kUnroll) {                                        \
    _Pragma("unroll") for (int j = 0; j < kUnroll; ++j) {                                   \
      const int64_t i = base + (int64_t)j * kBS;                                            \
      if (i < (n)) { BODY_LOAD }                                                            \
    }                                                                                       \
    _Pragma("unroll") for (int j = 0; j < kUnroll; ++j) {                                   \
      const int64_t i = base + (int64_t)j * kBS;                                            \
      if (i < (n)) { BODY_STORE }                                                           \
    }                                                                                       \
  }

// the slots of a resident run start at zero (its meetings count from 1)
template <int BS>
__device__ __forceinline__ void clear_resident_slots(double* partials) {
  static_assert(kResidentSlotsAt == 2 * kMaxBlocks && kResidentClearWords <= 2 * kMaxBlocks, "slots behind two rows");
  for (int i = threadIdx.x; i < kResidentClearWords; i += BS) partials[kResidentSlotsAt + i] = 0.0;
}

struct PcgStart {
  double tol, atol, delta;
  int maxiter;
};
// the scalars of a run from r.z and r.r
__device__ __forceinline__ void pcg_start(KState* S, double rz, double rr, const PcgStart& A) {
  S->gamma = rz;
  S->gamma_prev = rz;
  S->rr = rr;
  S->rr0 = rr;
  S->bb = rr;
  S->rmax2 = rr;
  S->delta2 = A.delta * A.delta;
  S->atol2 = fmax(A.tol * A.tol * rr, A.atol * A.atol);
  S->beta = 0.0;
  S->k = 0;
  S->maxiter = A.maxiter;
  S->reliable = 0;
  S->done = !(rr > S->atol2 && 0 < A.maxiter);
}

// FULL: the right-hand side is -rfull on the free DOFs, else b.  ONE: the launch is one block, which
// finishes the sums itself (a second launch and its wait were 5 us of a small solve).
template <class T, bool FULL, bool ONE>
__global__ __launch_bounds__(kBS) void k_pcg_init(int64_t n, const T* __restrict__ b,
                                                  const int32_t* __restrict__ red2full,
                                                  const double* __restrict__ rfull, const T* __restrict__ inv,
                                                  T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                  T* __restrict__ pa, KState* S, double* partials, PcgStart A) {
  double v[2] = {0.0, 0.0};
  T bv[kUnroll], iv[kUnroll];
  APX_FOR_ELEMENTS(n, { bv[j] = FULL ? (T)(-rfull[red2full[i]]) : b[i]; iv[j] = inv[i]; }, {
    const T zi = iv[j] * bv[j];
    x[i] = 0;
    r[i] = bv[j];
    z[i] = zi;
    pa[i] = 0;
    v[0] += (double)bv[j] * (double)zi;
    v[1] += (double)bv[j] * (double)bv[j];
  })
  if constexpr (ONE) {
    __shared__ double lds[kBS / 64];
    clear_resident_slots<kBS>(partials);
    const double rz = block_sum<kBS>(v[0], lds), rr = block_sum<kBS>(v[1], lds);
    if (threadIdx.x == 0) pcg_start(S, rz, rr, A);
  } else {
    block_partials<kBS, 2>(v, partials);
  }
}

__global__ __launch_bounds__(kFinBS) void k_pcg_init_fin(KState* S, double* partials, int nb, PcgStart A) {
  double s[2];
  finalize_sums<2>(partials, nb, s);
  clear_resident_slots<kFinBS>(partials);
  if (threadIdx.x == 0) pcg_start(S, s[0], s[1], A);
}

template <class M, class T, int U, class C>
__global__ __launch_bounds__(kSpmvBS) void k_pcg_spmv(int64_t n, int64_t n_chunks, const int32_t* __restrict__ sptr,
                                                      const C* __restrict__ cols, const M* __restrict__ vals,
                                                      const T* __restrict__ z, T* __restrict__ pa, T* __restrict__ pb,
                                                      T* __restrict__ q, KState* S, double* partials) {
  if (halted(S)) return;
  constexpr int wpb = kSpmvBS / 64;
  const T beta = (T)S->beta;
  const bool odd = S->k & 1;
  const T* __restrict__ po = odd ? pb : pa;
  T* __restrict__ pn = odd ? pa : pb;
  const int lane = threadIdx.x & 63;
  double v[1] = {0.0};
  for (int64_t c = blockIdx.x * (int64_t)wpb + (threadIdx.x >> 6); c < n_chunks; c += (int64_t)gridDim.x * wpb) {
    const int32_t off = sptr[c], w = (sptr[c + 1] - off) >> 6;
    const int64_t row = c * 64 + lane;
    const T s = sell_row<M, T, U>(vals + off + lane, cols + off + lane, w, sell_base(row, n),
                                  [&](int32_t col) { return z[col] + beta * po[col]; });
    if (row < n) {
      const T pi = z[row] + beta * po[row];
      pn[row] = pi;
      q[row] = s;
      v[0] += (double)pi * (double)s;
    }
  }
  block_partials<kSpmvBS, 1>(v, partials);
}

// ---- PCG on a symmetric 9-point matrix ---------------------------------------------------
// Where the pattern is that of a 9-point stencil on lines of m rows (Plan::line) and A_ij and A_ji
// have the same bits, the streaming iterations read the matrix as its upper diagonals
// A[d][i] = A(i, i + o_d), o = 0, 1, m - 1, m, m + 1: five values a row and no columns.
//
// A wavefront owns up to 62 neighbouring rows on each of `lines` consecutive lines (lanes 0 and
// W + 1 hold the rows beside them) and walks down the lines: p of the line below is formed once
// and stays in registers for three lines, the values that couple a line to the one above are kept
// from that line, and neighbours within a line come from the lane beside (DPP).  Seven loads of
// 64 consecutive values a line, all issued a line ahead.  The matrix is read past the caches
// (non-temporal), which leaves them to the vectors: the update kernel after it 43.9 -> 41.4 us.
//
// Bound by HBM: at 2047^2 rows, FP64, 302 MB in 56.5 us (5.3 TB/s) against 512 MB in 109 us for
// k_pcg_spmv; with x's update 369 MB in 64.5 us (5.7 TB/s) and the update kernel 41.4 -> 26.1 us; the
// iteration 157 -> 104 us.  The same diagonals read without the walk (27 loads a
// row, neighbours' lines from L2) took 89 us.  Which rows form a line is arithmetic
// only: entries that a grid's end takes out of the pattern are stored zeros.  Rows of the chunks
// with entries elsewhere (Plan::irregular) are summed from the SELL values.
constexpr int kLineLanes = 62;
constexpr int kLineBS = 256;

struct LineGrid {
  int m;        // rows per line
  int width;    // rows per wavefront and line
  int segments; // wavefronts side by side on a line
  int lines;    // lines per wavefront
  int64_t tasks;
};

template <class T>
__device__ __forceinline__ T from_lane_below(T v) {  // lane i: lane i - 1's
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, false));
  } else {
    const int2 w = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(T, int2{__builtin_amdgcn_update_dpp(0, w.x, 0x138, 0xf, 0xf, false),
                                      __builtin_amdgcn_update_dpp(0, w.y, 0x138, 0xf, 0xf, false)});
  }
}
template <class T>
__device__ __forceinline__ T from_lane_above(T v) {  // lane i: lane i + 1's
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, false));
  } else {
    const int2 w = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(T, int2{__builtin_amdgcn_update_dpp(0, w.x, 0x130, 0xf, 0xf, false),
                                      __builtin_amdgcn_update_dpp(0, w.y, 0x130, 0xf, 0xf, false)});
  }
}

// The upper diagonals of a SELL matrix, zero where the pattern has no entry; clears the flag that
// k_lines_check sets.
template <class M, class C>
__global__ __launch_bounds__(kBS) void k_lines_from_sell(int64_t n, int m, const int32_t* __restrict__ indptr,
                                                         const int32_t* __restrict__ sptr, const C* __restrict__ cols,
                                                         const M* __restrict__ vals, M* __restrict__ A,
                                                         int* asymmetric) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *asymmetric = 0;
  const int o[5] = {0, 1, m - 1, m, m + 1};
  for (int64_t i = blockIdx.x * (int64_t)kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const int64_t at = sptr[i >> 6] + (i & 63);
    const int w = indptr[i + 1] - indptr[i];
    M a[5] = {};
    for (int k = 0; k < w; ++k) {
      const int off = sell_col(cols[at + k * 64], (int32_t)i) - (int32_t)i;
      const M v = vals[at + k * 64];
#pragma unroll
      for (int d = 0; d < 5; ++d)
        if (off == o[d]) a[d] = v;
    }
#pragma unroll
    for (int d = 0; d < 5; ++d) A[d * n + i] = a[d];
  }
}

// Sets the flag where an entry below the diagonal differs from its mirror image in any bit.
template <class M, class C>
__global__ __launch_bounds__(kBS) void k_lines_check(int64_t n, int m, const int32_t* __restrict__ indptr,
                                                     const int32_t* __restrict__ sptr, const C* __restrict__ cols,
                                                     const M* __restrict__ vals, const M* __restrict__ A,
                                                     int* asymmetric) {
  using B = std::conditional_t<sizeof(M) == 8, unsigned long long, unsigned>;
  const int o[5] = {0, 1, m - 1, m, m + 1};
  bool differs = false;
  for (int64_t i = blockIdx.x * (int64_t)kBS + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBS) {
    const int64_t at = sptr[i >> 6] + (i & 63);
    const int w = indptr[i + 1] - indptr[i];
    for (int k = 0; k < w; ++k) {
      const int col = sell_col(cols[at + k * 64], (int32_t)i);
      const M v = vals[at + k * 64];
      if (col >= i) break;  // columns ascend
#pragma unroll
      for (int d = 1; d < 5; ++d)
        if (i - col == o[d]) differs |= __builtin_bit_cast(B, A[d * n + col]) != __builtin_bit_cast(B, v);
    }
  }
  if (differs) *asymmetric = 1;
}

// DOT: flexible CG, which wants p.r (second partial) beside p.q.  Else the last iteration's x += alpha p
// is made up for here (where there was one since iteration k0), whose p is at hand: the update kernel
// then reads neither x nor p, 8 of an iteration's 136 bytes a row less in FP64.
template <class M, class T, class C, bool DOT>
__global__ __launch_bounds__(kLineBS) void k_pcg_lines(int64_t n, LineGrid L, const M* __restrict__ A,
                                                       const uint32_t* __restrict__ irregular,
                                                       const int32_t* __restrict__ sptr, const C* __restrict__ cols,
                                                       const M* __restrict__ vals, const T* __restrict__ z,
                                                       T* __restrict__ pa, T* __restrict__ pb, T* __restrict__ q,
                                                       const T* __restrict__ res, T* __restrict__ x, int k0, KState* S,
                                                       double* partials) {
  if (halted(S)) return;
  const T beta = (T)S->beta, alpha = (T)S->alpha;
  const bool odd = S->k & 1, behind = !DOT && S->k > k0;
  const T* __restrict__ po = odd ? pb : pa;
  T* __restrict__ pn = odd ? pa : pb;
  const int lane = threadIdx.x & 63, N = (int)n;
  const int64_t block = xcd_block(blockIdx.x, gridDim.x);
  const int64_t task = block * (kLineBS / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double v[DOT ? 2 : 1] = {};
  if (task < L.tasks) {
    const int seg = (int)(task % L.segments), l0 = (int)(task / L.segments) * L.lines;
    const int j0 = seg * L.width, width = min(L.width, L.m - j0);
    const bool mine = lane >= 1 && lane <= width;
    // the wave's rows on line l0; later lines may run past the last row
    int64_t first = (int64_t)l0 * L.m + j0;  // row of lane 1
    const int last = min(l0 + L.lines, (N + L.m - 1) / L.m);
    struct Line {
      T z, po, r, x;
      M d[5];
    } next;
    // row of this lane `lines` lines further on, or out of range
    auto at = [&](int lines) { return first + (int64_t)lines * L.m + lane - 1; };
    auto inside = [&](int64_t r) { return r >= 0 && r < n && lane <= width + 1; };
    auto load_p = [&](int lines) {
      const int64_t r = at(lines);
      next.z = next.po = T(0);
      if (inside(r)) {
        next.z = z[r];
        next.po = po[r];
      }
    };
    auto load_d = [&](int lines) {
      const int64_t r = at(lines);
#pragma unroll
      for (int d = 0; d < 5; ++d) next.d[d] = M(0);
      next.r = next.x = T(0);
      if (inside(r)) {
        if constexpr (DOT)
          next.r = res[r];
        else if (behind)
          next.x = x[r];
#pragma unroll
        for (int d = 0; d < 5; ++d) next.d[d] = __builtin_nontemporal_load(A + d * n + r);
      }
    };
    load_p(-1);
    T pm = next.z + beta * next.po;
    load_p(0);
    T pc = next.z + beta * next.po, poc = next.po;
    load_d(-1);
    T u2 = from_lane_above((T)next.d[2]), u3 = (T)next.d[3], u4 = from_lane_below((T)next.d[4]);
    load_p(1);
    load_d(0);
    T pmL = from_lane_below(pm), pmR = from_lane_above(pm), pcL = from_lane_below(pc), pcR = from_lane_above(pc);
    for (int l = l0; l < last; ++l, first += L.m) {
      const Line now = next;
      if (l + 1 < last) {
        load_p(2);
        load_d(1);
      }
      const T pd = now.z + beta * now.po;
      const T pdL = from_lane_below(pd), pdR = from_lane_above(pd);
      const T d1 = (T)now.d[1];
      T s = u4 * pmL;
      s += u3 * pm;
      s += u2 * pmR;
      s += from_lane_below(d1) * pcL;
      s += (T)now.d[0] * pc;
      s += d1 * pcR;
      s += (T)now.d[2] * pdL;
      s += (T)now.d[3] * pd;
      s += (T)now.d[4] * pdR;
      const int64_t row = first + lane - 1;
      if (first < n) {
        const int64_t c0 = first >> 6, c1 = min(first + width - 1, n - 1) >> 6;
        if (((irregular[c0 >> 5] >> (c0 & 31)) | (irregular[c1 >> 5] >> (c1 & 31))) & 1) {
          const int64_t c = row >> 6;
          if (mine && row < n && ((irregular[c >> 5] >> (c & 31)) & 1)) {
            const int32_t e = sptr[c] + (int32_t)(row & 63), w = (sptr[c + 1] - sptr[c]) >> 6;
            s = sell_row<M, T>(vals + e, cols + e, w, (int32_t)row, [&](int32_t col) { return z[col] + beta * po[col]; });
          }
        }
      }
      if (mine && row < n) {
        pn[row] = pc;
        q[row] = s;
        v[0] += (double)pc * (double)s;
        if constexpr (DOT)
          v[DOT] += (double)pc * (double)now.r;
        else if (behind)
          x[row] = now.x + alpha * poc;
      }
      poc = now.po;
      u2 = from_lane_above((T)now.d[2]);
      u3 = (T)now.d[3];
      u4 = from_lane_below((T)now.d[4]);
      pm = pc;
      pmL = pcL;
      pmR = pcR;
      pc = pd;
      pcL = pdL;
      pcR = pdR;
    }
  }
  block_partials_at<kLineBS, DOT ? 2 : 1>(v, partials, block);
}

__global__ __launch_bounds__(kFinBS) void k_pcg_alpha_fin(KState* S, const double* partials, int nb) {
  if (halted(S)) return;
  double tot[1];
  finalize_sums<1>(partials, nb, tot);
  if (threadIdx.x == 0) {
    S->pAp = tot[0];
    S->alpha = S->gamma / tot[0];
  }
}

// WITH_X: or the next k_pcg_lines (after the last iteration k_pcg_finish_x) adds alpha p to x.
template <class T, bool WITH_X>
__global__ __launch_bounds__(kBS) void k_pcg_update(int64_t n, const T* __restrict__ inv, const T* __restrict__ pa,
                                                    const T* __restrict__ pb, const T* __restrict__ q,
                                                    T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                    KState* S, double* partials) {
  if (halted(S)) return;
  const T alpha = (T)S->alpha;
  const T* __restrict__ p = (S->k & 1) ? pa : pb;  // written by k_pcg_spmv of this iteration
  double v[2] = {0.0, 0.0};
  T pv[kUnroll], qv[kUnroll], xv[kUnroll], rv[kUnroll], iv[kUnroll];
  APX_FOR_ELEMENTS(n, {
    if constexpr (WITH_X) {
      pv[j] = p[i];
      xv[j] = x[i];
    }
    qv[j] = q[i];
    rv[j] = r[i];
    iv[j] = inv[i];
  }, {
    if constexpr (WITH_X) x[i] = xv[j] + alpha * pv[j];
    const T ri = rv[j] - alpha * qv[j];
    const T zi = iv[j] * ri;
    r[i] = ri;
    z[i] = zi;
    v[0] += (double)ri * (double)zi;
    v[1] += (double)ri * (double)ri;
  })
  block_partials<kBS, 2>(v, partials);
}

__global__ __launch_bounds__(kFinBS) void k_pcg_beta_fin(KState* S, const double* partials, int nb) {
  if (halted(S)) return;
  double s[2];
  finalize_sums<2>(partials, nb, s);
  if (threadIdx.x == 0) {
    S->gamma_prev = S->gamma;
    S->beta = s[0] / S->gamma;
    S->gamma = s[0];
    S->rr = s[1];
    S->k += 1;
    S->done = !(s[1] > S->atol2 && S->k < S->maxiter);
    if (!S->done && S->delta2 > 0.0 && s[1] < S->delta2 * S->rmax2) S->reliable = 1;
  }
}

template <class T>
__global__ __launch_bounds__(kBS) void k_pcg_finish_x(int64_t n, const T* __restrict__ pa, const T* __restrict__ pb,
                                                      T* __restrict__ x, const KState* S) {
  const T alpha = (T)S->alpha;
  const T* __restrict__ p = ((S->k - 1) & 1) ? pa : pb;  // of the last iteration
  T pv[kUnroll], xv[kUnroll];
  APX_FOR_ELEMENTS(n, { pv[j] = p[i]; xv[j] = x[i]; }, { x[i] = xv[j] + alpha * pv[j]; })
}

// Replace the recursive residual by b_new = -r_full[free] (a true residual
// computed in FP64 by the caller) and zero the correction x; the direction p
// is kept (reliable update, Sleijpen & van der Vorst 1996).
template <class T>
__global__ __launch_bounds__(kBS) void k_pcg_reanchor(int64_t n, const int32_t* __restrict__ red2full,
                                                      const double* __restrict__ rfull, const T* __restrict__ inv,
                                                      T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                      KState* S, double* partials) {
  double v[2] = {0.0, 0.0};
  T rv[kUnroll], iv[kUnroll];
  APX_FOR_ELEMENTS(n, { rv[j] = (T)(-rfull[red2full[i]]); iv[j] = inv[i]; }, {
    const T zi = iv[j] * rv[j];
    x[i] = 0;
    r[i] = rv[j];
    z[i] = zi;
    v[0] += (double)rv[j] * (double)zi;
    v[1] += (double)rv[j] * (double)rv[j];
  })
  block_partials<kBS, 2>(v, partials);
}

// RESIDENT: the last run left its scalars with its slots, not in S (a copy behind every run would be 10 us).
template <bool RESIDENT>
__global__ __launch_bounds__(kFinBS) void k_pcg_reanchor_fin(KState* S, double* partials, int nb) {
  if constexpr (RESIDENT) {
    if (threadIdx.x == 0) *S = ((const ResidentOut*)(partials + kResidentSlotsAt + kResidentSlotWords))->state;
    __syncthreads();  // before they are cleared
  }
  double s[2];
  finalize_sums<2>(partials, nb, s);
  clear_resident_slots<kFinBS>(partials);
  if (threadIdx.x == 0) {
    S->beta = s[0] / S->gamma_prev;
    S->gamma = s[0];
    S->rr = s[1];
    S->rmax2 = s[1];
    S->reliable = 0;
    S->done = !(s[1] > S->atol2 && S->k < S->maxiter);
  }
}

// ---- PCG driver ----------------------------------------------------------------------
static bool is_idle(hipStream_t st) {
  if (hipStreamQuery(st) == hipSuccess) return true;
  (void)hipGetLastError();  // not ready
  return false;
}

template <class M, class T>
PcgRun<M, T>::PcgRun(Plan& P_, const M* vals_, const T* inv_, hipStream_t st_)
    : P(P_), vals(vals_), inv(inv_), st(st_) {
  n = P.n_free;
  T* w;
  if constexpr (sizeof(T) == 8) {
    if (P.w64.n < (size_t)(7 * n)) P.w64.alloc(7 * n);
    w = (T*)P.w64.p;
  } else {
    if (P.w32.n < (size_t)(7 * n)) P.w32.alloc(7 * n);
    w = (T*)P.w32.p;
  }
  // (w + 4 n: q, or the resident run's 2 n words)
  r = w; z = w + n; pa = w + 2 * n; pb = w + 3 * n; q = w + 4 * n; xw = w + 6 * n;
  ensure_krylov_scratch(P, st);
  S = (KState*)P.kstate.p;
  part = P.partials.p;
  // SELL values + columns (int16 offsets or int32), chunk offsets, z and p_old read, p_new and q written
  spmv_bytes = P.sell_total * (int64_t)(sizeof(M) + (P.sell_dcol.p ? 2 : 4)) + (P.n_chunks + 1) * 4 +
               n * 4 * (int64_t)sizeof(T);
  upd_bytes = n * 8 * (int64_t)sizeof(T);  // reads D^-1, p, q, x, r; writes x, r, z
}

template <class M, class T>
PcgRun<M, T>::PcgRun(Plan& P_, const M* vals_, const T* inv_, hipStream_t st_, T* w, double* partials, KState* state)
    : P(P_), vals(vals_), inv(inv_), st(st_), S(state), part(partials), external(true) {
  n = P.n_free;
  r = w; z = w + n; pa = w + 2 * n; pb = w + 3 * n; q = w + 4 * n;  // and a further n: the caller gives x
}

template <class M, class T>
PcgRun<M, T>::~PcgRun() {
  if (evs[0]) (void)hipEventDestroy(evs[0]);
  if (evs[1]) (void)hipEventDestroy(evs[1]);
}

template <class M, class T>
void PcgRun<M, T>::init(const T* b, const double* r_full, T* x_, double tol, double atol, int maxiter_, double delta) {
  x = x_ ? x_ : xw;
  start_k = 0;
  resident_last = false;
  upper = nullptr;  // the matrix may be another one
  upper_known = false;
  maxiter = maxiter_ <= 0 ? (int)std::min<int64_t>(10 * n, INT32_MAX / 2) : maxiter_;
  idle = is_idle(st);
  const PcgStart A{tol, atol, delta, maxiter};
  const int g = grid_for(n);
  auto start = [&](auto full, auto one) {
    hipLaunchKernelGGL((k_pcg_init<T, decltype(full)::value, decltype(one)::value>), dim3(g), dim3(kBS), 0, st, n, b,
                       P.red2full.p, r_full, inv, x, r, z, pa, S, part, A);
  };
  if (r_full)
    g == 1 ? start(std::true_type{}, std::true_type{}) : start(std::true_type{}, std::false_type{});
  else
    g == 1 ? start(std::false_type{}, std::true_type{}) : start(std::false_type{}, std::false_type{});
  if (g > 1) hipLaunchKernelGGL(k_pcg_init_fin, dim3(1), dim3(kFinBS), 0, st, S, part, g, A);
  APX_LAUNCH_CHECK();
}

// Lines per wavefront: 32 wavefronts a compute unit where there are that many, at least 8 lines (the
// lines above and below a wavefront's are read twice).  2047^2 rows, FP64: 17 lines (16 wavefronts)
// 62.3 us, 12 lines 59.0, 8 lines 56.9, 6 lines 55.9, 4 lines 55.2.
static LineGrid line_grid(const Plan& P) {
  LineGrid L;
  L.m = P.line;
  L.segments = (P.line + kLineLanes - 1) / kLineLanes;
  L.width = (P.line + L.segments - 1) / L.segments;
  const int64_t lines = (P.n_free + P.line - 1) / P.line, waves = 256 * 32;
  L.lines = (int)std::max<int64_t>(8, (lines * L.segments + waves - 1) / waves);
  L.tasks = (lines + L.lines - 1) / L.lines * L.segments;
  return L;
}
int line_blocks(const Plan& P) {
  constexpr int wpb = kLineBS / 64;
  return (int)round_xcd((line_grid(P).tasks + wpb - 1) / wpb);
}

// Lines of fewer than 32 rows would leave more than half of a wavefront's lanes idle, where it no longer
// pays (FP64, us an iteration: 557,973 rows in lines of 31, SELL kernel 35.1; 575,972 in lines of 32
// 34.8, of 64 31.5; 571,377 in lines of 127 29.6).  Lines of over two million rows would need more
// workgroups than a row of partial sums holds.  Systems that apx_pcg_noalloc takes keep the SELL kernel,
// whose sums it shares bit by bit, and where the launches' latency, not the bytes, sets the pace.
// Flexible CG has no allocation-free twin, but its break-even lies there too (a Newton solve with the
// network, FP64, by lines against SELL: 65^2 nodes 8.47 and 8.24 ms, 129^2 14.23 and 14.08, 257^2 25.7 and
// 25.1, 385^2 33.8 and 33.3, 513^2 46.5 and 46.3).
static bool lines_pay(const Plan& P, size_t value_bytes) {
  return P.line >= 32 && line_blocks(P) <= kMaxBlocks && !noalloc_accepts(P, value_bytes);
}

// The upper diagonals of a SELL matrix into the plan's buffer for them, and the flag P.asymmetric that
// tells whether they are not the whole of it (copied to the host with the first stop flags); null:
// another pattern, or no memory (the run then reads the SELL matrix).
template <class M>
const M* line_matrix(Plan& P, const M* vals, size_t vector_bytes, hipStream_t st) {
  if (!lines_pay(P, vector_bytes)) return nullptr;
  const int64_t n = P.n_free;
  const size_t want = (size_t)(5 * n);
  auto room = [&](auto& buf) { return buf.n >= want || buf.try_alloc(want); };
  M* A = nullptr;
  if constexpr (sizeof(M) == 8) {
    if (room(P.lines64)) A = P.lines64.p;
  } else {
    if (room(P.lines32)) A = P.lines32.p;
  }
  if (!A) return nullptr;
  if (!P.asymmetric.p) P.asymmetric.alloc(1);
  const int g = (int)std::min<int64_t>((n + kBS - 1) / kBS, 65536);
  auto run = [&](auto cols) {
    using C = std::remove_const_t<std::remove_pointer_t<decltype(cols)>>;
    hipLaunchKernelGGL((k_lines_from_sell<M, C>), dim3(g), dim3(kBS), 0, st, n, P.line, P.indptr.p, P.sell_ptr.p, cols,
                       vals, A, P.asymmetric.p);
    hipLaunchKernelGGL((k_lines_check<M, C>), dim3(g), dim3(kBS), 0, st, n, P.line, P.indptr.p, P.sell_ptr.p, cols,
                       vals, (const M*)A, P.asymmetric.p);
  };
  if (P.sell_dcol.p)
    run((const int16_t*)P.sell_dcol.p);
  else
    run((const int32_t*)P.sell_cols.p);
  APX_LAUNCH_CHECK();
  return A;
}
template const float* line_matrix<float>(Plan&, const float*, size_t, hipStream_t);
template const double* line_matrix<double>(Plan&, const double*, size_t, hipStream_t);

template <class M, class T>
void line_product(Plan& P, const M* upper, const M* vals, const T* z, T* pa, T* pb, T* q, const T* r, T* x, int k0,
                  KState* S, double* part, hipStream_t st) {
  auto run = [&](auto cols, auto dot) {
    using C = std::remove_const_t<std::remove_pointer_t<decltype(cols)>>;
    launch_kernel(k_pcg_lines<M, T, C, decltype(dot)::value>, dim3(line_blocks(P)), dim3(kLineBS), 0, st, P.n_free,
                  line_grid(P), upper, P.irregular.p, P.sell_ptr.p, cols, vals, z, pa, pb, q, r, x, k0, S, part);
  };
  auto with = [&](auto cols) { r ? run(cols, std::true_type{}) : run(cols, std::false_type{}); };
  if (P.sell_dcol.p)
    with((const int16_t*)P.sell_dcol.p);
  else
    with((const int32_t*)P.sell_cols.p);
}
template void line_product<double, double>(Plan&, const double*, const double*, const double*, double*, double*,
                                           double*, const double*, double*, int, KState*, double*, hipStream_t);
template void line_product<float, double>(Plan&, const float*, const float*, const double*, double*, double*, double*,
                                          const double*, double*, int, KState*, double*, hipStream_t);
template void line_product<float, float>(Plan&, const float*, const float*, const float*, float*, float*, float*,
                                         const float*, float*, int, KState*, double*, hipStream_t);

template <class M, class T>
void PcgRun<M, T>::launch_iteration() {
  const int gs = upper ? line_blocks(P) : grid_chunks(P.n_chunks), gu = grid_for(n);
  const bool timed = P.timing && !external;
  // timed: the pairs take the SpMV's and the update's own start and end timestamps
  const EventPair e1 = timed ? timing_pair(P) : EventPair{}, e2 = timed ? timing_pair(P) : EventPair{};
  t_launch_events = timed ? &e1 : nullptr;
  auto spmv = [&](auto cols) {
    using C = std::remove_const_t<std::remove_pointer_t<decltype(cols)>>;
    if (P.sell_total >= 32 * (int64_t)P.n_free)  // rows of 32+ stored entries: deeper load batches
      launch_kernel((k_pcg_spmv<M, T, 8, C>), dim3(gs), dim3(kSpmvBS), 0, st, n, P.n_chunks, P.sell_ptr.p, cols, vals,
                    z, pa, pb, q, S, part);
    else
      launch_kernel((k_pcg_spmv<M, T, 4, C>), dim3(gs), dim3(kSpmvBS), 0, st, n, P.n_chunks, P.sell_ptr.p, cols, vals,
                    z, pa, pb, q, S, part);
  };
  if (upper)
    line_product<M, T>(P, upper, vals, z, pa, pb, q, nullptr, x, k0, S, part, st);
  else if (P.sell_dcol.p)
    spmv((const int16_t*)P.sell_dcol.p);
  else
    spmv((const int32_t*)P.sell_cols.p);
  hipLaunchKernelGGL(k_pcg_alpha_fin, dim3(1), dim3(kFinBS), 0, st, S, part, gs);
  t_launch_events = timed ? &e2 : nullptr;
  if (upper)
    launch_kernel(k_pcg_update<T, false>, dim3(gu), dim3(kBS), 0, st, n, inv, pa, pb, q, x, r, z, S, part);
  else
    launch_kernel(k_pcg_update<T, true>, dim3(gu), dim3(kBS), 0, st, n, inv, pa, pb, q, x, r, z, S, part);
  hipLaunchKernelGGL(k_pcg_beta_fin, dim3(1), dim3(kFinBS), 0, st, S, part, gu);
  if (timed) {
    ev_spmv.push_back(e1);
    ev_upd.push_back(e2);
  }
}

template <class M, class T>
KState PcgRun<M, T>::run() {
  {
    // in one launch where the system fits on the compute units (resident.hip)
    static_assert(sizeof(ResidentOut) <= 256, "ResidentOut must fit its pinned slot");
    KState* pinned_state = (KState*)((char*)P.pinned + 768);  // pinned bytes 768..1023
    const bool odd = start_k & 1;
    const bool timed = P.timing && !external;
    const EventPair e = timed ? timing_pair(P) : EventPair{};
    t_launch_events = timed ? &e : nullptr;
    const bool ran = !streaming && pcg_resident<M, T>(P, vals, inv, x, r, z, odd ? pb : pa, odd ? pa : pb,
                                                      (unsigned long long*)q, S, part, pinned_state, idle, st);
    if (timed && !t_launch_events)
      (ran ? ev_res : ev_given_up).push_back(e);
    else if (timed)
      P.evpool.insert(P.evpool.end(), {e.a, e.b});
    t_launch_events = nullptr;
    if (ran) {
      iterations = pinned_state->k;
      resident_last = true;
      // the last direction was written beside p_old; iteration k reads it from pb (k odd) or pa
      if (iterations != start_k && ((iterations ^ start_k) & 1) == 0) std::swap(pa, pb);
      start_k = iterations;
      return *pinned_state;
    }
    streaming = true;
    resident_last = false;
  }
  if (!external && !evs[0]) {
    APX_HIP(hipEventCreateWithFlags(&evs[0], hipEventDisableTiming));
    APX_HIP(hipEventCreateWithFlags(&evs[1], hipEventDisableTiming));
  }
  constexpr int kBatch = 16;
  volatile int* flag = (volatile int*)P.pinned;  // [slot*4 + {k, maxiter, done, reliable}]
  auto enqueue_batch = [&](int slot) {
    for (int i = 0; i < kBatch; ++i) launch_iteration();
    APX_LAUNCH_CHECK();
    APX_HIP(hipMemcpyAsync((void*)(flag + 4 * slot), &S->k, 4 * sizeof(int), hipMemcpyDeviceToHost, st));
    APX_HIP(hipEventRecord(evs[slot], st));
    launched += kBatch;
  };
  auto halted_host = [&](int slot) { return flag[4 * slot + 2] != 0 || flag[4 * slot + 3] != 0; };
  // flags after init / reanchor
  if (!upper_known && !external) upper = line_matrix<M>(P, vals, sizeof(T), st);
  const bool extracted = !upper_known && upper;
  if (extracted) APX_HIP(hipMemcpyAsync((void*)(flag + 12), P.asymmetric.p, sizeof(int), hipMemcpyDeviceToHost, st));
  APX_HIP(hipMemcpyAsync((void*)(flag + 8), &S->k, 4 * sizeof(int), hipMemcpyDeviceToHost, st));
  APX_HIP(hipStreamSynchronize(st));
  if (extracted && flag[12]) upper = nullptr;
  upper_known = true;
  k0 = flag[8];
  if (external && !halted_host(2)) {
    // no events: enqueue a batch, copy the flags, wait for the stream, test
    const int64_t limit = (int64_t)launched + maxiter + kBatch;
    for (;;) {
      for (int i = 0; i < kBatch; ++i) launch_iteration();
      APX_LAUNCH_CHECK();
      launched += kBatch;
      APX_HIP(hipMemcpyAsync((void*)flag, &S->k, 4 * sizeof(int), hipMemcpyDeviceToHost, st));
      APX_HIP(hipStreamSynchronize(st));
      if (halted_host(0) || launched >= limit) break;
    }
  } else if (!halted_host(2)) {
    const int64_t limit = (int64_t)launched + maxiter + 2 * kBatch;
    enqueue_batch(0);
    int slot = 0;
    for (;;) {
      enqueue_batch(slot ^ 1);
      APX_HIP(hipEventSynchronize(evs[slot]));
      if (halted_host(slot) || launched >= limit) break;
      slot ^= 1;
    }
  }
  KState hs;
  if (external) {
    // through the plan's pinned block (bytes 768..1023), so no pageable staging is involved
    char* slot = (char*)P.pinned + 768;
    APX_HIP(hipMemcpyAsync(slot, S, sizeof(KState), hipMemcpyDeviceToHost, st));
    APX_HIP(hipStreamSynchronize(st));
    std::memcpy(&hs, slot, sizeof(KState));
  } else {
    APX_HIP(hipStreamSynchronize(st));
    APX_HIP(hipMemcpy(&hs, S, sizeof(KState), hipMemcpyDeviceToHost));
    if (upper && hs.k > k0) {
      hipLaunchKernelGGL(k_pcg_finish_x<T>, dim3(grid_for(n)), dim3(kBS), 0, st, n, pa, pb, x, S);
      APX_LAUNCH_CHECK();
      APX_HIP(hipStreamSynchronize(st));  // x is complete on return, on whatever stream it is read
    }
  }
  iterations = hs.k;
  return hs;
}

template <class M, class T>
void PcgRun<M, T>::reanchor(const double* r_full) {
  idle = is_idle(st);
  const int g = grid_for(n);
  hipLaunchKernelGGL(k_pcg_reanchor<T>, dim3(g), dim3(kBS), 0, st, n, P.red2full.p, r_full, inv, x, r, z, S, part);
  if (resident_last)
    hipLaunchKernelGGL(k_pcg_reanchor_fin<true>, dim3(1), dim3(kFinBS), 0, st, S, part, g);
  else
    hipLaunchKernelGGL(k_pcg_reanchor_fin<false>, dim3(1), dim3(kFinBS), 0, st, S, part, g);
  APX_LAUNCH_CHECK();
}

template <class M, class T>
void PcgRun<M, T>::collect_timing() {
  if (!P.timing || external) return;
  const bool f64 = sizeof(T) == 8;
  // only launches that executed an iteration are counted; the rest exited at entry
  const size_t k = (size_t)iterations - counted;
  // by lines: the upper values; z, p_old and x read, p_new, q and x written; D^-1, q, r read, r, z written
  const int64_t line_bytes = n * (5 * (int64_t)sizeof(M) + 6 * (int64_t)sizeof(T));
  timing_collect(P, sizeof(M) == sizeof(T) ? (f64 ? "pcg_spmv_f64" : "pcg_spmv_f32") : "pcg_spmv_f32m_f64v", ev_spmv,
                 upper ? line_bytes : spmv_bytes, k);
  timing_collect(P, f64 ? "pcg_update_f64" : "pcg_update_f32", ev_upd, upper ? n * 5 * (int64_t)sizeof(T) : upd_bytes, k);
  timing_collect(P, f64 ? "pcg_resident_f64" : "pcg_resident_f32", ev_res, 0, ev_res.size());
  timing_collect(P, "pcg_resident_given_up", ev_given_up, 0, ev_given_up.size());
  counted = iterations;
}

template struct PcgRun<double>;
template struct PcgRun<float>;
template struct PcgRun<float, double>;

template <class T>
static apx_krylov_stats pcg_t(Plan& P, const T* vals, const T* inv, const T* b, T* x, double tol, double atol,
                              int maxiter, hipStream_t st) {
  auto t0 = std::chrono::steady_clock::now();
  PcgRun<T> run(P, vals, inv, st);
  run.init(b, nullptr, x, tol, atol, maxiter, 0.0);
  KState hs = run.run();
  run.collect_timing();
  apx_krylov_stats out{};
  out.iterations = hs.k;
  out.converged = hs.rr <= hs.atol2;
  out.initial_residual = sqrt(hs.rr0);
  out.final_residual = sqrt(hs.rr);
  out.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return out;
}

apx_krylov_stats pcg(Plan& P, const void* vals, const void* inv, const void* b, void* x, int precision, double tol,
                     double atol, int maxiter, hipStream_t st) {
  if (precision == APX_FP64)
    return pcg_t<double>(P, (const double*)vals, (const double*)inv, (const double*)b, (double*)x, tol, atol,
                         maxiter, st);
  return pcg_t<float>(P, (const float*)vals, (const float*)inv, (const float*)b, (float*)x, tol, atol, maxiter, st);
}

// ---- Newton helpers -----------------------------------------------------------------
// The norm goes to the host's pinned word by the kernel itself (a copy behind it took 6 us).  ONE:
// one block, which finishes the sum.
template <bool ONE>
__global__ __launch_bounds__(kBS) void k_free_norm(int64_t n, const int32_t* red2full, const double* r, double* host,
                                                   double* partials) {
  double v[1] = {0.0};
  double rv[kUnroll];
  APX_FOR_ELEMENTS(n, { rv[j] = r[red2full[i]]; }, { v[0] += rv[j] * rv[j]; })
  if constexpr (ONE) {
    __shared__ double lds[kBS / 64];
    const double s = block_sum<kBS>(v[0], lds);
    if (threadIdx.x == 0) *host = sqrt(s);
  } else {
    block_partials<kBS, 1>(v, partials);
  }
}

__global__ __launch_bounds__(kFinBS) void k_norm_fin(double* host, const double* partials, int nb) {
  double s[1];
  finalize_sums<1>(partials, nb, s);
  if (threadIdx.x == 0) *host = sqrt(s[0]);
}

double free_norm(Plan& P, const double* r_full, hipStream_t st) {
  ensure_krylov_scratch(P, st);
  double* host = P.pinned + 16;
  const int g = grid_for(P.n_free);
  if (g == 1) {
    hipLaunchKernelGGL(k_free_norm<true>, dim3(1), dim3(kBS), 0, st, P.n_free, P.red2full.p, r_full, host,
                       P.partials.p);
  } else {
    hipLaunchKernelGGL(k_free_norm<false>, dim3(g), dim3(kBS), 0, st, P.n_free, P.red2full.p, r_full, host,
                       P.partials.p);
    hipLaunchKernelGGL(k_norm_fin, dim3(1), dim3(kFinBS), 0, st, host, (const double*)P.partials.p, g);
  }
  APX_LAUNCH_CHECK();
  APX_HIP(hipStreamSynchronize(st));
  return *(volatile double*)host;
}
__global__ void k_gather_rhs(int64_t n, const int32_t* red2full, const double* r, double* b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    b[i] = -r[red2full[i]];
}
void gather_rhs(Plan& P, const double* r_full, double* b, hipStream_t st) {
  const int g = std::max(1, (int)std::min<int64_t>((P.n_free + 255) / 256, 65536));
  hipLaunchKernelGGL(k_gather_rhs, dim3(g), dim3(256), 0, st, P.n_free, P.red2full.p, r_full, b);
  APX_LAUNCH_CHECK();
}

template <class T>
__global__ void k_scatter_update(int64_t n, const int32_t* red2full, double* u, const T* x, double damping) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    u[red2full[i]] += damping * (double)x[i];
}

void scatter_update(Plan& P, double* u, const void* x, double damping, int precision, hipStream_t st) {
  const int g = std::max(1, (int)std::min<int64_t>((P.n_free + 255) / 256, 65536));
  if (precision == APX_FP64)
    hipLaunchKernelGGL(k_scatter_update<double>, dim3(g), dim3(256), 0, st, P.n_free, P.red2full.p, u,
                       (const double*)x, damping);
  else
    hipLaunchKernelGGL(k_scatter_update<float>, dim3(g), dim3(256), 0, st, P.n_free, P.red2full.p, u,
                       (const float*)x, damping);
  APX_LAUNCH_CHECK();
}

__global__ void k_impose(int64_t n, const uint8_t* mask, double* u, const double* vals) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (mask[i]) u[i] = vals[i];
}

void impose_dirichlet(Plan& P, double* u, const double* values, hipStream_t st) {
  const int g = std::max(1, (int)std::min<int64_t>((P.n_dofs + 255) / 256, 65536));
  hipLaunchKernelGGL(k_impose, dim3(g), dim3(256), 0, st, P.n_dofs, P.dmask.p, u, values);
  APX_LAUNCH_CHECK();
}

}  // namespace apx
