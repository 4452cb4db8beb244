// Row-owner assembly for meshes without the owner-tile kernels (structured.hip): Hex8 bricks,
// plane-strain and Q2 elements, unstructured Q1 grids.
//
// Tangent.  One launch forms the element matrices, each once, into a scratch array; a second one
// forms the rows: a workgroup owns one 64-row chunk of the reduced matrix (the chunk of the SELL layout),
// adds the blocks K_ab of its row nodes a into LDS, in element order, and writes every stored entry
// once, coalesced, in SELL or canonical CSR order.  No colours, no read-modify-write of memory, no
// slot per element entry.  The matrices travel through memory (half of each: they are symmetric); that
// and the FP64 arithmetic of the element kernel are the bounds.
//
// Residual.  One launch forms all element vectors from r_a = sum_q S_q dN_a(q) - f_q N_a(q) (S_q: the
// first Piola-Kirchhoff stress, or k grad u, pulled back by w det J J^-T), element by element into
// a scratch array; a second one adds up every node's elements in element order.
//
// Measured on an MI355X (kernel trace), before with one launch per colour and a slot per element
// entry, and a pass from the SELL to the CSR order:
//   64^3 Hex8 Neo-Hooke, CSR tangent (63.3 M entries): 4,720 us -> 329 (755 MB of blocks written at
//     2.3 TB/s; LDS reads of the gradients and FP64 arithmetic bound it) + 464 (1.01 GB read, 0.5
//     written, 3.2 TB/s; three workgroups of 41 KB of rows per compute unit leave latency open);
//     residual 277 -> 56 + 37
//   512^2 plane-strain quads, CSR tangent: 263 us -> 38 + 38
// Tried and slower: the rows formed straight from the gradients, each element evaluated by all the
// chunks it touches (2,490 and 103 us); eight elements' blocks in flight per lane instead of four
// (556 against 464 us, fewer wavefronts fit); blocks brought in through LDS so that every load
// reads whole lines (1,150 us); row-major element matrices (578 us, without the symmetry).
//
// Both are bitwise reproducible.  Replaces jacfwd(jacrev) and the scatter of
// user_potential_assemble_tangent / _residual (autopdex/assembler.py:1064-1149).
#include <algorithm>
#include <type_traits>

#include "assembly.hpp"
#include "elements.hpp"

namespace apx {

namespace {
// columns of a chunk's rows formed at a time: 64 x 255 FP64 words of LDS
constexpr int kRowWindow = 254;

// gradients of the shape functions at every Gauss point, filled into LDS by the first threads
template <class M>
__device__ inline void fill_gradients(double* dn /* NQ x NPE x DIM */, double* n /* NQ x NPE or null */) {
  for (int q = threadIdx.x; q < M::NQ; q += blockDim.x) {
    double N[M::NPE], dN[M::NPE][M::DIM];
    Shape<M::NPE, M::DIM>::eval(q, N, dN);
#pragma unroll
    for (int a = 0; a < M::NPE; ++a) {
      if (n) n[q * M::NPE + a] = N[a];
#pragma unroll
      for (int j = 0; j < M::DIM; ++j) dn[(q * M::NPE + a) * M::DIM + j] = dN[a][j];
    }
  }
}

template <int DIM>
__device__ __forceinline__ double inverse(const double (&J)[DIM][DIM], double (&Ji)[DIM][DIM]) {
  if constexpr (DIM == 2) {
    const double det = J[0][0] * J[1][1] - J[0][1] * J[1][0], id = 1.0 / det;
    Ji[0][0] = J[1][1] * id;
    Ji[0][1] = -J[0][1] * id;
    Ji[1][0] = -J[1][0] * id;
    Ji[1][1] = J[0][0] * id;
    return det;
  } else {
    const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const double c01 = J[0][2] * J[2][1] - J[0][1] * J[2][2];
    const double c02 = J[0][1] * J[1][2] - J[0][2] * J[1][1];
    const double det = J[0][0] * c00 + J[1][0] * c01 + J[2][0] * c02, id = 1.0 / det;
    Ji[0][0] = c00 * id;
    Ji[0][1] = c01 * id;
    Ji[0][2] = c02 * id;
    Ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * id;
    Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    Ji[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * id;
    Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    return det;
  }
}

template <int DIM>
__device__ __forceinline__ void product(const double (&A)[DIM][DIM], const double (&B)[DIM][DIM], double (&C)[DIM][DIM]) {
#pragma unroll
  for (int i = 0; i < DIM; ++i)
#pragma unroll
    for (int j = 0; j < DIM; ++j) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) s += A[i][k] * B[k][j];
      C[i][j] = s;
    }
}

// gradient with respect to the reference coordinates, D components: sum_a f_a dN_a
template <int NPE, int D, int DIM, class F>
__device__ __forceinline__ void reference_gradient(const double* dn, F f, double (&g)[D][DIM]) {
#pragma unroll
  for (int i = 0; i < D; ++i)
#pragma unroll
    for (int j = 0; j < DIM; ++j) g[i][j] = 0.0;
#pragma unroll
  for (int a = 0; a < NPE; ++a)
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const double v = f(a, i);
#pragma unroll
      for (int j = 0; j < DIM; ++j) g[i][j] += v * dn[a * DIM + j];
    }
}

// What the tangent needs per model.  NG: doubles of geometry per Gauss point (J^-1, for elasticity
// F^-1, then NS scalars); PB: gradient components per node.
template <class M>
struct RowModel;  // geometry(q, dn, n, x(a, i), u(a, i), field(a), params, out); row(scalars, a).add(b, block)

template <int NPE, int DIM>
struct RowModel<NeoHooke<NPE, DIM>> {
  static constexpr int NS = 3, NG = 2 * DIM * DIM + NS, PB = 2 * DIM;
  template <class X, class U, class G>
  __device__ static void geometry(int q, const double* dn, const double*, X x, U u, G, const ModelParams& p, double* out) {
    double J[DIM][DIM], U0[DIM][DIM], Ji[DIM][DIM], F[DIM][DIM], Fi[DIM][DIM];
    reference_gradient<NPE, DIM, DIM>(dn, x, J);
    reference_gradient<NPE, DIM, DIM>(dn, u, U0);
    const double w = Shape<NPE, DIM>::weight(q) * inverse<DIM>(J, Ji);
    product<DIM>(U0, Ji, F);
#pragma unroll
    for (int i = 0; i < DIM; ++i) F[i][i] += 1.0;
    const double det = inverse<DIM>(F, Fi), lam = p.p[0], mu = p.p[1];
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) {
        out[i * DIM + j] = Ji[i][j];
        out[(DIM + i) * DIM + j] = Fi[i][j];
      }
    out[2 * DIM * DIM] = w * mu;
    out[2 * DIM * DIM + 1] = w * (mu - 0.5 * lam * (det * det - 1.0));
    out[2 * DIM * DIM + 2] = w * (lam * det * det);
  }
  // block K_ab += mu G_a.G_b d_ik + c1 H_ak H_bi + c2 H_ai H_bk, the weight in the scalars
  template <class T>
  struct Row {
    T g[DIM], h1[DIM], h2[DIM];
    __device__ __forceinline__ void add(const T* b, T (&k)[DIM * DIM]) const {
      T gg = 0;
#pragma unroll
      for (int j = 0; j < DIM; ++j) gg += g[j] * b[j];
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        k[i * DIM + i] += gg;
#pragma unroll
        for (int j = 0; j < DIM; ++j) k[i * DIM + j] += h1[j] * b[DIM + i] + h2[i] * b[DIM + j];
      }
    }
  };
  template <class T>
  __device__ static __forceinline__ Row<T> row(const T* s, const T* a) {
    Row<T> r;
#pragma unroll
    for (int j = 0; j < DIM; ++j) {
      r.g[j] = s[0] * a[j];
      r.h1[j] = s[1] * a[DIM + j];
      r.h2[j] = s[2] * a[DIM + j];
    }
    return r;
  }
};

template <int NPE, int DIM, bool VARK>
struct RowPoisson {
  static constexpr int NS = 1, NG = DIM * DIM + NS, PB = DIM;
  template <class X, class U, class G>
  __device__ static void geometry(int q, const double* dn, const double* n, X x, U, G g, const ModelParams&, double* out) {
    double J[DIM][DIM], Ji[DIM][DIM];
    reference_gradient<NPE, DIM, DIM>(dn, x, J);
    double w = Shape<NPE, DIM>::weight(q) * inverse<DIM>(J, Ji);
    if constexpr (VARK) {
      double e = 0.0;
#pragma unroll
      for (int a = 0; a < NPE; ++a) e += n[a] * g(a);
      w *= exp(e);
    }
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) out[i * DIM + j] = Ji[i][j];
    out[DIM * DIM] = w;
  }
  template <class T>
  struct Row {
    T g[DIM];
    __device__ __forceinline__ void add(const T* b, T (&k)[1]) const {
#pragma unroll
      for (int j = 0; j < DIM; ++j) k[0] += g[j] * b[j];
    }
  };
  template <class T>
  __device__ static __forceinline__ Row<T> row(const T* s, const T* a) {
    Row<T> r;
#pragma unroll
    for (int j = 0; j < DIM; ++j) r.g[j] = s[0] * a[j];
    return r;
  }
};
template <int NPE, int DIM>
struct RowModel<PoissonSource<NPE, DIM>> : RowPoisson<NPE, DIM, false> {};
template <int NPE, int DIM>
struct RowModel<PoissonVarK<NPE, DIM>> : RowPoisson<NPE, DIM, true> {};

// The tangents are symmetric: of each pair K_ab = K_ba^T one block is formed and stored, K_a,a+d
// (indices modulo NPE) for d = 0 .. NPE / 2, so every thread forms as many.
template <int NPE>
constexpr int kBlocks = NPE / 2 + 1;
// whether K_ab is the stored one, and the plane of the stored one
template <int NPE>
__device__ __forceinline__ bool stored_block(int a, int b, int& plane) {
  const int d = b >= a ? b - a : b - a + NPE;
  const bool own = 2 * d < NPE || (2 * d == NPE && a < b);
  plane = own ? a * kBlocks<NPE> + d : b * kBlocks<NPE> + (NPE - d);
  return own;
}

// Element matrices in planes (a, d), each (element, i, k): a run of nodes along a grid line reads, per
// element around them and neighbour, one contiguous run.  Thread (element, t) evaluates Gauss point t --
// geometry, then the gradients of all nodes into LDS -- and after that keeps the blocks of node t in
// registers (as many Gauss points as nodes in every model).  T: arithmetic and accumulation of the
// blocks (the geometry is FP64).
template <class M>
__host__ __device__ constexpr int elements_per_block() {
  return (M::NPE == 8 ? 64 : 128) / M::NPE;  // Hex8: 26 KB of gradients per wavefront
}
// Where element le's gradients begin.  The lanes of a half-wavefront read node b of Gauss point q of
// their element: 4 or 8 elements whose starts, apart by multiples of 32 words, are shifted by the
// words that the nodes' strides (6 and 4 words) leave free, so that the 64 LDS banks do not conflict
// (without the shifts half of the LDS cycles were conflicts; 64^3 Hex8 elements 347 -> 329 us,
// 512^2 plane-strain quads 46 -> 38 us).
template <int NPE>
__device__ __forceinline__ int gradient_shift(int le) {
  return NPE == 8 ? (le & 1) + ((le & 2) << 3) + ((le >> 2) << 5) : NPE == 4 ? (le & 3) + ((le & 4) << 2) : 0;
}

template <class M, class T>
__global__ __launch_bounds__(elements_per_block<M>() * M::NPE) void k_element_matrices(
    const int32_t* __restrict__ conn, int64_t n_elems, const double* __restrict__ coords, int64_t n_nodes,
    const double* __restrict__ u, ModelParams mp, T* __restrict__ out) {
  using R = RowModel<M>;
  constexpr int NPE = M::NPE, DIM = M::DIM, D = M::D, NQ = M::NQ, NS = R::NS, NG = R::NG, PB = R::PB;
  constexpr int EPB = elements_per_block<M>(), GS = (NPE * PB + NS) | 1, NB = kBlocks<NPE>, KB = D * D;
  constexpr bool USES_U = NS == 3;
  static_assert(NQ == NPE, "one thread per Gauss point and per node");
  __shared__ double dn[NQ * NPE * DIM], sn[NQ * NPE];
  __shared__ double xs[EPB][NPE][DIM], us[USES_U ? EPB : 1][NPE][D], gs[M::NODAL ? EPB : 1][NPE];
  // words per element (Hex8 elasticity: 416, its shifts of up to 17 words run into the next element's)
  constexpr int ES = NPE == 9 ? NQ * GS : NPE == 8 ? (NQ * GS + 31) / 32 * 32 : (NQ * GS + 19 + 31) / 32 * 32;
  static_assert(NPE != 8 || NQ * GS <= ES - 8, "the fourth element of a group ends before the next group");
  __shared__ T gh[EPB * ES + 49];
  const int le = threadIdx.x / NPE, t = threadIdx.x % NPE;
  const int64_t e = blockIdx.x * (int64_t)EPB + le;
  const bool on = e < n_elems;
  fill_gradients<M>(dn, sn);
  if (on) {
    const int32_t node = conn[e * NPE + t];
#pragma unroll
    for (int k = 0; k < DIM; ++k) xs[le][t][k] = coords[k * n_nodes + node];
    if constexpr (USES_U) {
#pragma unroll
      for (int i = 0; i < D; ++i) us[le][t][i] = u[(int64_t)node * D + i];
    }
    if constexpr (M::NODAL) gs[le][t] = mp.nodal[0][node];
  }
  __syncthreads();
  if (on) {
    double geo[NG];
    R::geometry(
        t, dn + t * NPE * DIM, sn + t * NPE, [&](int a, int i) { return xs[le][a][i]; },
        [&](int a, int i) { return us[USES_U ? le : 0][a][i]; }, [&](int a) { return gs[M::NODAL ? le : 0][a]; }, mp,
        geo);
    T* g = gh + le * ES + gradient_shift<NPE>(le) + t * GS;
    for (int a = 0; a < NPE; ++a) {
      double from[DIM];  // dN, then G = dN J^-1, then H = G F^-1
#pragma unroll
      for (int j = 0; j < DIM; ++j) from[j] = dn[(t * NPE + a) * DIM + j];
#pragma unroll
      for (int p = 0; p < PB / DIM; ++p) {
        double to[DIM];
#pragma unroll
        for (int k = 0; k < DIM; ++k) {
          to[k] = 0.0;
#pragma unroll
          for (int j = 0; j < DIM; ++j) to[k] += from[j] * geo[(p * DIM + j) * DIM + k];
          g[a * PB + p * DIM + k] = (T)to[k];
        }
#pragma unroll
        for (int j = 0; j < DIM; ++j) from[j] = to[j];
      }
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) g[NPE * PB + i] = (T)geo[NG - NS + i];
  }
  __syncthreads();
  T k[NB][KB];
#pragma unroll
  for (int d = 0; d < NB; ++d)
#pragma unroll
    for (int i = 0; i < KB; ++i) k[d][i] = 0;
#pragma unroll 1
  for (int q = 0; q < NQ; ++q) {
    const T* g = gh + le * ES + gradient_shift<NPE>(le) + q * GS;
    T s[NS], ga[PB];
#pragma unroll
    for (int i = 0; i < NS; ++i) s[i] = g[NPE * PB + i];
#pragma unroll
    for (int i = 0; i < PB; ++i) ga[i] = g[t * PB + i];
    const auto row = R::template row<T>(s, ga);
#pragma unroll
    for (int d = 0; d < NB; ++d) {
      const int b = t + d < NPE ? t + d : t + d - NPE;
      T gb[PB];
#pragma unroll
      for (int i = 0; i < PB; ++i) gb[i] = g[b * PB + i];
      row.add(gb, k[d]);
    }
  }
  // block d of every node through LDS, over the gradients, where it lies as in the planes: their
  // runs of this workgroup leave coalesced
  constexpr int BS = EPB * NPE, RUN = EPB * KB;  // RUN: words of a full run; KB words per thread and d
  static_assert(BS * KB <= EPB * ES, "the blocks fit over the gradients");
  T* stage = gh;
  const int64_t e0 = blockIdx.x * (int64_t)EPB, plane = n_elems * KB;
  const int run = (int)min((int64_t)EPB, n_elems - e0) * KB;
  T* to[KB];  // where the words threadIdx.x + i BS of d = 0 go, null: past the last element
  bool half[KB];
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int c = threadIdx.x + i * BS, a = c / RUN, r = c % RUN;
    to[i] = r < run ? out + (int64_t)a * NB * plane + e0 * KB + r : nullptr;
    half[i] = a < NPE / 2;
  }
#pragma unroll
  for (int d = 0; d < NB; ++d) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KB; ++i) stage[(t * EPB + le) * KB + i] = k[d][i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KB; ++i)
      if (to[i] && (2 * d < NPE || half[i])) to[i][d * plane] = stage[threadIdx.x + i * BS];
  }
}

struct RowArgs {
  const int32_t* rn_ptr;          // the chunk's row nodes
  const int32_t* rn;              // per row node: its pairs' range in inc, its first DOF
  const int32_t* inc;             // (element * NPE + local index), in element order
  const void* code;               // per such pair and element node: where its columns lie in the row
  const int32_t *full2red, *indptr, *sell_ptr;
  int n_free, stride;             // stride: words per row of the LDS rows
  int window;                     // columns formed at a time
  int max_row;
  int accumulate;                 // add to the stored values (a plan's second and further sets)
  int64_t n_elems;
  const void* matrices;
  void* vals;
};

// Rows of one chunk.  Lane (row node, b) adds the blocks K_ab of that node's elements one after the
// other: within a step no two lanes of a wavefront touch the same entry, and a row belongs to one
// wavefront, so LDS needs no ordering beyond the wavefront's own.  T: type of the element matrices and
// of the sums, TO: of the stored values, C: of the codes (32 bits where a row has over 8,192 entries).
template <int NPE, int D, class T, class TO, bool CSR, class C>
__global__ __launch_bounds__(256) void k_gather_rows(RowArgs A) {
  constexpr int NPW = 64 / NPE, KB = D * D, BATCH = 4, BITS = sizeof(C) == 2 ? 13 : 29;
  extern __shared__ __align__(16) double lds[];
  T* rows = (T*)lds;
  __shared__ int ptr[65];
  const int c = (int)xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x, TB = blockDim.x, NW = TB >> 6, w = tid >> 6, lane = tid & 63;
  const int r0 = c * 64;
  if (r0 >= A.n_free) return;  // the whole workgroup
  const int rn0 = A.rn_ptr[c], nrn = A.rn_ptr[c + 1] - rn0;
  TO* vals = (TO*)A.vals;
  if constexpr (CSR) {
    for (int t = tid; t < 65; t += TB) ptr[t] = A.indptr[min(r0 + t, A.n_free)];
  }
  for (int win = 0; win == 0 || win < A.max_row; win += A.window) {
    // rows of up to 32 entries: two of them per wavefront in the CSR order
    const int per = A.stride > 33 ? 64 : 32;
    const int off = CSR ? 0 : A.sell_ptr[c], width = CSR ? 0 : (A.sell_ptr[c + 1] - off) >> 6;
    auto entries = [&](auto f) {  // f(LDS word, stored position) over the stored entries of this window
      if constexpr (CSR) {
        for (int row = tid / per; row < 64 && r0 + row < A.n_free; row += TB / per) {
          const int p0 = ptr[row], len = min(ptr[row + 1] - p0, win + A.window);
          for (int e = win + tid % per; e < len; e += per) f(row * A.stride + e - win, p0 + e);
        }
      } else {
        for (int e = win + w; e < min(width, win + A.window); e += NW) f(lane * A.stride + e - win, off + e * 64 + lane);
      }
    };
    for (int t = tid; t < 64 * A.stride; t += TB) rows[t] = 0;
    __syncthreads();
    if (A.accumulate) {
      entries([&](int l, int64_t g) { rows[l] = (T)vals[g]; });
      __syncthreads();
    }
    for (int l0 = w * NPW; l0 < nrn; l0 += NW * NPW) {
      const int ln = l0 + lane / NPE, b = lane % NPE;
      const bool on = lane < NPW * NPE && ln < nrn;
      const int32_t* info = A.rn + (int64_t)(on ? rn0 + ln : rn0) * 3;
      const int p0 = on ? info[0] : 0, p1 = on ? info[1] : 0, dof = info[2];
      int r[D];  // rows of this node in the chunk, -1: Dirichlet or another chunk's
#pragma unroll
      for (int i = 0; i < D; ++i) {
        r[i] = on ? A.full2red[dof + i] - r0 : -1;
        if (r[i] >= 64) r[i] = -1;
      }
      for (int p = p0; __any(p < p1); p += BATCH) {
        T k[BATCH][KB];
        std::conditional_t<sizeof(C) == 2, int, uint32_t> code[BATCH];
        bool own[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
          const bool in = p + j < p1;
          const int pp = in ? p + j : p0;
          code[j] = in ? ((const C*)A.code)[(int64_t)pp * NPE + b] : 0;
          const int32_t ea = A.inc[pp], e = ea / NPE;
          int plane;
          own[j] = stored_block<NPE>(ea % NPE, b, plane);
          const T* m = (const T*)A.matrices + ((int64_t)plane * A.n_elems + e) * KB;
#pragma unroll
          for (int i = 0; i < KB; ++i) k[j][i] = m[i];
        }
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
          // all words of a block are read before the first is written back (they are distinct); what
          // has no place in the rows goes to a spare word
          int word[KB];
          T old[KB];
          const int at0 = (int)(code[j] & ((1u << BITS) - 1)) - win;
#pragma unroll
          for (int i = 0; i < D; ++i) {
            int at = at0;
#pragma unroll
            for (int kk = 0; kk < D; ++kk) {
              const bool free = code[j] >> (BITS + kk) & 1;
              word[i * D + kk] = free && r[i] >= 0 && at >= 0 && at < A.window ? r[i] * A.stride + at : 64 * A.stride;
              old[i * D + kk] = rows[word[i * D + kk]];
              at += free ? 1 : 0;
            }
          }
#pragma unroll
          for (int i = 0; i < KB; ++i) rows[word[i]] = old[i] + (own[j] ? k[j][i] : k[j][i % D * D + i / D]);
        }
      }
    }
    __syncthreads();
    entries([&](int l, int64_t g) { vals[g] = (TO)rows[l]; });
    __syncthreads();
  }
}

// ---- residual -----------------------------------------------------------------------------------
// S[D][DIM] and f of r_a,i = sum_q S_q[i].dN_a(q) - f_q N_a(q)
template <class M>
struct ResModel;

template <int NPE, int DIM>
struct ResModel<NeoHooke<NPE, DIM>> {
  template <class X, class U>
  __device__ static double eval(int q, const double* dn, const double*, X x, U u, const double (*)[2],
                                const ModelParams& p, double (&S)[DIM][DIM]) {
    double J[DIM][DIM], U0[DIM][DIM], Ji[DIM][DIM], F[DIM][DIM], Fi[DIM][DIM], P[DIM][DIM];
    reference_gradient<NPE, DIM, DIM>(dn, x, J);
    reference_gradient<NPE, DIM, DIM>(dn, u, U0);
    const double w = Shape<NPE, DIM>::weight(q) * inverse<DIM>(J, Ji);
    product<DIM>(U0, Ji, F);
#pragma unroll
    for (int i = 0; i < DIM; ++i) F[i][i] += 1.0;
    const double det = inverse<DIM>(F, Fi), lam = p.p[0], mu = p.p[1];
    const double c1 = mu - 0.5 * lam * (det * det - 1.0);
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) P[i][j] = w * (mu * F[i][j] - c1 * Fi[j][i]);
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < DIM; ++k) s += P[i][k] * Ji[j][k];
        S[i][j] = s;
      }
    return 0.0;
  }
};

template <class M>
struct ResScalar {
  static constexpr int NPE = M::NPE, DIM = M::DIM;
  template <class X, class U>
  __device__ static double eval(int q, const double* dn, const double* n, X x, U u, const double (*nod)[2],
                                const ModelParams& p, double (&S)[1][DIM]) {
    double J[DIM][DIM], U0[1][DIM], Ji[DIM][DIM];
    reference_gradient<NPE, DIM, DIM>(dn, x, J);
    reference_gradient<NPE, 1, DIM>(dn, u, U0);
    const double w = Shape<NPE, DIM>::weight(q) * inverse<DIM>(J, Ji);
    double k = w, b;
    if constexpr (M::NODAL) {
      double g = 0.0;
      b = 0.0;
#pragma unroll
      for (int a = 0; a < NPE; ++a) {
        g += n[a] * nod[a][0];
        b += n[a] * nod[a][1];
      }
      k *= exp(g);
    } else {
      // b = p0 (sin(p1 x.x) - cos(p1 |x - (p2, p3)|^2))
      double xx = 0.0, yy = 0.0;
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        double xq = 0.0;
#pragma unroll
        for (int a = 0; a < NPE; ++a) xq += n[a] * x(a, i);
        const double c = xq - (i == 0 ? p.p[2] : p.p[3]);
        xx += xq * xq;
        yy += c * c;
      }
      b = p.p[0] * (sin(p.p[1] * xx) - cos(p.p[1] * yy));
    }
#pragma unroll
    for (int j = 0; j < DIM; ++j) {
      double s = 0.0;
#pragma unroll
      for (int l = 0; l < DIM; ++l) {
        double grad = 0.0;  // du/dX_l
#pragma unroll
        for (int m = 0; m < DIM; ++m) grad += U0[0][m] * Ji[m][l];
        s += grad * Ji[j][l];
      }
      S[0][j] = k * s;
    }
    return w * b;
  }
};
template <int NPE, int DIM>
struct ResModel<PoissonSource<NPE, DIM>> : ResScalar<PoissonSource<NPE, DIM>> {};
template <int NPE, int DIM>
struct ResModel<PoissonVarK<NPE, DIM>> : ResScalar<PoissonVarK<NPE, DIM>> {};

// Element vectors: EPB elements per workgroup, thread (element, t) evaluates Gauss point t, then adds
// up the row of node t (as many Gauss points as nodes in every model).
template <class M, int EPB>
__global__ __launch_bounds__(EPB * M::NPE) void k_element_vectors(const int32_t* __restrict__ conn, int64_t n_elems,
                                                                  const double* __restrict__ coords, int64_t n_nodes,
                                                                  const double* __restrict__ u, ModelParams mp,
                                                                  double* __restrict__ out) {
  constexpr int NPE = M::NPE, DIM = M::DIM, D = M::D, NQ = M::NQ, SW = (D * DIM + 1) | 1;
  static_assert(NQ == NPE, "one thread per Gauss point and per node");
  __shared__ double dn[NQ * NPE * DIM], sn[NQ * NPE];
  __shared__ double xs[EPB][NPE][DIM], us[EPB][NPE][D], ns[M::NODAL ? EPB : 1][NPE][2];
  __shared__ double sq[EPB * NPE][SW];
  const int le = threadIdx.x / NPE, t = threadIdx.x % NPE;
  const int64_t e = blockIdx.x * (int64_t)EPB + le;
  const bool on = e < n_elems;
  fill_gradients<M>(dn, sn);
  if (on) {
    const int32_t node = conn[e * NPE + t];
#pragma unroll
    for (int k = 0; k < DIM; ++k) xs[le][t][k] = coords[k * n_nodes + node];
#pragma unroll
    for (int i = 0; i < D; ++i) us[le][t][i] = u[(int64_t)node * D + i];
    if constexpr (M::NODAL) {
      ns[le][t][0] = mp.nodal[0][node];
      ns[le][t][1] = mp.nodal[1][node];
    }
  }
  __syncthreads();
  if (on) {
    double S[D][DIM];
    const double f = ResModel<M>::eval(
        t, dn + t * NPE * DIM, sn + t * NPE, [&](int a, int i) { return xs[le][a][i]; },
        [&](int a, int i) { return us[le][a][i]; }, ns[M::NODAL ? le : 0], mp, S);
    double* s = sq[threadIdx.x];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) s[i * DIM + j] = S[i][j];
    s[D * DIM] = f;
  }
  __syncthreads();
  if (!on) return;
  double r[D];
#pragma unroll
  for (int i = 0; i < D; ++i) r[i] = 0.0;
  for (int q = 0; q < NQ; ++q) {
    const double* s = sq[le * NPE + q];
    const double* d = dn + (q * NPE + t) * DIM;
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < DIM; ++j) r[i] += s[i * DIM + j] * d[j];
    if constexpr (D == 1) r[0] -= s[DIM] * sn[q * NPE + t];
  }
#pragma unroll
  for (int i = 0; i < D; ++i) out[(e * NPE + t) * D + i] = r[i];
}

// r of the listed nodes (null: all): the element vectors of their elements, in element order
__global__ void k_gather_vectors(int64_t n_list, const int32_t* __restrict__ list, const int32_t* __restrict__ ptr,
                                 const int32_t* __restrict__ inc, const double* __restrict__ vec, int d, int overwrite,
                                 double* __restrict__ r) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n_list * d) return;
  const int64_t l = t / d, i = t % d, node = list ? list[l] : l, dof = node * d + i;
  double s = 0.0;
  for (int32_t k = ptr[node]; k < ptr[node + 1]; ++k) s += vec[(int64_t)inc[k] * d + i];
  r[dof] = overwrite ? s : r[dof] + s;
}

// The same sums, bit by bit, without element vectors in memory: NPB nodes per workgroup, NPE threads each,
// which evaluate the node's elements one after the other, every element as often as it has nodes.
// For captured calls that get no scratch (captured_scratch).  64^3 Hex8: 306 us a replay, with scratch 87;
// 512^2 plane-strain quads 19 either way.
template <class M, int NPB>
__global__ __launch_bounds__(NPB * M::NPE) void k_node_residuals(int64_t n_list, const int32_t* __restrict__ list,
                                                                 const int32_t* __restrict__ ptr,
                                                                 const int32_t* __restrict__ inc,
                                                                 const int32_t* __restrict__ conn,
                                                                 const double* __restrict__ coords, int64_t n_nodes,
                                                                 const double* __restrict__ u, ModelParams mp,
                                                                 int overwrite, double* __restrict__ r) {
  constexpr int NPE = M::NPE, DIM = M::DIM, D = M::D, NQ = M::NQ, SW = (D * DIM + 1) | 1;
  __shared__ double dn[NQ * NPE * DIM], sn[NQ * NPE];
  __shared__ double xs[NPB][NPE][DIM], us[NPB][NPE][D], ns[M::NODAL ? NPB : 1][NPE][2];
  __shared__ double sq[NPB * NPE][SW];
  const int ln = threadIdx.x / NPE, t = threadIdx.x % NPE;
  const int64_t l = blockIdx.x * (int64_t)NPB + ln;
  const int64_t node = l >= n_list ? -1 : list ? list[l] : l;
  const int32_t p0 = node < 0 ? 0 : ptr[node], p1 = node < 0 ? 0 : ptr[node + 1];
  fill_gradients<M>(dn, sn);
  double s = 0.0;  // thread i < D: component i
  for (int32_t p = p0; __syncthreads_or(p < p1); ++p) {
    const bool on = p < p1;
    const int32_t ea = on ? inc[p] : 0, a = ea % NPE;
    if (on) {
      const int32_t c = conn[(int64_t)(ea / NPE) * NPE + t];
#pragma unroll
      for (int k = 0; k < DIM; ++k) xs[ln][t][k] = coords[k * n_nodes + c];
#pragma unroll
      for (int i = 0; i < D; ++i) us[ln][t][i] = u[(int64_t)c * D + i];
      if constexpr (M::NODAL) {
        ns[ln][t][0] = mp.nodal[0][c];
        ns[ln][t][1] = mp.nodal[1][c];
      }
    }
    __syncthreads();
    if (on) {
      double S[D][DIM];
      const double f = ResModel<M>::eval(
          t, dn + t * NPE * DIM, sn + t * NPE, [&](int b, int i) { return xs[ln][b][i]; },
          [&](int b, int i) { return us[ln][b][i]; }, ns[M::NODAL ? ln : 0], mp, S);
#pragma unroll
      for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < DIM; ++j) sq[threadIdx.x][i * DIM + j] = S[i][j];
      sq[threadIdx.x][D * DIM] = f;
    }
    __syncthreads();
    if (on && t < D) {
      double row = 0.0;
      for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int j = 0; j < DIM; ++j) row += sq[ln * NPE + q][t * DIM + j] * dn[(q * NPE + a) * DIM + j];
        if constexpr (D == 1) row -= sq[ln * NPE + q][DIM] * sn[q * NPE + a];
      }
      s += row;
    }
  }
  if (node < 0 || t >= D) return;
  double& out = r[node * D + t];
  out = overwrite ? s : out + s;
}

// Boundary lines: every listed node evaluates its own (one or two) lines; one launch, nothing stored
template <class M>
__global__ void k_line_vectors(int64_t n_list, const int32_t* __restrict__ list, const int32_t* __restrict__ ptr,
                               const int32_t* __restrict__ inc, const int32_t* __restrict__ conn,
                               const double* __restrict__ coords, int64_t n_nodes, ModelParams mp,
                               double* __restrict__ r) {
  const int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (l >= n_list) return;
  const int64_t node = list ? list[l] : l;
  double s[2] = {0.0, 0.0};
  for (int32_t k = ptr[node]; k < ptr[node + 1]; ++k) {
    const int32_t e = inc[k] / M::NPE, a = inc[k] % M::NPE;
    double x[M::NPE][2];
#pragma unroll
    for (int c = 0; c < M::NPE; ++c) {
      const int32_t node = conn[e * M::NPE + c];
      x[c][0] = coords[node];
      x[c][1] = coords[n_nodes + node];
    }
    typename M::template QP<double> Q[M::NQ];
#pragma unroll
    for (int q = 0; q < M::NQ; ++q) M::template qp<double>(q, x, nullptr, nullptr, mp, true, Q[q]);
    double out[2];
    M::res_row(a, Q, mp, out);
    s[0] += out[0];
    s[1] += out[1];
  }
  r[node * 2] += s[0];
  r[node * 2 + 1] += s[1];
}

bool is_capturing(hipStream_t st, unsigned long long* id = nullptr) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long ignored;
  if (hipStreamGetCaptureInfo(st, &status, id ? id : &ignored) != hipSuccess) (void)hipGetLastError();
  return status != hipStreamCaptureStatusNone;
}

// Element vectors of captured residuals: replays may overlap with anything else of the plan, other
// graphs and other branches of their own graph among it, so every capture has its own on each of its streams
// (whose calls follow one another in the graph).  A graph may be replayed as long as the plan lives, so
// they stay with the plan, and it makes at most kMost; null: no more of them, or no memory.
double* captured_scratch(Plan& P, hipStream_t st, unsigned long long id) {
  constexpr size_t kMost = 16;
  std::lock_guard<std::mutex> lock(P.scratch_mutex);
  for (auto& c : P.captured)
    if (c.id == id && c.stream == st) return c.vectors.p;
  if (P.captured.size() == kMost) return nullptr;
  Plan::Captured c{id, st, {}};
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // an allocation is no part of the capture
  APX_HIP(hipThreadExchangeStreamCaptureMode(&mode));
  const bool room = c.vectors.try_alloc(P.element_vectors.n);
  APX_HIP(hipThreadExchangeStreamCaptureMode(&mode));
  if (!room) return nullptr;
  P.captured.push_back(std::move(c));
  return P.captured.back().vectors.p;
}

// The plan's scratch is one: a call's work on it waits on the device for the last call's, from
// whatever stream and thread that came, and no other call comes between its wait and its own event.  (The
// wait is made on one stream too: a handle may be that of a stream made since, or of another thread's
// default stream.)  Under capture, of a tangent, neither is recorded: replays that overlap with tangents
// of the same type are the caller's to order.
struct ScratchUse {
  Plan& P;
  hipStream_t st;
  std::unique_lock<std::mutex> lock;
  bool capturing = false;
  ScratchUse(Plan& p, hipStream_t s) : P(p), st(s), lock(p.scratch_mutex) {
    capturing = is_capturing(st);
    if (capturing) return;
    if (P.scratch_done)
      APX_HIP(hipStreamWaitEvent(st, P.scratch_done, 0));
    else
      APX_HIP(hipEventCreateWithFlags(&P.scratch_done, hipEventDisableTiming));
  }
  ~ScratchUse() {
    if (!capturing) (void)hipEventRecord(P.scratch_done, st);
  }
};

// Element matrices of the plan's largest set, one buffer per type: allocated by the first tangent of that
// type and kept with the plan, so a captured tangent's pointer stays good.
template <class T>
T* element_matrices(Plan& P) {
  DevBuf<T>* buf;
  if constexpr (sizeof(T) == 8)
    buf = &P.element_matrices64;
  else
    buf = &P.element_matrices32;
  if (!buf->p) {
    size_t words = 0;
    for (const auto& S : P.sets)
      if (S.model != APX_MODEL_LINE_TRACTION)
        words = std::max(words, (size_t)S.n_elems * S.npe * (S.npe / 2 + 1) * P.d * P.d);  // kBlocks per node
    buf->alloc(words);
  }
  return buf->p;
}

template <class M, class T, class TO, bool CSR>
void run_rows(Plan& P, ElemSet& S, const double* u, void* vals, bool accumulate, hipStream_t st) {
  if constexpr (M::NODAL) {
    APX_REQUIRE(S.params.nodal[0] && S.params.nodal[1], APX_ERR_STATE,
                "variable-coefficient Poisson set needs nodal fields g and f bound");
  }
  constexpr int EPB = elements_per_block<M>(), NPW = 64 / M::NPE;
  ScratchUse use(P, st);
  T* matrices = element_matrices<T>(P);
  hipLaunchKernelGGL((k_element_matrices<M, T>), dim3((unsigned)((S.n_elems + EPB - 1) / EPB)), dim3(EPB * M::NPE), 0, st,
                     S.conn_orig.p, S.n_elems, P.coords.p, P.n_nodes, u, S.params, matrices);
  RowArgs A;
  A.rn_ptr = S.rn_ptr.p;
  A.rn = S.rn.p;
  A.inc = S.inc.p;
  A.code = S.code32.p ? (const void*)S.code32.p : S.code.p;
  A.full2red = P.full2red.p;
  A.indptr = P.indptr.p;
  A.sell_ptr = P.sell_ptr.p;
  A.n_free = (int)P.n_free;
  A.max_row = P.max_row;
  A.window = std::min(P.max_row, kRowWindow);
  A.stride = A.window | 1;
  A.accumulate = accumulate ? 1 : 0;
  A.n_elems = S.n_elems;
  A.matrices = matrices;
  A.vals = vals;
  const int waves = std::max(1, std::min(4, (S.rn_max + NPW - 1) / NPW));
  const size_t bytes = ((size_t)64 * A.stride + 1) * sizeof(T);
  const auto kernel =
      S.code32.p ? k_gather_rows<M::NPE, M::D, T, TO, CSR, uint32_t> : k_gather_rows<M::NPE, M::D, T, TO, CSR, uint16_t>;
  if (bytes > 48 * 1024)
    APX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  hipLaunchKernelGGL(kernel, dim3((unsigned)round_xcd(P.n_chunks)), dim3(waves * 64), (uint32_t)bytes, st, A);
  APX_LAUNCH_CHECK();
}

template <class F>
bool with_model(const Plan& P, const ElemSet& S, F f) {
  const int key = S.model * 100 + S.npe * 10 + P.dim;
  const bool poisson = S.model == APX_MODEL_POISSON_SOURCE || S.model == APX_MODEL_POISSON_VARK;
  if (poisson && (key % 100 == 42 || key % 100 == 83))
    APX_REQUIRE(P.d == 1, APX_ERR_ARG, "Poisson model needs one DOF per node");
  if (S.model == APX_MODEL_NEO_HOOKE && (key % 100 == 42 || key % 100 == 92))
    APX_REQUIRE(P.d == 2, APX_ERR_ARG, "plane-strain Neo-Hooke needs 2 DOFs per node");
  if (S.model == APX_MODEL_NEO_HOOKE && key % 100 == 83)
    APX_REQUIRE(P.d == 3, APX_ERR_ARG, "3D Neo-Hooke needs 3 DOFs per node");
  switch (key) {
    case APX_MODEL_POISSON_SOURCE * 100 + 42: return f(PoissonSource<4, 2>{});
    case APX_MODEL_POISSON_SOURCE * 100 + 83: return f(PoissonSource<8, 3>{});
    case APX_MODEL_POISSON_VARK * 100 + 42: return f(PoissonVarK<4, 2>{});
    case APX_MODEL_POISSON_VARK * 100 + 83: return f(PoissonVarK<8, 3>{});
    case APX_MODEL_NEO_HOOKE * 100 + 42: return f(NeoHooke<4, 2>{});
    case APX_MODEL_NEO_HOOKE * 100 + 83: return f(NeoHooke<8, 3>{});
    case APX_MODEL_NEO_HOOKE * 100 + 92: return f(NeoHooke<9, 2>{});
    default: return false;
  }
}
}  // namespace

void rows_tangent(Plan& P, const double* u, void* vals, int precision, bool csr, hipStream_t st) {
  bool have = false;
  const int64_t entries = csr ? P.nnz : P.sell_total;
  const auto tangents = std::count_if(P.sets.begin(), P.sets.end(),
                                      [](const ElemSet& S) { return S.model != APX_MODEL_LINE_TRACTION; });
  if (precision == kFP64RoundedToFP32 && tangents > 1) {  // rounded once, after the last set
    if (P.vals64.n < (size_t)P.sell_total) P.vals64.alloc(P.sell_total);
    rows_tangent(P, u, P.vals64.p, APX_FP64, csr, st);
    return round_to_f32(P.vals64.p, (float*)vals, entries, st);
  }
  if (P.n_chunks > 0) {
    for (auto& S : P.sets) {
      if (S.model == APX_MODEL_LINE_TRACTION) continue;  // zero tangent
      const bool ok = with_model(P, S, [&](auto m) {
        using M = decltype(m);
        if (precision == APX_FP64)
          csr ? run_rows<M, double, double, true>(P, S, u, vals, have, st)
              : run_rows<M, double, double, false>(P, S, u, vals, have, st);
        else if (precision == kFP64RoundedToFP32)
          csr ? run_rows<M, double, float, true>(P, S, u, vals, have, st)
              : run_rows<M, double, float, false>(P, S, u, vals, have, st);
        else
          csr ? run_rows<M, float, float, true>(P, S, u, vals, have, st)
              : run_rows<M, float, float, false>(P, S, u, vals, have, st);
        return true;
      });
      APX_REQUIRE(ok, APX_ERR_UNSUPPORTED, "no kernel for model " + std::to_string(S.model) + " with " +
                                               std::to_string(S.npe) + "-node elements in " + std::to_string(P.dim) +
                                               "D");
      have = true;
    }
  }
  if (have) return;
  if (precision == APX_FP64)
    fill<double>((double*)vals, entries, 0.0, st);
  else
    fill<float>((float*)vals, entries, 0.0f, st);
}

// r (+)= the set's residual; false: no such kernel (nothing done)
bool gather_residual(Plan& P, ElemSet& S, const double* u, double* r, bool overwrite, hipStream_t st) {
  const int64_t n = S.touched_all ? P.n_nodes : S.n_touched;
  const int32_t* list = S.touched_all ? nullptr : S.touched.p;
  if (S.model == APX_MODEL_LINE_TRACTION) {
    if (P.d != 2 || P.dim != 2 || (S.npe != 2 && S.npe != 3)) return false;
    if (overwrite) fill<double>(r, P.n_dofs, 0.0, st);
    const dim3 g((unsigned)((n + 127) / 128)), t(128);
    if (S.npe == 2)
      hipLaunchKernelGGL(k_line_vectors<LineTraction>, g, t, 0, st, n, list, S.inc_ptr.p, S.inc.p, S.conn_orig.p,
                         P.coords.p, P.n_nodes, S.params, r);
    else
      hipLaunchKernelGGL(k_line_vectors<LineTraction3>, g, t, 0, st, n, list, S.inc_ptr.p, S.inc.p, S.conn_orig.p,
                         P.coords.p, P.n_nodes, S.params, r);
    APX_LAUNCH_CHECK();
    return true;
  }
  return with_model(P, S, [&](auto m) {
    using M = decltype(m);
    constexpr int EPB = 256 / M::NPE;
    if constexpr (M::NODAL) {
      APX_REQUIRE(S.params.nodal[0] && S.params.nodal[1], APX_ERR_STATE,
                  "variable-coefficient Poisson set needs nodal fields g and f bound");
    }
    if (overwrite && !S.touched_all) fill<double>(r, P.n_dofs, 0.0, st);
    const int set = overwrite && S.touched_all ? 1 : 0;
    auto by_elements = [&](double* vectors) {
      hipLaunchKernelGGL((k_element_vectors<M, EPB>), dim3((unsigned)((S.n_elems + EPB - 1) / EPB)), dim3(EPB * M::NPE),
                         0, st, S.conn_orig.p, S.n_elems, P.coords.p, P.n_nodes, u, S.params, vectors);
      hipLaunchKernelGGL(k_gather_vectors, dim3((unsigned)((n * M::D + 255) / 256)), dim3(256), 0, st, n, list,
                         S.inc_ptr.p, S.inc.p, vectors, (int)M::D, set, r);
    };
    unsigned long long capture = 0;
    if (!is_capturing(st, &capture)) {
      ScratchUse use(P, st);
      by_elements(P.element_vectors.p);  // (allocated with the plan)
    } else if (double* vectors = captured_scratch(P, st, capture)) {
      by_elements(vectors);
    } else {
      hipLaunchKernelGGL((k_node_residuals<M, EPB>), dim3((unsigned)((n + EPB - 1) / EPB)), dim3(EPB * M::NPE), 0, st, n,
                         list, S.inc_ptr.p, S.inc.p, S.conn_orig.p, P.coords.p, P.n_nodes, u, S.params, set, r);
    }
    APX_LAUNCH_CHECK();
    return true;
  });
}

}  // namespace apx
