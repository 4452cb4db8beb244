// Internal interfaces shared by the library's translation units.
#pragma once
#include "plan.hpp"

namespace apx {

template <class T>
void fill(T* p, int64_t n, T v, hipStream_t s);
// dst = src rounded to FP32 (nearest), element by element.
void round_to_f32(const double* src, float* dst, int64_t n, hipStream_t s);

void assemble_residual(Plan& P, const double* u, double* r, hipStream_t st);
void assemble_tangent(Plan& P, const double* u, void* vals, int precision, hipStream_t st);
// precision code of "FP64 element arithmetic, values rounded once to FP32"
constexpr int kFP64RoundedToFP32 = APX_FP64_ROUNDED;
// The FP64 tangent rounded once to FP32 into vals (FP32, SELL order): written directly by the
// owner-tile kernels, else assembled in FP64 into the plan's scratch values and rounded.
void assemble_tangent_rounded(Plan& P, const double* u, float* vals, hipStream_t st);
void assemble_diagonal(Plan& P, const double* u, double* diag, hipStream_t st);
// full tangent as BCOO with duplicates (data only; the reference's element-major order)
int64_t tangent_coo_entries(const Plan& P);
void assemble_tangent_coo(Plan& P, const double* u, void* data, int precision, hipStream_t st);
int64_t residual_bytes(const Plan& P);
int64_t tangent_bytes(const Plan& P, int precision);

// structured.hip: owner-tile kernels for structured Q1 grids
// mode: 0 residual, 1 tangent, 2 diagonal
bool tile_supported(const Plan& P, const ElemSet& S, int mode);
bool tangent_by_tiles(const Plan& P);
void tile_residual(Plan& P, ElemSet& S, const double* u, double* r, bool overwrite, hipStream_t st);
void tile_tangent(Plan& P, ElemSet& S, const double* u, void* vals, int precision, hipStream_t st);
void tile_diagonal(Plan& P, ElemSet& S, const double* u, double* diag, bool overwrite, hipStream_t st);

// rows.hip: row-owner kernels for all other meshes
// the whole tangent, every stored entry written, in SELL or canonical CSR order
void rows_tangent(Plan& P, const double* u, void* vals, int precision, bool csr, hipStream_t st);
// r (+)= the set's residual; false: no kernel for this set (nothing done)
bool gather_residual(Plan& P, ElemSet& S, const double* u, double* r, bool overwrite, hipStream_t st);

// krylov.hip
struct KState {
  double gamma, gamma_prev, pAp, alpha, beta, rr, atol2, bb, rr0, rmax2, delta2;
  double rsq;      // flexible CG: sum of squares of the network's input, r scaled by D^-1/2
  int k, maxiter, done, reliable;  // contiguous: copied to the host as one block
};

void ensure_krylov_scratch(Plan& P, hipStream_t st);
// reduction partials of the Krylov kernels: 4 rows of kMaxBlocks = 8192 doubles
constexpr int64_t kKrylovPartials = 4 * 8192;
// A resident run's slots and its ResidentOut lie behind the rows of partials that the kernels before
// it use; the kernels that finish those partials clear them.  What comes between a run and its
// re-anchoring (free_norm) uses the first row only.
constexpr int kResidentMaxGroups = 256;
constexpr int64_t kResidentSlotsAt = 2 * 8192;
constexpr int kResidentSlotWords = 6 * kResidentMaxGroups;
struct ResidentOut {
  KState state;      // the scalars at the end of the run
  long long aborted;  // a workgroup gave up waiting for the others
};
constexpr int kResidentClearWords = kResidentSlotWords + (int)(sizeof(ResidentOut) / 8);
void spmv(Plan& P, const void* vals, const void* x, void* y, int precision, hipStream_t st);
void sell_to_csr(Plan& P, const void* sell, void* csr, int precision, hipStream_t st);
void csr_to_sell(Plan& P, const void* csr, void* sell, int precision, hipStream_t st);
void jacobi_inverse(Plan& P, const void* vals, void* inv_diag, int precision, hipStream_t st);
// FP64 inverse diagonal of an FP32 SELL matrix
void jacobi_inverse_f32_to_f64(Plan& P, const float* vals, double* inv_diag, hipStream_t st);

// The iterations of a PCG run from x = 0, r, z = D^-1 r, p_old and the scalars S to a stop flag in one
// launch, waited for (resident.hip).  x and p_new receive the solution and the last direction,
// host_state (pinned, sizeof(ResidentOut)) and the ResidentOut in part the scalars; S stays as it was (a
// re-anchored run goes on from the latter).  zt: 2 n_free words of scratch of the vectors' type.  idle:
// the stream has nothing to do but the run's start.  false: the system does not fit, or the run was given
// up; x is 0, r, z and p_old are as they were.
template <class M, class V>
bool pcg_resident(Plan& P, const M* vals, const V* inv, V* x, const V* r, const V* z, const V* p_old, V* p_new,
                  unsigned long long* zt, KState* S, double* part, KState* host_state, bool idle, hipStream_t st);

// How a resident run deals out a system of n rows of at most `row` entries, bandwidth bw: T threads a
// workgroup, K rows a thread, rows of up to RW entries in registers (0: read in every iteration), xl:
// x and D^-1 in LDS, cpw 64-row chunks a workgroup, G workgroups, bytes of dynamic LDS each.  T = 0: it
// does not fit on `cus` compute units.
struct ResidentShape {
  int T = 0, K = 0, RW = 0, cpw = 0, G = 0;
  bool xl = false;
  size_t lds = 0;
};
ResidentShape resident_shape(int64_t n, int64_t bw, int row, size_t vector_bytes, int cus);

// Symmetric 9-point matrices by grid lines (krylov.hip): the upper diagonals of SELL values for
// line_product, with P.asymmetric set on the device where they are not the whole matrix; null: not
// applicable.  vector_bytes: of an entry of the vectors.
template <class M>
const M* line_matrix(Plan& P, const M* vals, size_t vector_bytes, hipStream_t st);
// p_new = z + beta p_old, q = A p_new, block partials of p.q; r given: also of p.r; else x += alpha p_old
// from the second iteration after k0 on.  Exits at once when S has a stop flag.
template <class M, class T>
void line_product(Plan& P, const M* upper, const M* vals, const T* z, T* pa, T* pb, T* q, const T* r, T* x, int k0,
                  KState* S, double* part, hipStream_t st);
int line_blocks(const Plan& P);  // its workgroups

// One preconditioned-CG solve on the plan's SELL matrix with values of type M
// and Krylov vectors and scalars of type T (M = float, T = double: an FP32
// matrix with FP64 vectors).  Workspace (r, z, two directions, q, x) comes
// from the plan.  run() returns when the device sets the stop flag or requests
// a reliable update (residual drop by delta since the last anchor); reanchor()
// then installs a new true residual.
template <class M, class T = M>
struct PcgRun {
  Plan& P;
  const M* vals;
  const T* inv;
  hipStream_t st;
  int64_t n = 0;
  T *r = nullptr, *z = nullptr, *pa = nullptr, *pb = nullptr, *q = nullptr, *xw = nullptr, *x = nullptr;
  KState* S = nullptr;
  double* part = nullptr;  // reduction partials
  // external = true: workspace, partials and scalars come from the caller, and the run
  // creates no events, records no timing and polls the stop flag synchronously (allocates
  // nothing)
  bool external = false;
  bool streaming = false;  // a resident run was given up: not tried again
  // the matrix as its upper diagonals (streaming runs; null: read as SELL), known from the first
  // streaming run on it
  const M* upper = nullptr;
  bool upper_known = false;
  int k0 = 0;  // iterations before the present streaming run
  int start_k = 0;         // iterations before the present resident run
  bool idle = false;       // the stream had nothing to do before the run's start
  bool resident_last = false;  // the last run was resident: S still holds the scalars from before it
  int maxiter = 0, iterations = 0;
  int64_t launched = 0;
  size_t counted = 0;
  int64_t spmv_bytes = 0, upd_bytes = 0;
  hipEvent_t evs[2] = {nullptr, nullptr};
  std::vector<EventPair> ev_spmv, ev_upd, ev_res, ev_given_up;

  PcgRun(Plan& P, const M* vals, const T* inv, hipStream_t st);
  // caller-provided workspace: work = 6 n_free vectors, partials = kKrylovPartials doubles,
  // state = one KState (its fields are all written by init before they are read)
  PcgRun(Plan& P, const M* vals, const T* inv, hipStream_t st, T* work, double* partials, KState* state);
  ~PcgRun();
  // right-hand side b, or (r_full given) -r_full on the free DOFs
  void init(const T* b, const double* r_full, T* x, double tol, double atol, int maxiter, double delta);
  void launch_iteration();
  KState run();
  void reanchor(const double* r_full);
  void collect_timing();
};

// Does apx_pcg_noalloc take a solve with values of this size on the plan?
bool noalloc_accepts(const Plan& P, size_t value_bytes);
// Jacobi-PCG; workspace taken from the plan.
apx_krylov_stats pcg(Plan& P, const void* vals, const void* inv_diag, const void* b, void* x, int precision,
                     double tol, double atol, int maxiter, hipStream_t st);
// ||r[red2full]||_2 of a full-length FP64 vector (deterministic).
double free_norm(Plan& P, const double* r_full, hipStream_t st);
void gather_rhs(Plan& P, const double* r_full, double* b, hipStream_t st);
void scatter_update(Plan& P, double* u, const void* x, double damping, int precision, hipStream_t st);
void impose_dirichlet(Plan& P, double* u, const double* values, hipStream_t st);

// timing helpers
struct ScopedTimer {
  Plan& P;
  const char* name;
  hipStream_t st;
  int64_t bytes;
  ScopedTimer(Plan& p, const char* n, hipStream_t s, int64_t b);
  ~ScopedTimer();
};

}  // namespace apx
