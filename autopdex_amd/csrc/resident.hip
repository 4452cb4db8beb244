// Jacobi-PCG in one launch, its vectors resident on the compute units.
//
// k_pcg_resident runs the iterations that launch_iteration() would run as four launches each.
// Every workgroup owns a contiguous range of rows: x, r and D^-1 of its rows stay in registers, the
// direction p of its rows and of the columns they reach (the bandwidth on either side) in LDS, and
// rows of at most RW stored entries keep their matrix entries in registers too.  Per iteration the
// workgroups meet twice, to add up p.q and r.z, r.r; the second meeting also makes the new z of
// the neighbours visible, from which every workgroup extends its window of p = z + beta p.
//
// What bounds it: the latency of the two meetings, 1 to 2 us each across the 8 XCDs, growing with
// the number of workgroups, where the four launches of the streaming kernels cost 14 to 20 us an
// iteration however small the system is.  us per iteration, streaming -> resident (MI355X):
//   Q1 Poisson FP64: 229 rows 14.2 -> 1.7, 9,805: 17.4 -> 3.7, 39,605: 17.3 -> 5.0,
//     195,717: 23.0 -> 7.0, 510,565: 29.6 -> 10.2, 1,046,533: 39.8 -> 16.6
//   panel (18 entries a row): 6,272: 18.6 -> 3.8, 320,800: 36.6 -> 10.1, 524,288: 46.1 -> 14.2
//   Q2 (50): 1,600: 23.2 -> 3.5, 96,480: 29.2 -> 8.6, 320,800: 60.7 -> 28.3
//   Hex8 (81): 26,019: 32.4 -> 11.2 (FP32 21.9 -> 6.0), 123,725: 39.6 -> 18.3 (FP32 27.0 -> 10.3)
// Of 14.0 us at 786,944 rows 6 are the products (matrix entries spilled from the registers), 2 the
// halo, 2 a meeting, the rest updates and sums; of 11 us of the smaller Hex8 4.5, 2.5 and 2.
//
// Meeting: a workgroup writes its partial sums into its own slots and reads everybody's, so a
// sum costs one write and one read of memory that all XCDs see.  A slot is a 64-bit word holding the
// meeting's number beside half of a double, so a word is either complete or not yet there.  Everyone
// adds the partials in the same order, so all workgroups hold the same scalars, take the same
// branches, and a run is bitwise reproducible.  The z that other workgroups read travels in the
// same kind of word: nobody waits for its own stores, the halo is fetched while the first wave
// meets the others.  All of these words go through relaxed agent-scope atomics (written through,
// never read from a stale line).  None is overwritten early: a workgroup writes its words of one
// meeting again only after the other meeting, which everyone enters after having read them.
//
// The meetings need all workgroups on the device at once: the grid is at most one workgroup per
// compute unit, and concurrent runs of one process share the compute units through ResidentLease.
// Work of other streams only delays a workgroup.  Every wait is bounded (Plan::resident_wait): a
// workgroup that waits longer raises ResidentOut::aborted and leaves, and so do those that wait for
// it.  What the run started from (r, z, p, the scalars) is not written, so the caller then starts
// the streaming kernels from there, whatever the other workgroups have done.
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <optional>
#include <type_traits>

#include "assembly.hpp"

namespace apx {

namespace {
constexpr int kMaxDevices = 64;
typedef unsigned long long u64;

struct ResidentArgs {
  int n, n_chunks;  // rows, 64-row chunks
  int cpw;          // chunks per workgroup
  int bw;           // bandwidth
  const int32_t* sptr;
  const int16_t* cols;
  const KState* S;
  u64* slots;  // [p.q: G x 2 words][r.z, r.r: G x 4 words], zero before the launch
  u64* zt;     // tagged z of the rows that other workgroups read (2 words a row, FP32: 1)
  ResidentOut* out;   // on the device
  ResidentOut* host;  // the same in the host's pinned memory (a copy behind the run took 6 us)
  long long wait_ticks;
};

// ---- wave and workgroup sums, every lane gets the total ---------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return v + __hiloint2double(__builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true),
                              __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// sum over groups of N = 4, 8 or 16 lanes
template <int N>
__device__ __forceinline__ double row_sum(double v) {
  static_assert(N == 4 || N == 8 || N == 16, "groups within a row of 16 lanes");
  v = dpp_add<0xB1>(v);  // quad_perm 1,0,3,2
  v = dpp_add<0x4E>(v);  // quad_perm 2,3,0,1
  if constexpr (N >= 8) v = dpp_add<0x141>(v);   // row_half_mirror
  if constexpr (N == 16) v = dpp_add<0x140>(v);  // row_mirror
  return v;
}
__device__ __forceinline__ double wave_total(double v) {
  v = row_sum<16>(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

__device__ __forceinline__ u64 load_agent(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 64-bit words that carry the meeting's number: two for a double, one for a float.
template <class V>
struct Tagged {
  static constexpr int words = sizeof(V) / 4;
  static __device__ __forceinline__ void store(u64* p, V v, uint32_t number) {
    const u64 tag = (u64)number << 32;
    if constexpr (words == 2) {
      store_agent(p, tag | (uint32_t)__double2hiint(v));
      store_agent(p + 1, tag | (uint32_t)__double2loint(v));
    } else {
      store_agent(p, tag | __float_as_uint(v));
    }
  }
  struct Raw {
    u64 w[words];
  };
  static __device__ __forceinline__ Raw load(const u64* p) {
    Raw r;
#pragma unroll
    for (int i = 0; i < words; ++i) r.w[i] = load_agent(p + i);
    return r;
  }
  // false: not there yet
  static __device__ __forceinline__ bool value(const Raw& r, V& v, uint32_t number) {
    bool here = true;
#pragma unroll
    for (int i = 0; i < words; ++i) here &= (uint32_t)(r.w[i] >> 32) == number;
    if constexpr (words == 2)
      v = __hiloint2double((int)(uint32_t)r.w[0], (int)(uint32_t)r.w[1]);
    else
      v = __uint_as_float((uint32_t)r.w[0]);
    return here;
  }
};

// Bounded wait: true while the caller may try again.
struct Patience {
  ResidentOut* out;
  ResidentOut* host;
  long long ticks;
  long long t0 = wall_clock64();
  int tries = 0;
  __device__ __forceinline__ bool again(int* fail) {
    if ((++tries & 63) != 0) return true;
    if (wall_clock64() - t0 <= ticks &&
        __hip_atomic_load(&out->aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
      return true;
    __hip_atomic_store(&out->aborted, 1LL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&host->aborted, 1LL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *fail = 1;
    return false;
  }
};

// N tagged values, value i at p(i), until all are there; all loads of a try are in flight together
// (each try is a trip past the L2).  false: given up.
template <class V, int N, class P>
__device__ __forceinline__ bool collect(V (&v)[N], P p, uint32_t number, Patience& wait, int* fail) {
  for (;;) {
    typename Tagged<V>::Raw raw[N];
#pragma unroll
    for (int i = 0; i < N; ++i) raw[i] = Tagged<V>::load(p(i));
    bool here = true;
#pragma unroll
    for (int i = 0; i < N; ++i) here &= Tagged<V>::value(raw[i], v[i], number);
    if (here) return true;
    if (!wait.again(fail)) return false;
  }
}

// The first wave's part of a meeting: add up the waves' sums in red (NV x NW), publish them, collect
// everybody's and leave the totals in out.
template <int NW, int NV>
__device__ __forceinline__ void meet(const double* red, double* out, int* fail, u64* slots, int G, uint32_t number,
                                     Patience wait) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const double s = row_sum<NW>(red[j * NW + (lane & (NW - 1))]);
    if (lane == 0) Tagged<double>::store(slots + ((size_t)blockIdx.x * NV + j) * 2, s, number);
  }
  double got[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) got[j] = 0.0;
  auto take = [&](auto u, int g0) {
    constexpr int U = decltype(u)::value;
    double v[U * NV];
    if (!collect<double, U * NV>(
            v, [&](int i) { return slots + ((size_t)min(g0 + lane + 64 * (i / NV), G - 1) * NV + i % NV) * 2; }, number,
            wait, fail))
      return false;
#pragma unroll
    for (int i = 0; i < U * NV; ++i)
      if (g0 + lane + 64 * (i / NV) < G) got[i % NV] += v[i];
    return true;
  };
  constexpr int kTwo = NW < 16 ? 2 : 1;  // 1,024 threads have no registers for a second slot
  if (G <= 64) {
    if (!take(std::integral_constant<int, 1>{}, 0)) return;
  } else {
    for (int g0 = 0; g0 < G; g0 += 64 * kTwo)
      if (!take(std::integral_constant<int, kTwo>{}, g0)) return;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const double s = wave_total(got[j]);
    if (lane == 0) out[j] = s;
  }
}

// T threads, K rows per thread; RW > 0: rows of at most RW entries, held in registers; RW = 0: the
// entries are read in every iteration (from the XCD's L2 or the Infinity Cache, not from HBM).  XL:
// x and D^-1 in LDS instead of registers.  Sums over a row run in the stored order.
template <class M, class V, int T, int K, int RW, bool XL>
__global__ __launch_bounds__(T) void k_pcg_resident(ResidentArgs A, const M* __restrict__ vals,
                                                    const V* __restrict__ inv, V* __restrict__ x,
                                                    const V* __restrict__ r, const V* __restrict__ z,
                                                    const V* __restrict__ p_old, V* __restrict__ p_new) {
  constexpr int NW = T / 64;
  // halo entries that a thread asks for at once: as registers are left beside the matrix (1,024 threads
  // have few and rarely a second entry)
  constexpr int kRegs = T > 256 ? 131072 / T : 512;
  constexpr int kLeft = kRegs - K * (RW * (int)(sizeof(M) / 4) + (RW + 1) / 2) - 4 * K * (int)(sizeof(V) / 4);
  // The positions are unpacked in every iteration where, hoisted by the compiler to a register each,
  // they would spill the matrix (which is then read back from scratch in every iteration): 81 entries
  // of FP64 20 x 19 x 21 Hex8 11.9 -> 9.8 us an iteration, 8 x 9 entries 18.3 -> 14.9 us; elsewhere
  // the unpacking costs up to 0.2 us.
  constexpr bool kPacked = 5 * K * RW * (int)(sizeof(M) / 4 + 1) > 4 * kRegs;
  constexpr int kHalo = T == 1024 ? 1 : kLeft >= 128 ? 8 : kLeft >= 96 ? 4 : kLeft >= 64 ? 2 : 1;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ double redA[NW], redB[2 * NW], totA[1], totB[2];
  __shared__ int fail;
  const KState* S = A.S;
  auto report = [&](KState* o) {
    o->rr0 = S->rr0;
    o->bb = S->bb;
    o->atol2 = S->atol2;
    o->rmax2 = S->rmax2;
    o->delta2 = S->delta2;
    o->maxiter = S->maxiter;
  };
  if (S->done | S->reliable) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      for (KState* o : {&A.out->state, &A.host->state}) {
        report(o);
        o->gamma = S->gamma;
        o->gamma_prev = S->gamma_prev;
        o->beta = S->beta;
        o->rr = S->rr;
        o->k = S->k;
        o->done = S->done;
        o->reliable = S->reliable;
      }
    }
    return;
  }
  const int G = gridDim.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c0 = blockIdx.x * A.cpw, c1 = min(c0 + A.cpw, A.n_chunks);
  const int row0 = c0 * 64, row1 = min(c1 * 64, A.n);
  const int w0 = max(0, row0 - A.bw), w1 = min(A.n, row1 + A.bw);
  const int n_lo = row0 - w0, n_halo = n_lo + (w1 - row1);  // window entries of other workgroups' rows
  V* pw = (V*)lds_raw;          // p on [w0, w1)
  V* zh = pw + (w1 - w0);       // the halo's new z
  V* xl = zh + n_halo;          // XL: x and D^-1 of the own rows
  V* il = xl + (row1 - row0);
  double gamma = S->gamma, gamma_prev = S->gamma_prev, beta = S->beta, alpha = 0.0, pAp = 0.0, rr = S->rr;
  const double atol2 = S->atol2, delta2 = S->delta2, rmax2 = S->rmax2;
  const int maxiter = S->maxiter;
  int k = S->k, done = 0, reliable = 0;
  if (tid == 0) fail = 0;
  for (int j = w0 + tid; j < w1; j += T) pw[j - w0] = z[j] + (V)beta * p_old[j];

  // row i of this thread
  const int lrow = w * 64 + lane, rows = row1 - row0;  // relative to row0
  auto at = [&](int i) { return lrow + i * T; };
  auto on = [&](int i) { return at(i) < rows; };
  // in another workgroup's window
  auto seen = [&](int i) { return G > 1 && on(i) && (at(i) < A.bw || rows - at(i) <= A.bw); };
  V xv[XL ? 1 : K], iv[XL ? 1 : K], rv[K], q[K];
  constexpr int RE = RW ? RW : 1;
  M a[K][RE];
  uint32_t ci[K][(RE + 1) / 2];  // window positions of the columns, two in a word
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int row = row0 + at(i);
    rv[i] = on(i) ? r[row] : V(0);
    q[i] = 0;
    if constexpr (XL) {
      if (on(i)) {
        xl[at(i)] = 0;
        il[at(i)] = inv[row];
      }
    } else {
      xv[i] = 0;
      iv[i] = on(i) ? inv[row] : V(0);
    }
    if (seen(i)) {  // no tag of an earlier run may stay
#pragma unroll
      for (int j = 0; j < Tagged<V>::words; ++j) store_agent(A.zt + (size_t)row * Tagged<V>::words + j, 0);
    }
    if constexpr (RW > 0) {
      const int c = c0 + w + i * NW;
      const int off = c < c1 ? A.sptr[c] : 0, width = c < c1 ? (A.sptr[c + 1] - off) >> 6 : 0;
      // an entry past the row's end is 0 times the row's own p
      const uint32_t self = on(i) ? row - w0 : 0;
#pragma unroll
      for (int e = 0; e < RW; ++e) {
        const bool in = on(i) && e < width;
        a[i][e] = in ? vals[off + lane + e * 64] : M(0);
        const uint32_t pos = in ? self + A.cols[off + lane + e * 64] : self;
        if (e & 1)
          ci[i][e >> 1] |= pos << 16;
        else
          ci[i][e >> 1] = pos;
      }
    }
  }
  uint32_t number = 0;
  if (G > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (;;) {
    ++number;
    double v1 = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      V s = 0;
      if constexpr (RW > 0) {
#pragma unroll
        for (int e = 0; e < RW; ++e) {
          // the positions are unpacked here: hoisted, each would take a register of its own
          if constexpr (kPacked)
            if ((e & 1) == 0) asm volatile("" : "+v"(ci[i][e >> 1]));
          const uint32_t pos = (e & 1) ? ci[i][e >> 1] >> 16 : ci[i][e >> 1] & 0xffffu;
          // FP32 entries of an FP64 run are widened here: hoisted, they would take two registers each
          if constexpr (sizeof(M) < sizeof(V)) asm volatile("" : "+v"(a[i][e]));
          s += (V)a[i][e] * pw[pos];
        }
      } else {
        // nine entries a step (9, 18 and 81 are the common row lengths), all loads issued first
        constexpr int U = 9;
        const int c = c0 + w + i * NW;
        const int off = c < c1 ? A.sptr[c] : 0, width = c < c1 ? (A.sptr[c + 1] - off) >> 6 : 0;
        const int self = on(i) ? row0 - w0 + at(i) : 0;
        for (int e = 0; e < width; e += U) {
          M av[U];
          int16_t d[U];
#pragma unroll
          for (int j = 0; j < U; ++j) {
            const int where = off + lane + min(e + j, width - 1) * 64;
            av[j] = vals[where];
            d[j] = A.cols[where];
          }
#pragma unroll
          for (int j = 0; j < U; ++j) {
            // lanes past the last row hold padding whose offset counts from that row
            const V t = (V)av[j] * pw[on(i) ? self + d[j] : 0];
            s += e + j < width ? t : V(0);
          }
        }
      }
      q[i] = s;
      if (on(i)) v1 += (double)pw[row0 - w0 + at(i)] * (double)s;
    }
    v1 = wave_total(v1);
    if (lane == 0) redA[w] = v1;
    __syncthreads();
    if (G > 1) {
      if (w == 0) meet<NW, 1>(redA, totA, &fail, A.slots, G, number, Patience{A.out, A.host, A.wait_ticks});
      __syncthreads();
      if (fail) return;
      pAp = totA[0];
    } else {
      pAp = row_sum<NW>(redA[lane & (NW - 1)]);
    }
    alpha = gamma / pAp;
    const V al = (V)alpha;
    double v2[2] = {0.0, 0.0};
    V zv[XL ? 1 : K];  // XL: formed again from r where it is needed
#pragma unroll
    for (int i = 0; i < K; ++i) {
      if (!on(i)) continue;
      const int o = at(i);
      const V p = pw[row0 - w0 + o];
      rv[i] -= al * q[i];
      V zi;
      if constexpr (XL) {
        xl[o] += al * p;
        zi = il[o] * rv[i];
      } else {
        xv[XL ? 0 : i] += al * p;
        zi = zv[XL ? 0 : i] = iv[XL ? 0 : i] * rv[i];
      }
      if (seen(i)) Tagged<V>::store(A.zt + (size_t)(row0 + o) * Tagged<V>::words, zi, number);
      v2[0] += (double)rv[i] * (double)zi;
      v2[1] += (double)rv[i] * (double)rv[i];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      v2[j] = wave_total(v2[j]);
      if (lane == 0) redB[j * NW + w] = v2[j];
    }
    __syncthreads();
    if (G > 1) {
      // the first wave meets the others while the rest fetch the halo
      if (w == 0) {
        meet<NW, 2>(redB, totB, &fail, A.slots + 2 * G, G, number, Patience{A.out, A.host, A.wait_ticks});
      } else {
        Patience wait{A.out, A.host, A.wait_ticks};
        for (int j0 = tid - 64; j0 < n_halo; j0 += kHalo * (T - 64)) {
          auto entry = [&](int i) { return min(j0 + i * (T - 64), n_halo - 1); };
          V v[kHalo];
          if (!collect<V, kHalo>(
                  v,
                  [&](int i) {
                    const int j = entry(i), row = j < n_lo ? w0 + j : row1 + (j - n_lo);
                    return A.zt + (size_t)row * Tagged<V>::words;
                  },
                  number, wait, &fail))
            break;
#pragma unroll
          for (int i = 0; i < kHalo; ++i) zh[entry(i)] = v[i];
        }
      }
      __syncthreads();
      if (fail) return;
      v2[0] = totB[0];
      v2[1] = totB[1];
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) v2[j] = row_sum<NW>(redB[j * NW + (lane & (NW - 1))]);
    }
    gamma_prev = gamma;
    beta = v2[0] / gamma;
    gamma = v2[0];
    rr = v2[1];
    k += 1;
    done = !(rr > atol2 && k < maxiter);
    reliable = !done && delta2 > 0.0 && rr < delta2 * rmax2;
    if (done | reliable) break;
    const V be = (V)beta;
    for (int j = tid; j < n_halo; j += T) {
      V* p = pw + (j < n_lo ? j : row1 - w0 + (j - n_lo));
      *p = zh[j] + be * *p;
    }
#pragma unroll
    for (int i = 0; i < K; ++i)
      if (on(i)) {
        V* p = pw + (row0 - w0) + at(i);
        *p = (XL ? il[at(i)] * rv[i] : zv[XL ? 0 : i]) + be * *p;
      }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (!on(i)) continue;
    x[row0 + at(i)] = XL ? xl[at(i)] : xv[XL ? 0 : i];
    p_new[row0 + at(i)] = pw[row0 - w0 + at(i)];
  }
  if (blockIdx.x == 0 && tid == 0) {
    for (KState* o : {&A.out->state, &A.host->state}) {
      report(o);
      o->gamma = gamma;
      o->gamma_prev = gamma_prev;
      o->beta = beta;
      o->alpha = alpha;
      o->pAp = pAp;
      o->rr = rr;
      o->k = k;
      o->done = done;
      o->reliable = reliable;
    }
  }
}

// The compute units that this process's resident runs hold, per device: a run waits until its
// workgroups fit beside those of the runs in flight on other threads, so that all of them can be
// on the device at once.
struct ResidentSlots {
  std::mutex mu;
  std::condition_variable cv;
  int used[kMaxDevices] = {};
};
ResidentSlots& resident_slots() {
  static ResidentSlots s;
  return s;
}

struct ResidentLease {
  ResidentSlots& s = resident_slots();
  const int dev, n;
  ResidentLease(int device, int groups, int cus) : dev(device), n(groups) {
    std::unique_lock<std::mutex> lock(s.mu);
    s.cv.wait(lock, [&] { return s.used[dev] + n <= cus; });
    s.used[dev] += n;
  }
  ~ResidentLease() {
    {
      std::lock_guard<std::mutex> lock(s.mu);
      s.used[dev] -= n;
    }
    s.cv.notify_all();
  }
};

int device_cus(int dev) {
  int cus = 0;
  APX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return cus;
}

}  // namespace

// LDS for the vectors: it leaves room for the reduction words in 160 KB.
constexpr size_t kResidentLds = 156 * 1024;

// Why the lines lie there (us per iteration, FP64; entries in registers against read each time):
// registers beat reading the entries everywhere they fit (39,605 rows of 9: 5.0 against 7.6 with
// the same 2,048 rows per workgroup; 80,400 of 18: 7.3 against 9.9; 25,960 of 81: 10.3 against
// 17.1).  Fewer workgroups meet faster, more share the work: 9,805 rows of 9 take 4.0 with 1,024
// rows per workgroup and 3.7 with 2,048; 195,717 take 9.6, 8.4 and (3,072 rows) 7.0, where the
// narrower row of threads also frees registers.  A single workgroup meets nobody: 1,525 rows of 9
// take 2.0 against 3.6 in two.  Wide rows: 1,600 of 50 take 3.6 with 256 threads and 3.8 with 512,
// 19,440 take 6.7 and 5.5; 1,863 of 81 5.8 and 8.2 (82 registers spill), 25,960 11.9 and 10.4.
// Wherever a shape fits it was faster than the streaming kernels, up to the largest (see above).
ResidentShape resident_shape(int64_t n, int64_t bw, int row, size_t vector_bytes, int cus) {
  const int64_t chunks = (n + kSellC - 1) / kSellC;
  ResidentShape s;
  if (bw > INT16_MAX || n < 1 || cus < 1) return s;
  // cpw chunks per workgroup of T threads, rows of up to RW entries in registers
  auto take = [&](int T, int K, int RW, bool xl, int64_t cpw) {
    const int64_t G = (chunks + cpw - 1) / cpw, own = std::min<int64_t>(n, cpw * 64);
    if (G > cus) return false;
    // The largest need of a workgroup, as the kernel lays out its LDS: the window of p, the halo's z, and
    // with xl the own rows' x and D^-1.  A last workgroup of a few rows has the whole bandwidth before it.
    int64_t words = 0, window = 0;
    for (int64_t row0 = 0; row0 < n; row0 += own) {
      const int64_t rows = std::min(own, n - row0), halo = std::min(bw, row0) + std::min(bw, n - row0 - rows);
      window = std::max(window, rows + halo);
      words = std::max(words, rows + 2 * halo + (xl ? 2 * rows : 0));
    }
    const size_t lds = (size_t)words * vector_bytes;
    if (window > 65536 || lds > kResidentLds) return false;
    s.T = T;
    s.K = K;
    s.RW = RW;
    s.xl = xl;
    s.cpw = (int)cpw;
    s.G = (int)G;
    s.lds = lds;
    return true;
  };
  if (row <= 9) {
    if (chunks <= 16 && take(1024, 1, 9, false, chunks)) return s;
    if (chunks <= 32 && take(1024, 2, 9, false, chunks)) return s;
    if (chunks <= 64 && take(1024, 1, 9, false, 16)) return s;
    if (chunks <= 1536 && take(1024, 2, 9, false, 32)) return s;
    if (take(512, 6, 9, true, 48)) return s;
    if (take(512, 8, 9, true, 64)) return s;
  } else if (row <= 18) {
    if (chunks <= 16 && take(1024, 1, 18, false, chunks)) return s;
    if (take(1024, 1, 18, false, 16)) return s;
    if (take(512, 3, 18, true, 24)) return s;
    if (take(512, 4, 18, true, 32)) return s;
  } else if (row <= 54) {
    if (chunks <= 32 && take(256, 1, 54, false, 4)) return s;
    if (take(512, 1, 54, false, 8)) return s;
  } else if (row <= 81) {
    if (chunks <= 64 && take(256, 1, 81, false, 4)) return s;
    if (take(512, 1, 81, false, 8)) return s;
  }
  if (take(1024, 1, 0, false, 16)) return s;
  if (take(1024, 2, 0, false, 32)) return s;
  if (take(1024, 4, 0, false, 64)) return s;
  s.T = 0;
  return s;
}

namespace {
template <class M, class V, int T, int K, int RW, bool XL>
bool launch_if(const ResidentShape& s, const ResidentArgs& A, const M* vals, const V* inv, V* x, const V* r, const V* z,
               const V* p_old, V* p_new, hipStream_t st) {
  if (s.T != T || s.K != K || s.RW != RW || s.xl != XL) return false;
  const auto kernel = k_pcg_resident<M, V, T, K, RW, XL>;
  if (s.lds > 48 * 1024)
    APX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResidentLds));
  launch_kernel(kernel, dim3(s.G), dim3(T), (uint32_t)s.lds, st, A, vals, inv, x, r, z, p_old, p_new);
  APX_LAUNCH_CHECK();
  return true;
}
}  // namespace

template <class M, class V>
bool pcg_resident(Plan& P, const M* vals, const V* inv, V* x, const V* r, const V* z, const V* p_old, V* p_new, u64* zt,
                  KState* S, double* part, KState* host_state, bool idle, hipStream_t st) {
  int dev = 0;
  APX_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices || P.resident_wait < 0.0) return false;
  if (P.cus == 0) {
    P.cus = device_cus(dev);
    int khz = 0;
    APX_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    P.clock_khz = khz > 0 ? khz : 100000;
  }
  if (!P.sell_dcol.p) return false;
  const ResidentShape s = resident_shape(P.n_free, P.bandwidth, P.max_row, sizeof(V), std::min(P.cus, kResidentMaxGroups));
  if (s.T == 0) return false;
  if (P.resident_skip > 0) {
    --P.resident_skip;
    return false;
  }
  ResidentArgs A;
  A.n = (int)P.n_free;
  A.n_chunks = (int)P.n_chunks;
  A.cpw = s.cpw;
  A.bw = (int)P.bandwidth;
  A.sptr = P.sell_ptr.p;
  A.cols = P.sell_dcol.p;
  A.S = S;
  A.slots = (u64*)(part + kResidentSlotsAt);
  A.zt = zt;
  A.out = (ResidentOut*)(A.slots + kResidentSlotWords);
  A.wait_ticks = (long long)(P.resident_wait * 1e3 * P.clock_khz);
  auto on = [&](auto t, auto k, auto rw, auto xl) {
    return launch_if<M, V, decltype(t)::value, decltype(k)::value, decltype(rw)::value, decltype(xl)::value>(
        s, A, vals, inv, x, r, z, p_old, p_new, st);
  };
#define APX_SHAPE(T, K, RW, XL)                                                                                \
  on(std::integral_constant<int, T>{}, std::integral_constant<int, K>{}, std::integral_constant<int, RW>{}, \
     std::integral_constant<bool, XL>{})
  ResidentOut* host = (ResidentOut*)host_state;
  A.host = host;
  std::memset(host, 0, sizeof(ResidentOut));
  {
    // The compute units are held only while the run is on the device: what else the stream has to do before
    // it is waited for first, or a solve on another thread would wait for all of that (10 us a solve, none
    // where only the run's own start is queued, as in Newton).  A single workgroup meets nobody and holds none;
    // others at most wait for it to end.
    std::optional<ResidentLease> lease;
    if (s.G > 1) {
      if (!idle) APX_HIP(hipStreamSynchronize(st));
      lease.emplace(dev, s.G, P.cus);
    }
    const bool launched = APX_SHAPE(1024, 1, 9, false) || APX_SHAPE(1024, 2, 9, false) || APX_SHAPE(512, 6, 9, true) || APX_SHAPE(512, 8, 9, true) ||
                          APX_SHAPE(1024, 1, 18, false) || APX_SHAPE(512, 3, 18, true) ||
                          APX_SHAPE(512, 4, 18, true) || APX_SHAPE(256, 1, 54, false) ||
                          APX_SHAPE(256, 1, 81, false) || APX_SHAPE(512, 1, 54, false) ||
                          APX_SHAPE(512, 1, 81, false) || APX_SHAPE(1024, 1, 0, false) ||
                          APX_SHAPE(1024, 2, 0, false) || APX_SHAPE(1024, 4, 0, false);
    APX_REQUIRE(launched, APX_ERR_INTERNAL, "resident PCG: no kernel of this shape");
    APX_HIP(hipStreamSynchronize(st));
  }
#undef APX_SHAPE
  std::atomic_thread_fence(std::memory_order_acquire);  // written by the kernel
  if (host->aborted) {
    fill<V>(x, P.n_free, V(0), st);
    // Where the workgroups do not get onto the device together (another process's runs hold its compute
    // units, a masked queue), every further run would wait as long in vain: the plan's next 16 runs go to the
    // streaming kernels at once, after a second give-up 64, then 256, 1,024 and 4,096.
    P.resident_skip = 16 << 2 * P.resident_given_up;
    P.resident_given_up = std::min(P.resident_given_up + 1, 4);
    return false;
  }
  P.resident_given_up = 0;
  return true;
}

template bool pcg_resident<double, double>(Plan&, const double*, const double*, double*, const double*, const double*,
                                           const double*, double*, u64*, KState*, double*, KState*, bool, hipStream_t);
template bool pcg_resident<float, float>(Plan&, const float*, const float*, float*, const float*, const float*,
                                         const float*, float*, u64*, KState*, double*, KState*, bool, hipStream_t);
template bool pcg_resident<float, double>(Plan&, const float*, const double*, double*, const double*, const double*,
                                          const double*, double*, u64*, KState*, double*, KState*, bool, hipStream_t);

}  // namespace apx
