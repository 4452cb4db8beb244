// Host-side plan construction: reduced CSR pattern, element colouring and the
// lists of the row-owner kernels.  Replaces, once per mesh and Dirichlet mask, the
// per-call index construction of _get_indices (assembler.py:47-141) and the
// scipy COO -> CSR -> [:, free][free] reduction of scipy_assembling
// (solver.py:1180-1222).  The reduced pattern equals scipy's canonical CSR:
// rows and columns are the free DOFs in increasing order, one entry per
// coupled (free, free) DOF pair of any element of any set, columns sorted.
#include <algorithm>
#include <chrono>
#include <cstring>

#include "assembly.hpp"

namespace apx {

Plan::~Plan() {
  if (scratch_done) (void)hipEventDestroy(scratch_done);
  if (pinned) (void)hipHostFree(pinned);
  if (ev0) (void)hipEventDestroy(ev0);
  if (ev1) (void)hipEventDestroy(ev1);
  for (auto e : evpool) (void)hipEventDestroy(e);
}

static hipEvent_t pool_event(Plan& P) {
  if (!P.evpool.empty()) {
    hipEvent_t e = P.evpool.back();
    P.evpool.pop_back();
    return e;
  }
  hipEvent_t e;
  APX_HIP(hipEventCreate(&e));
  return e;
}

EventPair timing_begin(Plan& P, hipStream_t st) {
  EventPair e;
  if (!P.timing) return e;
  e.a = pool_event(P);
  e.b = pool_event(P);
  APX_HIP(hipEventRecord(e.a, st));
  return e;
}

EventPair timing_pair(Plan& P) {
  EventPair e;
  e.a = pool_event(P);
  e.b = pool_event(P);
  return e;
}

void timing_end(Plan& P, EventPair& e, hipStream_t st) {
  if (e.b) APX_HIP(hipEventRecord(e.b, st));
}

void timing_collect(Plan& P, const char* name, std::vector<EventPair>& pairs, int64_t bytes, size_t count_limit) {
  if (pairs.empty()) return;
  auto& t = P.timers[name];
  for (size_t i = 0; i < pairs.size(); ++i) {
    auto& e = pairs[i];
    if (!e.a) continue;
    if (i < count_limit) {
      APX_HIP(hipEventSynchronize(e.b));
      float ms = 0.f;
      APX_HIP(hipEventElapsedTime(&ms, e.a, e.b));
      t.total_ms += ms;
      t.count += 1;
      t.bytes = bytes;
    } else {
      APX_HIP(hipEventSynchronize(e.b));
    }
    P.evpool.push_back(e.a);
    P.evpool.push_back(e.b);
  }
  pairs.clear();
}

int64_t Plan::device_bytes() const {
  int64_t b = coords.bytes() + dmask.bytes() + full2red.bytes() + red2full.bytes() + indptr.bytes() +
              indices.bytes() + diag_slot.bytes() + sell_ptr.bytes() + sell_cols.bytes() + sell_dcol.bytes() +
              csr2sell.bytes() + vals64.bytes() + vals32.bytes() + w64.bytes() + w32.bytes() + r_full.bytes() +
              diag_full.bytes() + partials.bytes() + lines64.bytes() + lines32.bytes() + element_vectors.bytes() +
              element_matrices64.bytes() + element_matrices32.bytes();
  for (auto& s : sets)
    b += s.conn.bytes() + s.conn_orig.bytes() + s.inc_ptr.bytes() + s.inc.bytes() + s.touched.bytes() + s.rn_ptr.bytes() +
         s.rn.bytes() + s.code.bytes() + s.code32.bytes();
  for (auto& c : captured) b += c.vectors.bytes();
  return b;
}

// Is the reduced matrix that of a 9-point stencil on lines of m rows, but for a few chunks (the
// corners of a grid whose Dirichlet mask leaves them free)?  m is read off a fullest row in the
// middle.
static void find_lines(Plan& P) {
  P.line = 0;
  if (P.max_row != 9 || P.n_free >= INT32_MAX / 2) return;
  int64_t full = P.n_free / 2;
  while (P.indptr_h[full + 1] - P.indptr_h[full] != 9) full = (full + 1) % P.n_free;
  const int32_t* c = P.indices_h.data() + P.indptr_h[full];
  const int32_t m = c[8] - (int32_t)full - 1;
  const int32_t off[9] = {-m - 1, -m, -m + 1, -1, 0, 1, m - 1, m, m + 1};
  std::vector<uint32_t> irregular((P.n_chunks + 31) / 32, 0);
  // up to one chunk in sixteen may be read from the SELL values
  int64_t left = P.n_chunks / 16;
  for (int64_t ch = 0; ch < P.n_chunks; ++ch) {
    bool regular = true;
    for (int64_t r = ch * kSellC; r < std::min<int64_t>(P.n_free, (ch + 1) * kSellC) && regular; ++r) {
      int at = 0;  // both ascend
      for (int32_t k = P.indptr_h[r]; k < P.indptr_h[r + 1] && regular; ++k, ++at) {
        const int32_t o = P.indices_h[k] - (int32_t)r;
        while (at < 9 && off[at] < o) ++at;
        regular = at < 9 && off[at] == o;
      }
    }
    if (regular) continue;
    if (--left < 0) return;
    irregular[ch / 32] |= 1u << (ch % 32);
  }
  P.line = m;
  P.irregular_h.swap(irregular);
}

// Node -> (element, local index) pairs of a set, in element order.
static void build_incidence(const Plan& P, ElemSet& s) {
  const int64_t m = s.n_elems * s.npe;
  APX_REQUIRE(m < INT32_MAX, APX_ERR_UNSUPPORTED, "element set exceeds int32 indexing");
  s.inc_ptr_h.assign(P.n_nodes + 1, 0);
  for (int64_t k = 0; k < m; ++k) s.inc_ptr_h[s.conn_host[k] + 1]++;
  for (int64_t n = 0; n < P.n_nodes; ++n) s.inc_ptr_h[n + 1] += s.inc_ptr_h[n];
  std::vector<int32_t> at(s.inc_ptr_h.begin(), s.inc_ptr_h.end() - 1);
  s.inc_h.resize(m);
  for (int64_t k = 0; k < m; ++k) s.inc_h[at[s.conn_host[k]]++] = (int32_t)k;
}

// ElemSet::code: the first position of a node's columns in BITS bits, its free DOFs above.
template <int BITS, class C>
static void build_codes(const Plan& P, const ElemSet& s, std::vector<C>& code, const std::vector<int64_t>& adj_ptr,
                        const std::vector<int32_t>& adj) {
  const int d = P.d, npe = s.npe;
  code.assign((size_t)s.n_elems * npe * npe, 0);
  std::vector<C> place;
  for (int64_t n = 0; n < P.n_nodes; ++n) {
    if (s.inc_ptr_h[n + 1] == s.inc_ptr_h[n]) continue;
    const int32_t *b = adj.data() + adj_ptr[n], *e = adj.data() + adj_ptr[n + 1];
    place.clear();
    uint32_t at = 0;
    for (const int32_t* p = b; p != e; ++p) {
      uint32_t free = 0, count = 0;
      for (int k = 0; k < d; ++k)
        if (!P.dmask_host[(int64_t)*p * d + k]) {
          free |= 1u << k;
          ++count;
        }
      place.push_back((C)((count ? at : 0) | free << BITS));
      at += count;
    }
    for (int32_t k = s.inc_ptr_h[n]; k < s.inc_ptr_h[n + 1]; ++k) {
      const int64_t* c = &s.conn_host[(int64_t)(s.inc_h[k] / npe) * npe];
      for (int a = 0; a < npe; ++a) code[(size_t)k * npe + a] = place[std::lower_bound(b, e, (int32_t)c[a]) - b];
    }
  }
}

// The lists of a set's row-owner tangent (ElemSet::rn, code).  adj: sorted neighbours of a node.
static void build_rows(const Plan& P, ElemSet& s, const std::vector<int64_t>& adj_ptr, const std::vector<int32_t>& adj) {
  const int d = P.d;
  s.rn_ptr_h.assign(1, 0);
  s.rn_h.clear();
  s.rn_max = 0;
  for (int64_t c = 0; c < P.n_chunks; ++c) {
    const int64_t end = std::min<int64_t>(P.n_free, (c + 1) * kSellC);
    for (int64_t row = c * kSellC, last = -1; row < end; ++row) {
      const int32_t n = P.red2full_h[row] / d;
      if (n == last) continue;
      last = n;
      if (s.inc_ptr_h[n + 1] > s.inc_ptr_h[n])
        s.rn_h.insert(s.rn_h.end(), {s.inc_ptr_h[n], s.inc_ptr_h[n + 1], n * d});
    }
    s.rn_ptr_h.push_back((int32_t)(s.rn_h.size() / 3));
    s.rn_max = std::max(s.rn_max, s.rn_ptr_h[c + 1] - s.rn_ptr_h[c]);
  }
  s.code_h.clear();
  s.code32_h.clear();
  if (P.max_row <= 1 << 13)
    build_codes<13>(P, s, s.code_h, adj_ptr, adj);
  else
    build_codes<29>(P, s, s.code32_h, adj_ptr, adj);
}

// Build the host-side reduced pattern, colours and row-owner lists (no device calls).
void plan_build_host(Plan& P, std::vector<std::vector<int32_t>>& conn_perm) {
  const int d = P.d;
  const int64_t N = P.n_nodes, ndof = P.n_dofs;
  APX_REQUIRE(!P.sets.empty(), APX_ERR_STATE, "plan has no element sets");

  // 1. free-DOF numbering (monotone, so reduced columns stay sorted)
  P.full2red_h.assign(ndof, -1);
  P.red2full_h.clear();
  for (int64_t g = 0; g < ndof; ++g)
    if (!P.dmask_host[g]) {
      P.full2red_h[g] = (int32_t)P.red2full_h.size();
      P.red2full_h.push_back((int32_t)g);
    }
  P.n_free = (int64_t)P.red2full_h.size();

  // 2. node -> element incidence over all sets
  std::vector<int64_t> inc_ptr(N + 1, 0);
  for (auto& s : P.sets)
    for (int64_t i = 0; i < s.n_elems * s.npe; ++i) {
      int64_t n = s.conn_host[i];
      APX_REQUIRE(n >= 0 && n < N, APX_ERR_ARG, "connectivity references a node outside [0, n_nodes)");
      inc_ptr[n + 1]++;
    }
  for (int64_t n = 0; n < N; ++n) inc_ptr[n + 1] += inc_ptr[n];
  std::vector<int64_t> fill(inc_ptr.begin(), inc_ptr.end() - 1);
  std::vector<std::pair<int32_t, int64_t>> inc(inc_ptr[N]);  // (set, element)
  for (int si = 0; si < (int)P.sets.size(); ++si) {
    auto& s = P.sets[si];
    for (int64_t e = 0; e < s.n_elems; ++e)
      for (int a = 0; a < s.npe; ++a) inc[fill[s.conn_host[e * s.npe + a]]++] = {si, e};
  }

  // 3. node adjacency (sorted unique) -> reduced DOF rows
  std::vector<int64_t> adj_ptr(N + 1, 0);
  std::vector<int32_t> adj;
  adj.reserve((size_t)N * (P.dim == 3 ? 27 : 9));
  std::vector<int32_t> tmp;
  for (int64_t n = 0; n < N; ++n) {
    tmp.clear();
    for (int64_t k = inc_ptr[n]; k < inc_ptr[n + 1]; ++k) {
      auto& s = P.sets[inc[k].first];
      const int64_t* c = &s.conn_host[inc[k].second * s.npe];
      for (int a = 0; a < s.npe; ++a) tmp.push_back((int32_t)c[a]);
    }
    std::sort(tmp.begin(), tmp.end());
    tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
    adj.insert(adj.end(), tmp.begin(), tmp.end());
    adj_ptr[n + 1] = (int64_t)adj.size();
  }
  P.indptr_h.assign(P.n_free + 1, 0);
  int64_t nnz = 0;
  for (int64_t row = 0; row < P.n_free; ++row) {
    int64_t g = P.red2full_h[row], n = g / d;
    for (int64_t k = adj_ptr[n]; k < adj_ptr[n + 1]; ++k)
      for (int c = 0; c < d; ++c) nnz += P.dmask_host[(int64_t)adj[k] * d + c] ? 0 : 1;
    APX_REQUIRE(nnz < (int64_t)INT32_MAX, APX_ERR_UNSUPPORTED, "reduced CSR exceeds int32 indexing");
    P.indptr_h[row + 1] = (int32_t)nnz;
  }
  P.nnz = nnz;
  P.indices_h.resize(nnz);
  for (int64_t row = 0; row < P.n_free; ++row) {
    int64_t g = P.red2full_h[row], n = g / d;
    int64_t o = P.indptr_h[row];
    for (int64_t k = adj_ptr[n]; k < adj_ptr[n + 1]; ++k)
      for (int c = 0; c < d; ++c) {
        int32_t col = P.full2red_h[(int64_t)adj[k] * d + c];
        if (col >= 0) P.indices_h[o++] = col;
      }
  }

  // 4. SELL-64 layout of the reduced matrix
  P.n_chunks = (P.n_free + kSellC - 1) / kSellC;
  P.sell_ptr_h.assign(P.n_chunks + 1, 0);
  P.bandwidth = 0;
  P.max_row = 0;
  for (int64_t c = 0; c < P.n_chunks; ++c) {
    int32_t w = 0;
    for (int64_t r = c * kSellC; r < std::min<int64_t>(P.n_free, (c + 1) * kSellC); ++r) {
      w = std::max(w, P.indptr_h[r + 1] - P.indptr_h[r]);
      if (P.indptr_h[r + 1] > P.indptr_h[r])  // columns are sorted
        P.bandwidth = std::max<int64_t>({P.bandwidth, r - P.indices_h[P.indptr_h[r]], P.indices_h[P.indptr_h[r + 1] - 1] - r});
    }
    P.max_row = std::max(P.max_row, (int)w);
    APX_REQUIRE((int64_t)P.sell_ptr_h[c] + (int64_t)w * kSellC < (int64_t)INT32_MAX, APX_ERR_UNSUPPORTED,
                "SELL layout exceeds int32 indexing");
    P.sell_ptr_h[c + 1] = P.sell_ptr_h[c] + w * kSellC;
  }
  P.sell_total = P.sell_ptr_h[P.n_chunks];
  P.sell_cols_h.assign(P.sell_total, 0);
  P.csr2sell_h.assign(P.nnz, 0);
  for (int64_t r = 0; r < P.n_free; ++r) {
    const int64_t c = r / kSellC, lane = r % kSellC;
    for (int32_t k = P.indptr_h[r]; k < P.indptr_h[r + 1]; ++k) {
      const int64_t s = P.sell_ptr_h[c] + (int64_t)(k - P.indptr_h[r]) * kSellC + lane;
      P.sell_cols_h[s] = P.indices_h[k];
      P.csr2sell_h[k] = (int32_t)s;
    }
  }

  find_lines(P);

  // 4b. structured Q1 grids (owner-tile kernels)
  for (auto& s : P.sets) {
    s.structured = 0;
    if (P.dim != 2 || s.npe != 4 || s.n_elems < 1 || s.conn_host[0] != 0) continue;
    const int64_t ny = s.conn_host[3] - 1;
    if (ny < 1 || s.n_elems % ny) continue;
    const int64_t nx = s.n_elems / ny;
    if ((nx + 1) * (ny + 1) != P.n_nodes) continue;
    bool ok = true;
    for (int64_t e = 0; e < s.n_elems && ok; ++e) {
      const int64_t i = e / ny, j = e % ny, b = i * (ny + 1) + j;
      const int64_t* c = &s.conn_host[e * 4];
      ok = c[0] == b && c[1] == b + 1 && c[2] == b + ny + 2 && c[3] == b + ny + 1;
    }
    if (ok) {
      s.structured = 1;
      s.gnx = nx;
      s.gny = ny;
    }
  }
  // 4c. is the reduced pattern the free-node 3 x 3 stencil of that grid (one DOF per node)?
  P.stencil_pattern = false;
  for (auto& s : P.sets) {
    if (!s.structured || P.d != 1) continue;
    const int64_t nx = s.gnx, ny = s.gny;
    bool ok = true;
    for (int64_t I = 0; I <= nx && ok; ++I)
      for (int64_t J = 0; J <= ny && ok; ++J) {
        const int32_t row = P.full2red_h[I * (ny + 1) + J];
        if (row < 0) continue;
        int32_t k = P.indptr_h[row];
        for (int dI = -1; dI <= 1 && ok; ++dI)
          for (int dJ = -1; dJ <= 1 && ok; ++dJ) {
            const int64_t I2 = I + dI, J2 = J + dJ;
            if (I2 < 0 || I2 > nx || J2 < 0 || J2 > ny) continue;
            const int32_t col = P.full2red_h[I2 * (ny + 1) + J2];
            if (col < 0) continue;
            ok = k < P.indptr_h[row + 1] && P.indices_h[k] == col;
            ++k;
          }
        ok = ok && k == P.indptr_h[row + 1];
      }
    P.stencil_pattern = ok;
    break;
  }

  // 4d. lists of the row-owner kernels, for sets whose residual or tangent has no owner tiles
  const bool tiles = tangent_by_tiles(P);
  for (auto& s : P.sets) {
    const bool rows = !tiles && s.model != APX_MODEL_LINE_TRACTION;
    if (!rows && tile_supported(P, s, 0)) continue;
    build_incidence(P, s);
    if (rows) build_rows(P, s, adj_ptr, adj);
  }

  // 5. greedy element colouring per set (node-disjoint colours)
  conn_perm.assign(P.sets.size(), {});
  std::vector<uint64_t> used(N);
  for (int si = 0; si < (int)P.sets.size(); ++si) {
    auto& s = P.sets[si];
    std::fill(used.begin(), used.end(), 0ull);
    std::vector<uint8_t> colour(s.n_elems);
    int ncol = 0;
    for (int64_t e = 0; e < s.n_elems; ++e) {
      uint64_t m = 0;
      const int64_t* c = &s.conn_host[e * s.npe];
      for (int a = 0; a < s.npe; ++a) m |= used[c[a]];
      APX_REQUIRE(~m != 0ull, APX_ERR_UNSUPPORTED, "element colouring needs more than 64 colours");
      int col = __builtin_ctzll(~m);
      colour[e] = (uint8_t)col;
      ncol = std::max(ncol, col + 1);
      for (int a = 0; a < s.npe; ++a) used[c[a]] |= (1ull << col);
    }
    s.colour_offsets.assign(ncol + 1, 0);
    for (int64_t e = 0; e < s.n_elems; ++e) s.colour_offsets[colour[e] + 1]++;
    for (int c = 0; c < ncol; ++c) s.colour_offsets[c + 1] += s.colour_offsets[c];
    std::vector<int64_t> pos(s.colour_offsets.begin(), s.colour_offsets.end() - 1);
    std::vector<int64_t> perm(s.n_elems);
    for (int64_t e = 0; e < s.n_elems; ++e) perm[pos[colour[e]]++] = e;  // stable within a colour

    auto& cp = conn_perm[si];
    cp.resize(s.n_elems * s.npe);
    for (int64_t i = 0; i < s.n_elems; ++i) {
      const int64_t* c = &s.conn_host[perm[i] * s.npe];
      for (int a = 0; a < s.npe; ++a) cp[i * s.npe + a] = (int32_t)c[a];
    }
  }
}

// The row-owner lists of a set (build_incidence, build_rows) to the device.
static void upload_rows(Plan& P, ElemSet& S) {
  if (S.inc_ptr_h.empty()) return;
  std::vector<int32_t> c32(S.conn_host.begin(), S.conn_host.end()), nodes;
  S.conn_orig.upload(c32.data(), c32.size());
  for (int64_t n = 0; n < P.n_nodes; ++n)
    if (S.inc_ptr_h[n + 1] > S.inc_ptr_h[n]) nodes.push_back((int32_t)n);
  S.n_touched = (int64_t)nodes.size();
  S.touched_all = S.n_touched == P.n_nodes;
  if (!S.touched_all) S.touched.upload(nodes.data(), nodes.size());
  S.inc_ptr.upload(S.inc_ptr_h.data(), S.inc_ptr_h.size());
  S.inc.upload(S.inc_h.data(), S.inc_h.size());
  if (!S.rn_ptr_h.empty()) {
    S.rn_ptr.upload(S.rn_ptr_h.data(), S.rn_ptr_h.size());
    S.rn.upload(S.rn_h.data(), S.rn_h.size());
    if (S.code32_h.empty())
      S.code.upload(S.code_h.data(), S.code_h.size());
    else
      S.code32.upload(S.code32_h.data(), S.code32_h.size());
  }
  std::vector<int32_t>().swap(S.inc_ptr_h);
  std::vector<int32_t>().swap(S.inc_h);
  std::vector<int32_t>().swap(S.rn_ptr_h);
  std::vector<int32_t>().swap(S.rn_h);
  std::vector<uint16_t>().swap(S.code_h);
  std::vector<uint32_t>().swap(S.code32_h);
}

void plan_finalize(Plan& P) {
  auto t0 = std::chrono::steady_clock::now();
  std::vector<std::vector<int32_t>> conn_perm;
  plan_build_host(P, conn_perm);

  // SoA coordinates
  std::vector<double> soa(P.n_nodes * P.dim);
  for (int64_t n = 0; n < P.n_nodes; ++n)
    for (int k = 0; k < P.dim; ++k) soa[k * P.n_nodes + n] = P.coords_host[n * P.dim + k];
  P.coords.upload(soa.data(), soa.size());
  P.dmask.upload(P.dmask_host.data(), P.dmask_host.size());
  P.full2red.upload(P.full2red_h.data(), P.full2red_h.size());
  P.red2full.upload(P.red2full_h.data(), P.red2full_h.size());
  P.indptr.upload(P.indptr_h.data(), P.indptr_h.size());
  P.indices.upload(P.indices_h.data(), P.indices_h.size());
  std::vector<int32_t> ds(P.n_free);
  for (int64_t r = 0; r < P.n_free; ++r) {
    const int32_t* b = P.indices_h.data() + P.indptr_h[r];
    const int32_t* e = P.indices_h.data() + P.indptr_h[r + 1];
    const int32_t* f = std::lower_bound(b, e, (int32_t)r);
    APX_REQUIRE(f != e && *f == r, APX_ERR_INTERNAL, "missing diagonal entry in reduced CSR");
    ds[r] = P.csr2sell_h[f - P.indices_h.data()];
  }
  P.diag_slot.upload(ds.data(), ds.size());
  P.sell_ptr.upload(P.sell_ptr_h.data(), P.sell_ptr_h.size());
  {
    // int16 column offsets when every stored entry's offset from its row fits
    std::vector<int16_t> dcol(P.sell_total, 0);
    bool fits = true;
    for (int64_t r = 0; r < P.n_free && fits; ++r) {
      const int64_t c = r / kSellC, lane = r % kSellC;
      for (int32_t k = P.indptr_h[r]; k < P.indptr_h[r + 1]; ++k) {
        const int64_t s = P.sell_ptr_h[c] + (int64_t)(k - P.indptr_h[r]) * kSellC + lane;
        const int64_t d = (int64_t)P.sell_cols_h[s] - r;
        if (d < INT16_MIN || d > INT16_MAX) {
          fits = false;
          break;
        }
        dcol[s] = (int16_t)d;
      }
    }
    if (fits) {
      P.sell_dcol.upload(dcol.data(), dcol.size());
      P.sell_cols = DevBuf<int32_t>();
    } else {
      P.sell_dcol = DevBuf<int16_t>();
      P.sell_cols.upload(P.sell_cols_h.data(), P.sell_cols_h.size());
    }
  }
  P.csr2sell.upload(P.csr2sell_h.data(), P.csr2sell_h.size());
  if (P.line) P.irregular.upload(P.irregular_h.data(), P.irregular_h.size());
  std::vector<int32_t>().swap(P.sell_cols_h);
  std::vector<int32_t>().swap(P.csr2sell_h);
  size_t words = 0;  // of element vectors
  for (size_t si = 0; si < P.sets.size(); ++si) {
    ElemSet& S = P.sets[si];
    S.conn.upload(conn_perm[si].data(), conn_perm[si].size());
    const bool vectors = !S.inc_ptr_h.empty() && !tile_supported(P, S, 0) && S.model != APX_MODEL_LINE_TRACTION;
    if (vectors) words = std::max(words, (size_t)(S.n_elems * S.npe * P.d));
    upload_rows(P, S);
  }
  if (words) P.element_vectors.alloc(words);
  // pinned host scalars: [0, 512) B PCG flags and norms, [512, 768) B FCG state copies,
  // [768, 1024) B the final Krylov state of an allocation-free PCG run
  if (!P.pinned) APX_HIP(hipHostMalloc((void**)&P.pinned, 128 * sizeof(double), hipHostMallocDefault));
  if (!P.ev0) APX_HIP(hipEventCreate(&P.ev0));
  if (!P.ev1) APX_HIP(hipEventCreate(&P.ev1));
  P.finalized = true;
  P.build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace apx
