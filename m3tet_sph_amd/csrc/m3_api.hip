// C ABI of libm3stokes: mesh/BC set-up (host), assembly, Galerkin
// restriction, coarse factorisation, MGPCG and the Patera pressure iteration
// (flow3d_patera_mg_sph_p.m:374-681), all on one HIP stream.
#include <omp.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <numeric>
#include <unordered_map>

#include "m3_internal.h"

namespace m3 {
void chol_analyse(m3_ctx *c);
}

// ------------------------------------------------------------------ Sell build
void Sell::build(int64_t nrow_, int64_t ncol_, const std::vector<int64_t> &ptr,
                 const std::vector<int32_t> &cols, int bs_, const std::vector<int32_t> *place) {
  nrow = nrow_;
  ncol = ncol_;
  bs = bs_;
  const int64_t nsl = (nrow + 63) / 64;
  h_slice_ptr.assign(nsl + 1, 0);
  h_rowlen.assign(nrow, 0);
  for (int64_t r = 0; r < nrow; ++r) h_rowlen[r] = (int32_t)(ptr[r + 1] - ptr[r]);
  h_perm.clear();
  h_ipos.clear();
  h_vperm.clear();
  h_vpos.clear();
  nwin = 0;
  if (place) {
    h_perm = *place;
    h_ipos.resize(nrow);
    for (int64_t q = 0; q < nrow; ++q) h_ipos[h_perm[q]] = (int32_t)q;
  }
  auto row_at = [&](int64_t q) { return h_perm.empty() ? q : (int64_t)h_perm[q]; };
  for (int64_t sl = 0; sl < nsl; ++sl) {
    int mx = 0;
    for (int64_t q = 64 * sl; q < std::min(nrow, 64 * sl + 64); ++q) mx = std::max(mx, h_rowlen[row_at(q)]);
    h_slice_ptr[sl + 1] = h_slice_ptr[sl] + 64 * (int64_t)mx;
  }
  nslot = h_slice_ptr[nsl];
  nnz = ptr[nrow];
  h_col.assign(nslot, -1);
  for (int64_t r = 0; r < nrow; ++r) {
    const int64_t base = base_of(r);
    for (int64_t k = ptr[r]; k < ptr[r + 1]; ++k) h_col[base + (k - ptr[r]) * 64] = cols[k];
  }
  slice_ptr.upload(h_slice_ptr);
  rowlen.upload(h_rowlen);
  col.upload(h_col);
  if (!h_perm.empty()) {
    perm.upload(h_perm);
    ipos.upload(h_ipos);
  }
  val.alloc((size_t)nslot * bs);
}

namespace {

// Host array whose pages the threads that fill it touch first (a vector clears
// them one after the other: half the time of a large one's whole use)
template <class T>
struct HostArr {
  std::unique_ptr<T[]> p;
  size_t n;
  explicit HostArr(size_t count) : p(new T[count]), n(count) {}
  T &operator[](size_t i) { return p[i]; }
};

// The different vector places that a window of rows gathers: an open-addressed
// table of SIZE entries (at most half of them taken), so that a thread needs
// 128 KB whatever the mesh, and a look-up stays in its L2.
struct WindowTable {
  static constexpr int SIZE = 16384, FULL = SIZE / 2;
  std::vector<int32_t> key = std::vector<int32_t>(SIZE, -1), rank = std::vector<int32_t>(SIZE);
  std::vector<int32_t> list;  // the places, in the order of their first look-up
  WindowTable() { list.reserve(FULL + 1); }
  void clear() {
    std::fill(key.begin(), key.end(), -1);
    list.clear();
  }
  // entry of place i, added if it is new; no more than FULL places
  int at(int32_t i) {
    uint32_t h = ((uint32_t)i * 2654435761u) >> 18;
    while (key[h] != i) {
      if (key[h] < 0) {
        key[h] = i;
        list.push_back(i);
        break;
      }
      h = (h + 1) & (SIZE - 1);
    }
    return (int)h;
  }
  // list ascending, rank of every entry in it
  void number() {
    std::sort(list.begin(), list.end());
    for (size_t r = 0; r < list.size(); ++r) rank[at(list[r])] = (int32_t)r;
  }
};

}  // namespace

m3::WindowFit Sell::build_windows(const std::vector<int32_t> &order, const std::vector<int32_t> &first,
                                  const m3::SweepRule &rule) {
  const int64_t nw = (int64_t)first.size() - 1;
  std::vector<std::vector<int32_t>> lists(nw);
  HostArr<uint16_t> h_idx((size_t)nslot), h_lrow(nrow);
  HostArr<int32_t> h_plen(nrow);
  std::vector<int32_t> pos(nrow);
#pragma omp parallel for schedule(static)
  for (int64_t i = 0; i < nrow; ++i) pos[order[i]] = (int32_t)i;
  bool fits = true, memory = true;  // an exception must not leave a parallel region
  std::vector<WindowTable> tables(omp_get_max_threads());
#pragma omp parallel for schedule(dynamic, 4) reduction(&& : fits, memory)
  for (int64_t b = 0; b < nw; ++b) {
    WindowTable &t = tables[omp_get_thread_num()];
    t.clear();
    const int64_t q0 = first[b], q1 = first[b + 1];
    const int cap = rule.most(q1 - q0);
    // padding slots are never read; they hold the window's first place
    std::fill(&h_idx[h_slice_ptr[q0 >> 6]], &h_idx[0] + h_slice_ptr[(q1 + 63) >> 6], (uint16_t)0);
    bool ok = true;
    for (int64_t q = q0; q < q1 && ok; ++q) {
      const int len = h_rowlen[h_perm[q]];
      const int64_t base = h_slice_ptr[q >> 6] + (q & 63);
      h_plen[q] = len;
      h_lrow[q] = (uint16_t)(pos[h_perm[q]] - q0);
      for (int k = 0; k < len && ok; ++k) {
        h_idx[base + 64 * (int64_t)k] = (uint16_t)t.at(pos[h_col[base + 64 * (int64_t)k]]);
        ok = (int)t.list.size() <= cap;
      }
    }
    if (!ok) {
      fits = false;
      continue;
    }
    t.number();
    for (int64_t q = q0; q < q1; ++q) {
      const int64_t base = h_slice_ptr[q >> 6] + (q & 63);
      for (int k = 0; k < h_plen[q]; ++k) {
        uint16_t &e = h_idx[base + 64 * (int64_t)k];
        e = (uint16_t)t.rank[e];
      }
    }
    try {
      lists[b] = t.list;
    } catch (const std::bad_alloc &) {
      memory = false;
    }
  }
  if (!memory) throw std::bad_alloc();
  if (!fits) return m3::WindowFit::oversized;
  int64_t total = 0;
  for (const auto &l : lists) total += (int64_t)l.size();
  if (total > rule.per_row * nrow || total > INT32_MAX) return m3::WindowFit::scattered;
  std::vector<int2> h_win(nw + 1, int2{0, 0});
  umax = 0;
  for (int64_t b = 0; b < nw; ++b) {
    umax = std::max(umax, (int)lists[b].size());
    h_win[b + 1] = int2{first[b + 1], h_win[b].y + (int32_t)lists[b].size()};
  }
  HostArr<int32_t> h_list(h_win[nw].y);
#pragma omp parallel for schedule(static)
  for (int64_t b = 0; b < nw; ++b) std::copy(lists[b].begin(), lists[b].end(), &h_list[h_win[b].y]);
  nwin = (int)nw;
  plen.upload(h_plen.p.get(), h_plen.n);
  win.upload(h_win);
  list.upload(h_list.p.get(), h_list.n);
  idx.upload(h_idx.p.get(), h_idx.n);
  lrow.upload(h_lrow.p.get(), h_lrow.n);
  h_vperm = order;
  h_vpos.swap(pos);
  vperm.upload(h_vperm);
  vpos.upload(h_vpos);
  return m3::WindowFit::ok;
}

namespace {

// The nodes along a Hilbert curve of their coordinates (J. Skilling,
// "Programming the Hilbert curve", AIP Conf. Proc. 707, 2004: axes to the
// transposed Hilbert integer), 16 bits an axis; equal keys in index order.
std::vector<int32_t> hilbert_order(const double *X, int64_t n) {
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int64_t i = 0; i < n; ++i)
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], X[3 * i + k]);
      hi[k] = std::max(hi[k], X[3 * i + k]);
    }
  const double w = std::max({hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]});
  constexpr int BITS = 16;
  std::vector<std::pair<uint64_t, int32_t>> key(n);
#pragma omp parallel for schedule(static)
  for (int64_t i = 0; i < n; ++i) {
    uint32_t x[3];
    for (int k = 0; k < 3; ++k) x[k] = w > 0 ? (uint32_t)((X[3 * i + k] - lo[k]) / w * 65535.0) : 0u;
    for (uint32_t q = 1u << (BITS - 1); q > 1; q >>= 1) {
      const uint32_t m = q - 1;
      for (int k = 0; k < 3; ++k) {
        if (x[k] & q) {
          x[0] ^= m;
        } else {
          const uint32_t t = (x[0] ^ x[k]) & m;
          x[0] ^= t;
          x[k] ^= t;
        }
      }
    }
    for (int k = 1; k < 3; ++k) x[k] ^= x[k - 1];
    uint32_t t = 0;
    for (uint32_t q = 1u << (BITS - 1); q > 1; q >>= 1)
      if (x[2] & q) t ^= q - 1;
    uint64_t code = 0;
    for (int b = BITS - 1; b >= 0; --b)
      for (int k = 0; k < 3; ++k) code = (code << 1) | (((x[k] ^ t) >> b) & 1u);
    key[i] = {code, (int32_t)i};
  }
  // sorted in pieces, then merged pairwise
  constexpr int PIECES = 16;
  std::vector<int64_t> cut(PIECES + 1);
  for (int p = 0; p <= PIECES; ++p) cut[p] = n * p / PIECES;
#pragma omp parallel for schedule(dynamic, 1)
  for (int p = 0; p < PIECES; ++p) std::sort(key.begin() + cut[p], key.begin() + cut[p + 1]);
  for (int s = 1; s < PIECES; s *= 2) {
#pragma omp parallel for schedule(dynamic, 1)
    for (int p = 0; p < PIECES; p += 2 * s)
      std::inplace_merge(key.begin() + cut[p], key.begin() + cut[p + s], key.begin() + cut[p + 2 * s]);
  }
  std::vector<int32_t> order(n);
  for (int64_t i = 0; i < n; ++i) order[i] = key[i].second;
  return order;
}

// Placement of a level whose sweeps run on windows: the Hilbert order of the
// nodes, longest rows first inside every window.
std::vector<int32_t> window_placement(const std::vector<int32_t> &order, const std::vector<int32_t> &first,
                                      const std::vector<int64_t> &ptr) {
  std::vector<int32_t> p = order;
#pragma omp parallel for schedule(static)
  for (size_t b = 0; b < first.size() - 1; ++b)
    std::stable_sort(p.begin() + first[b], p.begin() + first[b + 1],
                     [&](int32_t i, int32_t j) { return ptr[i + 1] - ptr[i] > ptr[j + 1] - ptr[j]; });
  return p;
}

// The windows again, those that gather too much halved (at a slice) until they
// do not; empty if a slice alone does
std::vector<int32_t> split_windows(const std::vector<int32_t> &order, const std::vector<int32_t> &first,
                                   const std::vector<int64_t> &ptr, const std::vector<int32_t> &cols,
                                   const m3::SweepRule &rule) {
  std::vector<int32_t> pos(order.size());
  for (size_t i = 0; i < order.size(); ++i) pos[order[i]] = (int32_t)i;
  WindowTable t;
  auto fits = [&](int32_t q0, int32_t q1) {
    t.clear();
    for (int32_t q = q0; q < q1; ++q)
      for (int64_t k = ptr[order[q]]; k < ptr[order[q] + 1]; ++k) {
        t.at(pos[cols[k]]);
        if ((int)t.list.size() > rule.most(q1 - q0)) return false;
      }
    return true;
  };
  std::vector<int32_t> out{0}, todo;  // todo: ends of the pieces still to look at, the next one last
  for (size_t b = 0; b + 1 < first.size(); ++b) {
    todo.assign(1, first[b + 1]);
    while (!todo.empty()) {
      const int32_t q0 = out.back(), q1 = todo.back();
      if (fits(q0, q1)) {
        out.push_back(q1);
        todo.pop_back();
      } else if (q1 - q0 <= 64) {
        return {};
      } else {
        todo.push_back(q0 + ((q1 - q0 + 127) / 128) * 64);
      }
    }
  }
  return out;
}

using clk = std::chrono::steady_clock;
double secs(clk::time_point a, clk::time_point b) {
  return std::chrono::duration<double>(b - a).count();
}

// rows = nodes 0..nrow-1; for each element, row nodes rsel[] x col nodes csel[].
// Sorted, duplicate-free column lists: every row gathers the columns of its
// incident elements into its own stretch of one buffer (sized by the
// incidence counts), sorts and compacts it; rows are independent (OpenMP).
void adjacency(const std::vector<int32_t> &el2nod, int64_t nel, int64_t nrow, int nr, const int *rsel,
               int nc, const int *csel, std::vector<int64_t> &ptr, std::vector<int32_t> &cols) {
  // node -> elements
  std::vector<int64_t> eptr(nrow + 1, 0);
  for (int64_t e = 0; e < nel; ++e)
    for (int i = 0; i < nr; ++i) eptr[el2nod[10 * e + rsel[i]] + 1]++;
  for (int64_t n = 0; n < nrow; ++n) eptr[n + 1] += eptr[n];
  std::vector<int64_t> fill(eptr.begin(), eptr.end() - 1);
  std::vector<int32_t> elist(eptr[nrow]);
  for (int64_t e = 0; e < nel; ++e)
    for (int i = 0; i < nr; ++i) elist[fill[el2nod[10 * e + rsel[i]]]++] = (int32_t)e;
  std::vector<int32_t> buf((size_t)eptr[nrow] * nc);
  std::vector<int64_t> len(nrow);
#pragma omp parallel for schedule(dynamic, 1024)
  for (int64_t n = 0; n < nrow; ++n) {
    int32_t *b = buf.data() + eptr[n] * nc, *w = b;
    for (int64_t k = eptr[n]; k < eptr[n + 1]; ++k)
      for (int j = 0; j < nc; ++j) *w++ = el2nod[10 * (int64_t)elist[k] + csel[j]];
    std::sort(b, w);
    len[n] = std::unique(b, w) - b;
  }
  ptr.assign(nrow + 1, 0);
  for (int64_t n = 0; n < nrow; ++n) ptr[n + 1] = ptr[n] + len[n];
  cols.resize(ptr[nrow]);
#pragma omp parallel for schedule(static)
  for (int64_t n = 0; n < nrow; ++n)
    std::copy(buf.begin() + eptr[n] * nc, buf.begin() + eptr[n] * nc + len[n], cols.begin() + ptr[n]);
}

const int ALL10[10] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9};
const int V4[4] = {0, 1, 2, 3};

struct Timer {
  hipEvent_t a, b;
  hipStream_t s;
  explicit Timer(hipStream_t st) : s(st) {
    (void)hipEventCreate(&a);
    (void)hipEventCreate(&b);
    (void)hipEventRecord(a, s);
  }
  double stop() {
    (void)hipEventRecord(b, s);
    (void)hipEventSynchronize(b);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, a, b);
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return ms * 1e-3;
  }
};

int check_err(m3_ctx *c) {
  int e = 0;
  HIPCHECK(hipMemcpyAsync(&e, c->errflag.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  HIPCHECK(hipStreamSynchronize(c->stream));
  return e;
}

void raise_flags(int e) {
  if (e & 1) throw M3Error(M3_E_NUMERIC, "negative Jacobi");
  if (e & 2) throw M3Error(M3_E_NUMERIC, "integration point has theta = 0 (det(J_CS) = Inf)");
  if (e & 4) throw M3Error(M3_E_NUMERIC, "Calculated a zero or negative viscosity");
  if (e & 8) throw M3Error(M3_E_MESH, "element block missing from the sparse pattern");
  if (e & 16) throw M3Error(M3_E_NUMERIC, "coarse matrix is not positive definite");
  if (e & 32) throw M3Error(M3_E_NUMERIC, "Solution contains NaNs");
}

template <class F>
int guard(m3_ctx *c, F &&f) {
  if (!c) {
    m3::set_context_free_error("null context");
    return M3_E_ARG;
  }
  try {
    HIPCHECK(hipSetDevice(c->device));
    f();
    c->err.clear();
    return M3_OK;
  } catch (const M3Error &e) {
    c->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    c->err = e.what();
    return M3_E_ARG;
  }
}

void ensure(DBuf<double> &b, size_t n) {
  if (b.n != n) b.alloc(n);
}

}  // namespace

extern "C" {

int m3_create(m3_ctx **ctx, int hip_device) {
  if (!ctx) return M3_E_ARG;
  *ctx = nullptr;
  m3_ctx *c = new m3_ctx();
  c->device = hip_device;
  try {
    int ndev = 0;
    HIPCHECK(hipGetDeviceCount(&ndev));
    M3_REQUIRE(ndev > 0, M3_E_HIP, "no HIP device visible");
    M3_REQUIRE(hip_device >= 0 && hip_device < ndev, M3_E_ARG, "invalid HIP device index");
    HIPCHECK(hipSetDevice(hip_device));
    HIPCHECK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIPCHECK(hipHostMalloc(&c->h_scal, 64 * sizeof(double)));
    HIPCHECK(hipHostMalloc(&c->h_part, m3::HOST_PARTS * sizeof(double)));
    c->scal.alloc(64);
    c->errflag.alloc(1);
    m3::upload_sf_tables();
  } catch (const M3Error &e) {
    c->err = e.what();
    const int code = e.code;
    *ctx = c;  // returned so that m3_last_error works; caller destroys it
    return code;
  }
  *ctx = c;
  return M3_OK;
}

void m3_destroy(m3_ctx *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  {
    m3_ctx tmp;  // release device buffers before the stream
    std::swap(tmp.L, c->L);
  }
  if (c->h_scal) (void)hipHostFree(c->h_scal);
  if (c->h_part) (void)hipHostFree(c->h_part);
  if (c->ev_start) (void)hipEventDestroy(c->ev_start);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char *m3_last_error(const m3_ctx *c) { return c ? c->err.c_str() : m3::context_free_error(); }

int m3_set_mesh(m3_ctx *c, const m3_mesh_desc *m) {
  return guard(c, [&] {
    M3_REQUIRE(m, M3_E_ARG, "null mesh descriptor");
    M3_REQUIRE(m->nmg >= 2 && m->nmg <= M3_MAX_LEVELS, M3_E_ARG, "nmg must be in 2..8");
    const int nmg = m->nmg;
    c->nmg = nmg;
    // M3_SETUP_TIMING=1 prints the time of each set-up phase to stderr
    const bool report = std::getenv("M3_SETUP_TIMING") != nullptr;
    auto tp = clk::now();
    auto mark = [&](const char *what) {
      if (!report) return;
      const auto now = clk::now();
      std::fprintf(stderr, "[m3_set_mesh] %-34s %8.3f s\n", what, secs(tp, now));
      tp = now;
    };
    c->L.clear();
    c->adv.ready = c->slm.ready = c->dif.ready = c->dif.assembled = false;
    c->L.resize(nmg);
    c->have_mesh = c->have_bc = c->assembled = c->restricted = c->factored = c->have_mixed = false;
    c->pack16_fresh = false;
    c->have_fields = false;
    c->have_solution = false;
    c->have_ref = false;  // a refined region belongs to the mesh it was set for
    c->g_valid = false;
    c->csc.reset();
    for (int l = 0; l < nmg; ++l) {
      LevelDev &lv = c->L[l];
      lv.nel = m->nel[l];
      lv.nnod = m->nnod[l];
      lv.nV = m->nVnod[l];
      M3_REQUIRE(m->EL2NOD[l] && lv.nel > 0 && lv.nnod > 0, M3_E_ARG, "empty level");
      lv.h_el2nod.resize(10 * lv.nel);
      for (int64_t i = 0; i < 10 * lv.nel; ++i) {
        const int64_t v = (int64_t)m->EL2NOD[l][i] - 1;
        M3_REQUIRE(v >= 0 && v < lv.nnod, M3_E_MESH, "EL2NOD entry out of range");
        lv.h_el2nod[i] = (int32_t)v;
      }
      for (int64_t e = 0; e < lv.nel; ++e)
        for (int i = 0; i < 4; ++i)
          M3_REQUIRE(lv.h_el2nod[10 * e + i] < lv.nV, M3_E_MESH, "vertices must be numbered first");
      if (l > 0) {
        M3_REQUIRE(c->L[l - 1].nel == 8 * lv.nel, M3_E_MESH, "finer level must have 8x the elements");
        M3_REQUIRE(c->L[l - 1].nV == lv.nnod, M3_E_MESH, "fine vertices must be the coarse P2 nodes");
      }
      lv.el2nod.upload(lv.h_el2nod);
      std::vector<int64_t> ptr;
      std::vector<int32_t> cols;
      adjacency(lv.h_el2nod, lv.nel, lv.nnod, 10, ALL10, 10, ALL10, ptr, cols);
      const int w = l < nmg - 1 ? m3::sweep_window(c->sweep_rule, lv.nnod) : 0;
      if (w) {
        M3_REQUIRE(m->GCOORD, M3_E_ARG, "missing GCOORD");
        const std::vector<int32_t> order = hilbert_order(m->GCOORD, lv.nnod);
        std::vector<int32_t> first;
        for (int64_t q = 0; q < lv.nnod; q += w) first.push_back((int32_t)q);
        first.push_back((int32_t)lv.nnod);
        auto build = [&] {
          const std::vector<int32_t> place = window_placement(order, first, ptr);
          lv.K.build(lv.nnod, lv.nnod, ptr, cols, 9, &place);
        };
        build();
        mark("level connectivity + K pattern");
        m3::WindowFit fit = lv.K.build_windows(order, first, c->sweep_rule);
        if (fit == m3::WindowFit::oversized) {
          first = split_windows(order, first, ptr, cols, c->sweep_rule);
          if (!first.empty()) {
            build();
            fit = lv.K.build_windows(order, first, c->sweep_rule);
          }
        }
        if (fit != m3::WindowFit::ok) lv.K.build(lv.nnod, lv.nnod, ptr, cols, 9);
        mark("sweep windows");
      } else {
        lv.K.build(lv.nnod, lv.nnod, ptr, cols, 9);
      }
      if (l < nmg - 1) lv.Kel.alloc((size_t)lv.nel * KEL);
      mark("level connectivity + K pattern");
    }
    LevelDev &f = c->L[0];
    c->nel = f.nel;
    c->nnod = f.nnod;
    c->nV = f.nV;
    // G (velocity node x vertex), GT, M
    {
      std::vector<int64_t> ptr;
      std::vector<int32_t> cols;
      adjacency(f.h_el2nod, f.nel, f.nnod, 10, ALL10, 4, V4, ptr, cols);
      c->G.build(f.nnod, f.nV, ptr, cols, 3);
      adjacency(f.h_el2nod, f.nel, f.nV, 4, V4, 10, ALL10, ptr, cols);
      c->GT.build(f.nV, f.nnod, ptr, cols, 3);
      adjacency(f.h_el2nod, f.nel, f.nV, 4, V4, 4, V4, ptr, cols);
      c->M.build(f.nV, f.nV, ptr, cols, 1);
      mark("G, GT, M patterns");
      // slot of every element block in K (10x10), G (10x4), GT (4x10), M (4x4):
      // the assembly scatters without searching the sparse rows
      M3_REQUIRE(std::max({f.K.nslot, c->G.nslot, c->GT.nslot, c->M.nslot}) < (int64_t)INT32_MAX, M3_E_MESH,
                 "sparse pattern too large for 32-bit slots");
      c->asm_slots.alloc((size_t)f.nel * ASM_SLOTS);
      c->errflag.zero(c->stream);
      m3::launch_slots(c);
      raise_flags(check_err(c));
      mark("element slot map");
      // node -> (element, local node) incidence for the row-owner assembly of K
      std::vector<int64_t> iptr(f.nnod + 1, 0);
      for (int64_t k = 0; k < 10 * f.nel; ++k) ++iptr[f.h_el2nod[k] + 1];
      for (int64_t n = 0; n < f.nnod; ++n) iptr[n + 1] += iptr[n];
      std::vector<int64_t> fill(iptr.begin(), iptr.end() - 1);
      std::vector<int32_t> inc(10 * f.nel);
      for (int64_t e = 0; e < f.nel; ++e)
        for (int a = 0; a < 10; ++a) inc[fill[f.h_el2nod[10 * e + a]]++] = (int32_t)(10 * e + a);
      c->inc_ptr.upload(iptr);
      c->inc.upload(inc);
      int maxlen = 0;
      for (int64_t r = 0; r < f.nnod; ++r) maxlen = std::max(maxlen, f.K.h_rowlen[r]);
      c->gather_K = maxlen <= 128 && 10 * f.nel < (int64_t)INT32_MAX;
      f.K.val.zero(c->stream);  // padding slots stay zero
      mark("node incidence");
      if (m3::build_contrib(c, 0)) c->gather_K = true;
      mark("slot contribution lists");
    }
    // coarse levels: the Galerkin products write element matrices, summed per
    // row by the same gather (slot map of the 100 element blocks, incidence)
    for (int l = 1; l < nmg; ++l) {
      LevelDev &lv = c->L[l];
      int maxlen = 0;
      for (int64_t r = 0; r < lv.nnod; ++r) maxlen = std::max(maxlen, lv.K.h_rowlen[r]);
      lv.gather = maxlen <= 128 && 10 * lv.nel < (int64_t)INT32_MAX && lv.K.nslot < (int64_t)INT32_MAX;
      lv.K.val.zero(c->stream);  // padding slots stay zero
      if (!lv.gather) continue;
      if (!lv.Kel.p) lv.Kel.alloc((size_t)lv.nel * KEL);
      lv.kslots.alloc((size_t)lv.nel * 100);
      c->errflag.zero(c->stream);
      m3::launch_kslots(c, l);
      raise_flags(check_err(c));
      std::vector<int64_t> iptr(lv.nnod + 1, 0);
      for (int64_t k = 0; k < 10 * lv.nel; ++k) ++iptr[lv.h_el2nod[k] + 1];
      for (int64_t n = 0; n < lv.nnod; ++n) iptr[n + 1] += iptr[n];
      std::vector<int64_t> fill(iptr.begin(), iptr.end() - 1);
      std::vector<int32_t> inc(10 * lv.nel);
      for (int64_t e = 0; e < lv.nel; ++e)
        for (int a = 0; a < 10; ++a) inc[fill[lv.h_el2nod[10 * e + a]]++] = (int32_t)(10 * e + a);
      lv.inc_ptr.upload(iptr);
      lv.inc.upload(inc);
      m3::build_contrib(c, l);
    }
    mark("coarse slot maps + incidence");
    // coordinates and nodal frames (make_rotation_matrix.m:69-110)
    std::vector<double> X(3 * f.nnod), S(3 * f.nnod), fr(9 * f.nnod);
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < f.nnod; ++n) {
      for (int k = 0; k < 3; ++k) {
        X[3 * n + k] = m->GCOORD[3 * n + k];
        S[3 * n + k] = m->GCOORD_SPH[3 * n + k];
      }
      const double x = X[3 * n], y = X[3 * n + 1], z = X[3 * n + 2];
      const double th = std::atan2(std::sqrt(x * x + y * y), z);
      double ph = std::atan2(y, x);
      if (ph < 0) ph += 2 * M_PI;
      const double ct = std::cos(th), st = std::sin(th), cp = std::cos(ph), sp = std::sin(ph);
      const double R[9] = {cp * ct, -sp, cp * st, sp * ct, cp, sp * st, -st, 0.0, ct};
      for (int k = 0; k < 9; ++k) fr[9 * n + k] = R[k];
    }
    c->h_coord = X;
    c->h_sph = S;
    c->X.upload(X);
    c->S.upload(S);
    c->frames.upload(fr);
    // classes
    std::vector<uint8_t> cls(f.nel, 255);
    std::vector<int32_t> iso(f.nel, -1);
    for (int k = 0; k < 4; ++k) {
      M3_REQUIRE(m->nels_class[k] == 0 || m->els_class[k], M3_E_ARG, "missing class list");
      for (int64_t i = 0; i < m->nels_class[k]; ++i) {
        const int64_t e = (int64_t)m->els_class[k][i] - 1;
        M3_REQUIRE(e >= 0 && e < f.nel && cls[e] == 255, M3_E_MESH, "element classes must partition the mesh");
        cls[e] = (uint8_t)k;
        if (k == 3) iso[e] = (int32_t)i;
      }
    }
    for (int64_t e = 0; e < f.nel; ++e) M3_REQUIRE(cls[e] != 255, M3_E_MESH, "element without class");
    c->cls.upload(cls);
    c->iso_idx.upload(iso);
    c->n_iso = m->nels_class[3];
    std::vector<double> X20(std::max<int64_t>(1, 60 * c->n_iso), 0.0);
    for (int64_t i = 0; i < c->n_iso; ++i)
      for (int n = 0; n < 20; ++n) {
        const int64_t g = (int64_t)m->EL2NOD_cubic[20 * i + n] - 1;
        M3_REQUIRE(g >= 0 && g < f.nnod + m->ncubic, M3_E_MESH, "EL2NOD_cubic out of range");
        for (int k = 0; k < 3; ++k)
          X20[60 * i + 3 * n + k] = g < f.nnod ? m->GCOORD[3 * g + k] : m->GCOORD_cubic[3 * (g - f.nnod) + k];
      }
    c->X20.upload(X20);
    mark("coordinates, frames, classes");
    // transfers and child interpolation tables
    for (int l = 0; l < nmg - 1; ++l) {
      LevelDev &fl = c->L[l];
      LevelDev &cl = c->L[l + 1];
      M3_REQUIRE(m->Ic2f_ptr[l] && m->Ic2f_col[l] && m->Ic2f_val[l], M3_E_ARG, "missing Ic2f");
      const int64_t *P_ptr = m->Ic2f_ptr[l];
      const int64_t nnzP = P_ptr[fl.nnod];
      const int32_t *P_col = m->Ic2f_col[l];
      const double *P_val = m->Ic2f_val[l];
      for (int64_t k = 0; k < nnzP; ++k)
        M3_REQUIRE(P_col[k] >= 0 && P_col[k] < cl.nnod, M3_E_MESH, "Ic2f column out of range");
      // both directions in the levels' vector orders: row q of P is the node at
      // place q of the fine level
      const std::vector<int32_t> &fperm = fl.K.h_vperm, &cipos = cl.K.h_vpos;
      auto fnode = [&](int64_t q) { return fperm.empty() ? q : (int64_t)fperm[q]; };
      std::vector<int64_t> PP(fl.nnod + 1, 0), R_ptr(cl.nnod + 1, 0);
#pragma omp parallel for schedule(static)
      for (int64_t q = 0; q < fl.nnod; ++q) PP[q + 1] = P_ptr[fnode(q) + 1] - P_ptr[fnode(q)];
      for (int64_t q = 0; q < fl.nnod; ++q) PP[q + 1] += PP[q];
      HostArr<int32_t> PC(nnzP), R_col(nnzP);
      HostArr<double> PV(nnzP), R_val(nnzP);
#pragma omp parallel for schedule(static)
      for (int64_t q = 0; q < fl.nnod; ++q)
        for (int64_t k = P_ptr[fnode(q)], o = PP[q]; k < P_ptr[fnode(q) + 1]; ++k, ++o) {
          PC[o] = cipos.empty() ? P_col[k] : cipos[P_col[k]];
          PV[o] = P_val[k];
        }
      // the transpose: every thread reads all of P and keeps the entries of its
      // own range of coarse rows (fine rows ascending in each)
      const int nt = omp_get_max_threads();
      auto first = [&](int t) { return (int32_t)(cl.nnod * t / nt); };
#pragma omp parallel for schedule(static, 1)
      for (int t = 0; t < nt; ++t) {
        const int32_t j0 = first(t), j1 = first(t + 1);
        for (int64_t k = 0; k < nnzP; ++k)
          if (PC[k] >= j0 && PC[k] < j1) R_ptr[PC[k] + 1]++;
      }
      for (int64_t j = 0; j < cl.nnod; ++j) R_ptr[j + 1] += R_ptr[j];
      std::vector<int64_t> fill(R_ptr.begin(), R_ptr.end() - 1);
#pragma omp parallel for schedule(static, 1)
      for (int t = 0; t < nt; ++t) {
        const int32_t j0 = first(t), j1 = first(t + 1);
        for (int64_t i = 0; i < fl.nnod; ++i)
          for (int64_t k = PP[i]; k < PP[i + 1]; ++k) {
            if (PC[k] < j0 || PC[k] >= j1) continue;
            const int64_t q = fill[PC[k]]++;
            R_col[q] = (int32_t)i;
            R_val[q] = PV[k];
          }
      }
      mark("transfers");
      fl.P_ptr.upload(PP);
      fl.P_col.upload(PC.p.get(), PC.n);
      fl.P_val.upload(PV.p.get(), PV.n);
      fl.R_ptr.upload(R_ptr);
      fl.R_col.upload(R_col.p.get(), R_col.n);
      fl.R_val.upload(R_val.p.get(), R_val.n);
      // Q_e[i][a] = Ic2f(node_e(i), node_parent(a)); every nonzero of the
      // rows of a child must lie on its parent's nodes (nesting invariant).
      // Distinct tables are numbered in order of first appearance: a 64-bit
      // hash per element in parallel, then the tables themselves compared.
      auto table = [&](int64_t e, double *Q) {
        const int64_t pc = e / 8;
        std::fill(Q, Q + 100, 0.0);
        for (int i = 0; i < 10; ++i) {
          const int node = fl.h_el2nod[10 * e + i];
          for (int64_t k = P_ptr[node]; k < P_ptr[node + 1]; ++k) {
            int a = -1;
            for (int q = 0; q < 10; ++q)
              if (cl.h_el2nod[10 * pc + q] == P_col[k]) a = q;
            if (a < 0) return false;
            Q[10 * i + a] = P_val[k];
          }
        }
        return true;
      };
      std::vector<uint64_t> qhash(fl.nel);
      bool outside = false;
#pragma omp parallel for schedule(static) reduction(|| : outside)
      for (int64_t e = 0; e < fl.nel; ++e) {
        double Q[100];
        outside = outside || !table(e, Q);
        uint64_t h = 1469598103934665603ull;  // FNV-1a over the bytes of the table
        const unsigned char *b = reinterpret_cast<const unsigned char *>(Q);
        for (size_t k = 0; k < sizeof(Q); ++k) h = (h ^ b[k]) * 1099511628211ull;
        qhash[e] = h;
      }
      M3_REQUIRE(!outside, M3_E_MESH, "Ic2f row of a fine node references a node outside the parent element");
      std::unordered_map<uint64_t, int32_t> types;
      std::vector<int32_t> ctype(fl.nel);
      std::vector<double> qtab;
      for (int64_t e = 0; e < fl.nel; ++e) {
        auto it = types.find(qhash[e]);
        if (it == types.end()) {
          it = types.emplace(qhash[e], (int32_t)types.size()).first;
          qtab.resize(qtab.size() + 100);
          table(e, &qtab[qtab.size() - 100]);
        }
        ctype[e] = it->second;
      }
      bool clash = false;
#pragma omp parallel for schedule(static) reduction(|| : clash)
      for (int64_t e = 0; e < fl.nel; ++e) {
        double Q[100];
        table(e, Q);
        clash = clash || std::memcmp(Q, &qtab[100 * (size_t)ctype[e]], sizeof(Q)) != 0;
      }
      M3_REQUIRE(!clash, M3_E_MESH, "child interpolation tables with equal hashes differ");
      fl.child_type.upload(ctype);
      fl.Qtab.upload(qtab);
      fl.nqtypes = (int)types.size();
      mark("transfer + child tables");
    }
    // work space
    int64_t maxpart = 2048;
    for (auto &lv : c->L) maxpart = std::max<int64_t>(maxpart, (lv.nnod + 63) / 64 + 16);
    c->partial.alloc(2 * maxpart);
    for (auto &lv : c->L) {
      const size_t n3 = 3 * lv.nnod;
      lv.r0.alloc(n3); lv.r1.alloc(n3); lv.d.alloc(n3); lv.dn.alloc(n3); lv.dd.alloc(n3); lv.rr.alloc(n3);
      lv.dinv.alloc(n3);
      lv.mask.alloc(n3);
    }
    const size_t n3 = 3 * f.nnod;
    for (auto *b : {&c->cg_r, &c->cg_q, &c->cg_Kq, &c->cg_x, &c->cg_b, &c->Uv,
                    &c->Zv, &c->Yv, &c->Rhs, &c->Fb, &c->bc_rhs, &c->U0, &c->fbbc, &c->Usol})
      b->alloc(n3);
    for (auto *b : {&c->pr, &c->prlast, &c->pd, &c->pq, &c->pSq, &c->pP, &c->LiMM, &c->gU0, &c->Psol})
      b->alloc(f.nV);
    c->visc.alloc(f.nnod);
    c->dens.alloc(f.nnod);
    mark("work space");
    c->have_mesh = true;
  });
}

int m3_sweep_windows(m3_ctx *c, int64_t rows, int32_t split, int32_t limit, int32_t per_row) {
  return guard(c, [&] {
    M3_REQUIRE(rows >= 0 && split >= 0 && per_row >= 0 && limit >= 0 && limit <= m3::SWEEP_LIMIT, M3_E_ARG,
               "sweep windows: sizes must not be negative, limit at most 6300");
    m3::SweepRule r;
    if (rows) r.rows = rows;
    if (split) r.split = split;
    if (limit) r.limit = limit;
    if (per_row) r.per_row = per_row;
    c->sweep_rule = r;
  });
}

int m3_set_bc(m3_ctx *c, const int64_t *ifix, const double *vfix, int64_t nfix) {
  return guard(c, [&] {
    M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_set_mesh must be called first");
    M3_REQUIRE(nfix == 0 || (ifix && vfix), M3_E_ARG, "null BC arrays");
    LevelDev &f = c->L[0];
    const int64_t n3 = 3 * f.nnod;
    std::vector<double> mask(n3, 1.0), U0(n3, 0.0);
    for (int64_t i = 0; i < nfix; ++i) {
      const int64_t d = ifix[i] - 1;
      M3_REQUIRE(d >= 0 && d < n3, M3_E_ARG, "UBC.ifix out of range");
      mask[d] = 0.0;
      U0[d] = vfix[i];
    }
    c->h_ifix.assign(ifix, ifix + nfix);
    c->h_vfix.assign(vfix, vfix + nfix);
    for (int l = 0; l < c->nmg; ++l) {
      LevelDev &lv = c->L[l];
      std::vector<double> ml(mask.begin(), mask.begin() + 3 * lv.nnod);
      lv.mask.upload(ml);
      m3::launch_vmask(c->stream, lv);
      lv.nfree = (int64_t)std::count(ml.begin(), ml.end(), 1.0);
    }
    c->U0.upload(U0);
    m3::chol_analyse(c);
    c->have_bc = true;
    c->assembled = c->restricted = c->factored = false;
  });
}

int m3_set_els_ref(m3_ctx *c, const int32_t *els_ref, int64_t nels_ref, const double *Dens0_T_bary) {
  return guard(c, [&] {
    M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_set_mesh must be called first");
    M3_REQUIRE(nels_ref >= 0, M3_E_ARG, "negative number of refined-region elements");
    if (nels_ref == 0 && !c->have_ref) return;  // nothing changes
    c->assembled = c->restricted = c->factored = false;
    if (nels_ref == 0) {  // isempty(MESH.els_ref): buoyancy relative to NUMSCALE.Dens0 everywhere
      c->have_ref = false;
      c->ref_in.release();
      c->ref_d0.release();
      return;
    }
    M3_REQUIRE(els_ref && Dens0_T_bary, M3_E_ARG, "null refined-region arrays");
    const int64_t nel = c->L[0].nel;
    std::vector<uint8_t> in(nel, 0);
    std::vector<double> d0(nel, 0.0);
    int64_t prev = 0;
    for (int64_t j = 0; j < nels_ref; ++j) {
      const int64_t e = els_ref[j];
      M3_REQUIRE(e >= 1 && e <= nel, M3_E_ARG, "MESH.els_ref entry out of range");
      // MESH.els_ref is 1:nel filtered (init_mesh_curved_p.m:320-324); the
      // class kernels pair its entries with the elements of a block in that order
      M3_REQUIRE(e > prev, M3_E_ARG, "MESH.els_ref must be strictly increasing");
      prev = e;
      in[e - 1] = 1;
      d0[e - 1] = Dens0_T_bary[j];
    }
    c->ref_in.upload(in);
    c->ref_d0.upload(d0);
    c->have_ref = true;
  });
}

static void do_assemble(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys) {
  M3_REQUIRE(c->have_bc, M3_E_STATE, "m3_set_bc must be called before assembly");
  M3_REQUIRE(phys && phys->nip == 14, M3_E_ARG, "only OPTS.nip = 14 is supported");
  M3_REQUIRE(phys->type_Dmat == 0 || phys->type_Dmat == 1, M3_E_ARG, "type_Dmat must be 0 or 1");
  c->phys = *phys;
  LevelDev &f = c->L[0];
  hipStream_t s = c->stream;
  M3_REQUIRE((Visc == nullptr) == (Dens == nullptr), M3_E_ARG, "Visc and Dens must both be given or both be NULL");
  if (Visc) {
    HIPCHECK(hipMemcpyAsync(c->visc.p, Visc, sizeof(double) * f.nnod, hipMemcpyHostToDevice, s));
    HIPCHECK(hipMemcpyAsync(c->dens.p, Dens, sizeof(double) * f.nnod, hipMemcpyHostToDevice, s));
  } else {
    M3_REQUIRE(c->have_fields, M3_E_STATE, "Visc = Dens = NULL needs m3_set_fields or m3_rock_prop first");
  }
  if (!c->gather_K) f.K.val.zero(s);  // the row-owner gather writes every stored block
  c->pack16_fresh = false;             // set again by the slot gather of the finest level
  if (!c->g_valid) {  // G and G' depend on the mesh only: assembled once per mesh
    c->G.val.zero(s);
    c->GT.val.zero(s);
  }
  c->M.val.zero(s);
  c->Fb.zero(s);
  c->bc_rhs.zero(s);
  c->errflag.zero(s);
  m3::launch_assemble(c, nullptr, nullptr, nullptr, nullptr, true);
  if (c->gather_K) m3::launch_gather_K(c);
  m3::launch_fix_diag(c, 0);
  m3::launch_lumped_mm(c);
  raise_flags(check_err(c));
  c->g_valid = true;
  c->assembled = true;
  c->restricted = c->factored = c->have_mixed = false;
}

int m3_assemble(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys) {
  return guard(c, [&] { do_assemble(c, Visc, Dens, phys); });
}

// element-packed matrices of the finest level into host arrays (reference
// layout, Cartesian frame, before rotation and BC elimination)
static void element_matrices_host(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys,
                                  double *KKv, double *GGv, double *MMv, double *Fbv) {
    M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_set_mesh must be called first");
    M3_REQUIRE(phys && phys->nip == 14, M3_E_ARG, "only OPTS.nip = 14 is supported");
    c->phys = *phys;
    LevelDev &f = c->L[0];
    hipStream_t s = c->stream;
    HIPCHECK(hipMemcpyAsync(c->visc.p, Visc, sizeof(double) * f.nnod, hipMemcpyHostToDevice, s));
    HIPCHECK(hipMemcpyAsync(c->dens.p, Dens, sizeof(double) * f.nnod, hipMemcpyHostToDevice, s));
    DBuf<double> k, g, mm, fb;
    k.alloc((size_t)465 * f.nel);
    g.alloc((size_t)120 * f.nel);
    mm.alloc((size_t)10 * f.nel);
    fb.alloc((size_t)30 * f.nel);
    if (!c->have_bc) {  // mask / U0 are read even when nothing is scattered
      std::vector<double> one(3 * f.nnod, 1.0);
      f.mask.upload(one);
      c->U0.zero(s);
    }
    c->errflag.zero(s);
    m3::launch_assemble(c, k.p, g.p, mm.p, fb.p, false);
    raise_flags(check_err(c));
    k.download(KKv, k.n);
    g.download(GGv, g.n);
    mm.download(MMv, mm.n);
    fb.download(Fbv, fb.n);
}

int m3_element_matrices(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys,
                        double *KKv, double *GGv, double *MMv, double *Fbv) {
  return guard(c, [&] { element_matrices_host(c, Visc, Dens, phys, KKv, GGv, MMv, Fbv); });
}

int m3_assembly_stokes_sph_3d_double_jacobian(m3_ctx *c, const double *Visc, const double *Dens,
                                              const m3_phys *phys, m3_csc *KK, double *Fb, m3_csc *GG,
                                              m3_csc *MM, double *Fpdil) {
  return guard(c, [&] {
    M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_set_mesh must be called first");
    LevelDev &f = c->L[0];
    if (!c->csc) c->csc = std::make_unique<m3::CscPatterns>(m3::csc_patterns(f.h_el2nod, f.nel, f.nnod, f.nV));
    const m3::CscPatterns &pt = *c->csc;
    bool query = false;
    for (m3_csc *m : {KK, GG, MM})
      if (m && !m->colptr) query = true;
    m3::csc_sizes(pt, KK, GG, MM);
    if (Fpdil) *Fpdil = 0.0;  // no VAR.DilEl on this path (assembly_stokes_sph_3d_double_jacobian.m:485-490)
    if (query) return;
    M3_REQUIRE(Visc && Dens && phys, M3_E_ARG, "null fields");
    std::vector<double> KKv((size_t)465 * f.nel), GGv((size_t)120 * f.nel), MMv((size_t)10 * f.nel),
        Fbv((size_t)30 * f.nel);
    element_matrices_host(c, Visc, Dens, phys, KKv.data(), GGv.data(), MMv.data(), Fbv.data());
    m3::csc_fill(pt, f.h_el2nod, f.nel, KKv.data(), GGv.data(), MMv.data(), Fbv.data(), KK, Fb, GG, MM);
  });
}

static void do_restrict(m3_ctx *c) {
  M3_REQUIRE(c->assembled, M3_E_STATE, "m3_assemble must be called first");
  hipStream_t s = c->stream;
  c->errflag.zero(s);
  for (int l = 0; l < c->nmg - 1; ++l) {
    if (!c->L[l + 1].gather) c->L[l + 1].K.val.zero(s);
    m3::launch_rap(c, l);
    if (c->L[l + 1].gather) m3::launch_gather_K(c, l + 1);
    m3::launch_fix_diag(c, l + 1);
  }
  raise_flags(check_err(c));
  c->restricted = true;
  c->factored = c->have_mixed = false;
}

int m3_restrict_stiffmat(m3_ctx *c) {
  return guard(c, [&] { do_restrict(c); });
}

static void do_factor(m3_ctx *c) {
  M3_REQUIRE(c->restricted, M3_E_STATE, "m3_restrict_stiffmat must be called first");
  c->errflag.zero(c->stream);
  m3::chol_factor(c);
  raise_flags(check_err(c));
}

int m3_cholesky_factorization(m3_ctx *c) {
  return guard(c, [&] { do_factor(c); });
}

int m3_cholesky_solve(m3_ctx *c, const double *rhs, double *x) {
  return guard(c, [&] {
    M3_REQUIRE(c->factored, M3_E_STATE, "m3_cholesky_factorization must be called first");
    LevelDev &cl = c->L[c->nmg - 1];
    const size_t n3 = 3 * cl.nnod;
    HIPCHECK(hipMemcpyAsync(cl.rr.p, rhs, sizeof(double) * n3, hipMemcpyHostToDevice, c->stream));
    m3::scale_mask(c->stream, cl.rr.p, cl.mask.p, cl.rr.p, (int64_t)n3);
    m3::chol_solve_dev(c, cl.rr.p, cl.dn.p);
    HIPCHECK(hipMemcpyAsync(x, cl.dn.p, sizeof(double) * n3, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

int m3_mgpcg(m3_ctx *c, const double *b, double *x, double tol, int32_t is_abs_tol, int32_t itmax,
             int32_t precision, int32_t *it, double *rrms_vec) {
  return guard(c, [&] {
    M3_REQUIRE(c->factored, M3_E_STATE, "operators are not ready (assemble, restrict, factorise)");
    M3_REQUIRE(itmax >= 1, M3_E_ARG, "itmax must be >= 1");
    LevelDev &f = c->L[0];
    const int64_t n3 = 3 * f.nnod;
    if (precision == M3_PREC_MIXED && !c->have_mixed) m3::build_mixed(c);
    HIPCHECK(hipMemcpyAsync(c->Rhs.p, b, sizeof(double) * n3, hipMemcpyHostToDevice, c->stream));
    HIPCHECK(hipMemcpyAsync(c->Zv.p, x, sizeof(double) * n3, hipMemcpyHostToDevice, c->stream));
    m3::scale_mask(c->stream, c->Zv.p, f.mask.p, c->Zv.p, n3);
    std::vector<double> hist;
    const int n = m3::mgpcg_run(c, c->Zv.p, c->Rhs.p, tol, is_abs_tol != 0, itmax, precision, &hist);
    HIPCHECK(hipMemcpyAsync(x, c->Zv.p, sizeof(double) * n3, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    if (it) *it = n;
    if (rrms_vec)
      for (size_t i = 0; i < hist.size() && i < (size_t)itmax + 1; ++i) rrms_vec[i] = hist[i];
  });
}

// ---------------------------------------------------------------- Patera
static void do_patera(m3_ctx *c, double *U, double *P, const m3_patera_opts *o, m3_info *info,
                      const double *U0d = nullptr, const double *P0d = nullptr) {
  M3_REQUIRE(c->factored, M3_E_STATE, "operators are not ready (assemble, restrict, factorise)");
  M3_REQUIRE(o && o->pc_Pat == 3, M3_E_ARG, "only pc_Pat = 3 is supported");
  c->have_solution = false;  // until this solve has written its own
  hipStream_t s = c->stream;
  LevelDev &f = c->L[0];
  const int64_t n3 = 3 * f.nnod, nV = f.nV;
  const int prec = o->precision;
  if (prec == M3_PREC_MIXED && !c->have_mixed) m3::build_mixed(c);
  const double rtol_Pat = o->rtol_Pat, rtol_restart = 0.8 * o->rtol_Pat, wMM = o->wght_MM;
  double rtol_U = o->rtol_U;
  const int itmax_U = o->itmax_U;
  double t_vel = 0, t_pres = 0;
  auto t_start = clk::now();
  double *Uf = c->Uv.p, *Z = c->Zv.p, *Y = c->Yv.p, *Rhs = c->Rhs.p;
  double *r = c->pr.p, *q = c->pq.p, *Pd = c->pP.p;
  DBuf<double> &fbbc = c->fbbc, &gU0 = c->gU0;
  // fbbc = mask (Fb - bc_rhs); gU0 = GG' U0
  m3::copy(s, c->Fb.p, fbbc.p, n3);
  m3::axpy(s, -1.0, c->bc_rhs.p, fbbc.p, n3);
  m3::scale_mask(s, fbbc.p, f.mask.p, fbbc.p, n3);
  m3::spmv_GT(s, c->GT, c->U0.p, gU0.p);
  M3_REQUIRE(P0d || P, M3_E_ARG, "null argument");
  M3_REQUIRE(!o->warm_U || U0d || U, M3_E_ARG, "null argument");
  if (P0d)  // starting point already on the device
    HIPCHECK(hipMemcpyAsync(Pd, P0d, sizeof(double) * nV, hipMemcpyDeviceToDevice, s));
  else
    HIPCHECK(hipMemcpyAsync(Pd, P, sizeof(double) * nV, hipMemcpyHostToDevice, s));
  if (o->warm_U) {
    if (U0d)
      HIPCHECK(hipMemcpyAsync(Uf, U0d, sizeof(double) * n3, hipMemcpyDeviceToDevice, s));
    else
      HIPCHECK(hipMemcpyAsync(Uf, U, sizeof(double) * n3, hipMemcpyHostToDevice, s));
    m3::scale_mask(s, Uf, f.mask.p, Uf, n3);
  } else {
    Uf = c->Uv.p;
    c->Uv.zero(s);
  }
  auto rhs_of_P = [&]() {  // Rhs = mask (Fb + GG P - bc_rhs)
    m3::spmv_G(s, c->G, Pd, Rhs, f.mask.p, fbbc.p);
  };
  auto pres_res = [&](bool rm0) {  // r = -GG' U (U = Uf + U0), mean removed
    m3::spmv_GT(s, c->GT, Uf, r);
    m3::axpy(s, 1.0, gU0.p, r, nV);
    m3::scal(s, -1.0, r, nV);
    if (rm0) m3::add_scalar(s, r, -m3::mean(c, r, nV), nV);
  };
  auto normdf = [&](const double *v, int64_t n, double nf) { return std::sqrt(m3::dot(c, v, v, n) / nf); };
  auto vel_solve = [&](double *x, const double *b, double tol, bool abs, bool x_zero = false) {
    auto t0 = clk::now();
    const int n = m3::mgpcg_run(c, x, b, tol, abs, itmax_U, prec, nullptr, x_zero);
    t_vel += secs(t0, clk::now());
    return n;
  };
  rhs_of_P();
  int nitU = 0;
  if (o->rtol_U_first > 0) {  // fixed-denominator initial velocity tolerance
    const double normf = std::sqrt(m3::dot(c, Rhs, Rhs, n3) / (double)f.nfree);
    nitU = vel_solve(Uf, Rhs, o->rtol_U_first * normf, true, !o->warm_U);
  } else {
    nitU = vel_solve(Uf, Rhs, rtol_U * rtol_restart, false, !o->warm_U);
  }
  pres_res(true);
  double norm_rP = normdf(r, nV, (double)nV);
  const double norm_rP_init = norm_rP;
  const double tol_Pat = o->tol_Pat_abs > 0 ? o->tol_Pat_abs : rtol_Pat * norm_rP;
  // second velocity solve: rtol_U rtol_restart norm_rP in the reference, i.e.
  // rtol_U (rtol_restart / rtol_Pat) tol_Pat (flow3d_patera_mg_sph_p.m:74,437-443);
  // a fixed tol_Pat keeps that relation instead of tying it to norm_rP, which
  // from a good start would solve far below what tol_Pat needs
  const double tol_U2 =
      o->tol_Pat_abs > 0 ? rtol_U * (rtol_restart / rtol_Pat) * tol_Pat : rtol_U * rtol_restart * norm_rP;
  nitU += vel_solve(Uf, Rhs, tol_U2, true);
  const double tol_U_abs = rtol_U * tol_Pat;
  int nitZ = 0, itPat = 0;
  bool restart = true, conv_problem = false;
  double norm_rP0 = norm_rP, tolZ = 0;
  int it0 = 1, ip = 0;
  for (int pass_out = 0;; ++pass_out) {
  for (itPat = it0; itPat <= o->itmax_Pat; ++itPat) {
    auto tp = clk::now();
    // d = r ./ LMM; d += w LiMM (r - MM d)   (precondition_P, pc_Pat = 3); the
    // search direction q, its mean removed
    if (restart) {
      norm_rP0 = norm_rP;
      tolZ = rtol_U * std::max(rtol_restart * norm_rP0, tol_Pat);
    }
    m3::patera_direction(c, nV, wMM, restart, ++ip);
    restart = false;
    m3::spmv_G(s, c->G, q, Y, f.mask.p);
    c->Zv.zero(s);
    t_pres += secs(tp, clk::now());
    nitZ += vel_solve(Z, Y, tolZ, true, true);
    tp = clk::now();
    const double norm_rP_last = norm_rP;
    norm_rP = m3::patera_step(c, nV, n3, Uf, Z, ip) / std::sqrt((double)nV);
    const double norm_rP_min = std::min(norm_rP_last, norm_rP);
    t_pres += secs(tp, clk::now());
    if (norm_rP < tol_Pat && itPat >= o->itmin_Pat) break;
    if (norm_rP < rtol_restart * norm_rP0 || norm_rP > 10 * norm_rP0) {
      rhs_of_P();
      nitU += vel_solve(Uf, Rhs, tol_U_abs, true);
      pres_res(false);
      const double norm_rP_true = normdf(r, nV, (double)nV);
      if (norm_rP_true > 1.1 * norm_rP) rtol_U = rtol_U * 0.75 * (norm_rP / norm_rP_true);
      if (norm_rP > 10 * norm_rP0 || norm_rP > 1.2 * norm_rP_min) {
        if (conv_problem) break;
        rtol_U = 0.1 * rtol_U;
        conv_problem = true;
      }
      restart = true;
    }
  }
  if (itPat > o->itmax_Pat) itPat = o->itmax_Pat;
  rhs_of_P();
  if (o->rtol_U_final > 0) {
    const double normf = std::sqrt(m3::dot(c, Rhs, Rhs, n3) / (double)f.nfree);
    const double tol = std::min(tol_U_abs, o->rtol_U_final * normf);
    auto t0 = clk::now();
    const int itf = std::max(itmax_U, o->itmax_U_final);
    nitU += m3::mgpcg_run(c, Uf, Rhs, tol, true, itf, prec, nullptr);
    // The pressure residual of the final velocity, -GG' U, must also meet
    // tol_Pat.  A velocity error that is small in |K u - f| can still move
    // it (high viscosity contrast): tighten the velocity solve once.  The
    // Patera recurrence residual can also drift from the true one (inexact
    // inner solves): then continue the pressure iteration from the true
    // residual, as the reference's restart does.
    pres_res(true);
    norm_rP = normdf(r, nV, (double)nV);
    if (norm_rP > tol_Pat) {
      nitU += m3::mgpcg_run(c, Uf, Rhs, 0.1 * tol, true, itf, prec, nullptr);
      pres_res(true);
      norm_rP = normdf(r, nV, (double)nV);
    }
    t_vel += secs(t0, clk::now());
    if (norm_rP > tol_Pat && itPat < o->itmax_Pat && pass_out < 3) {
      it0 = itPat + 1;
      restart = true;
      continue;
    }
  } else {
    nitU += vel_solve(Uf, Rhs, tol_U_abs, true);
  }
  break;
  }
  // U = Uf + U0 (rotated frame), P: kept on the device, copied out when the
  // caller passes host buffers
  m3::copy(s, Uf, c->Usol.p, n3);
  m3::axpy(s, 1.0, c->U0.p, c->Usol.p, n3);
  m3::copy(s, Pd, c->Psol.p, nV);
  c->errflag.zero(s);  // NaN test on the device (flow3d_patera_mg_sph_p.m:663)
  m3::nan_flag(s, c->Usol.p, n3, c->errflag.p);
  m3::nan_flag(s, c->Psol.p, nV, c->errflag.p);
  if (U) HIPCHECK(hipMemcpyAsync(U, c->Usol.p, sizeof(double) * n3, hipMemcpyDeviceToHost, s));
  if (P) HIPCHECK(hipMemcpyAsync(P, c->Psol.p, sizeof(double) * nV, hipMemcpyDeviceToHost, s));
  raise_flags(check_err(c));  // synchronises the stream
  c->have_solution = true;
  if (info) {
    info->nitP = itPat;
    info->nitU = nitU;
    info->nitZ = nitZ;
    info->norm_rP = norm_rP;
    info->norm_rP0 = norm_rP_init;
    info->t_pressure = t_pres;
    info->t_velocity = t_vel;
  }
  (void)t_start;
}

int m3_patera(m3_ctx *c, double *U, double *P, const m3_patera_opts *opts, m3_info *info) {
  return guard(c, [&] {
    M3_REQUIRE(U && P, M3_E_ARG, "null argument");
    do_patera(c, U, P, opts, info);
  });
}

int m3_flow3d_patera_sph(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys,
                         double *U, double *P, const m3_patera_opts *opts, m3_info *info) {
  return guard(c, [&] {
    M3_REQUIRE(U && P && opts, M3_E_ARG, "null argument");
    auto t0 = clk::now();
    Timer ta(c->stream);
    do_assemble(c, Visc, Dens, phys);
    const double t_as = ta.stop();
    Timer tr(c->stream);
    do_restrict(c);
    const double t_re = tr.stop();
    Timer tf(c->stream);
    do_factor(c);
    const double t_fa = tf.stop();
    do_patera(c, U, P, opts, info);
    if (info) {
      info->t_assemble = t_as;
      info->t_restrict = t_re;
      info->t_factor = t_fa;
      info->t_total = secs(t0, clk::now());
    }
  });
}

// p must be device memory on the context's GPU
static void require_device_ptr(const m3_ctx *c, const void *p, const char *what) {
  M3_REQUIRE(p, M3_E_ARG, what);
  hipPointerAttribute_t a{};
  const hipError_t e = hipPointerGetAttributes(&a, p);
  if (e != hipSuccess) (void)hipGetLastError();  // not a HIP allocation: clear the error state
  M3_REQUIRE(e == hipSuccess && a.type == hipMemoryTypeDevice && a.device == c->device, M3_E_ARG, what);
}

int m3_flow3d_patera_sph_dstart(m3_ctx *c, const double *Visc, const double *Dens, const m3_phys *phys,
                                const double *U0_dev, const double *P0_dev, double *U, double *P,
                                const m3_patera_opts *opts, m3_info *info) {
  return guard(c, [&] {
    M3_REQUIRE(opts, M3_E_ARG, "null argument");
    M3_REQUIRE((U == nullptr) == (P == nullptr), M3_E_ARG, "U and P must both be given or both be NULL");
    require_device_ptr(c, P0_dev, "P0_dev must be device memory on the context's GPU");
    if (opts->warm_U) require_device_ptr(c, U0_dev, "U0_dev must be device memory on the context's GPU");
    auto t0 = clk::now();
    Timer ta(c->stream);
    do_assemble(c, Visc, Dens, phys);
    const double t_as = ta.stop();
    Timer tr(c->stream);
    do_restrict(c);
    const double t_re = tr.stop();
    Timer tf(c->stream);
    do_factor(c);
    const double t_fa = tf.stop();
    do_patera(c, U, P, opts, info, opts->warm_U ? U0_dev : nullptr, P0_dev);
    if (info) {
      info->t_assemble = t_as;
      info->t_restrict = t_re;
      info->t_factor = t_fa;
      info->t_total = secs(t0, clk::now());
    }
  });
}

int m3_flow3d_patera_sph_learned(m3_ctx *c, m3_gnn *g, double t, int32_t order, const m3_phys *phys, double *U,
                                 double *P, const m3_patera_opts *opts, m3_info *info) {
  return guard(c, [&] {
    M3_REQUIRE(g && opts, M3_E_ARG, "null argument");
    M3_REQUIRE(opts->warm_U, M3_E_ARG, "the learned start sets U and P: opts->warm_U must be 1");
    M3_REQUIRE((U == nullptr) == (P == nullptr), M3_E_ARG, "U and P must both be given or both be NULL");
    M3_REQUIRE(c->have_fields, M3_E_STATE, "the learned solve reads the fields of m3_set_fields or m3_rock_prop");
    if (!c->ev_start) HIPCHECK(hipEventCreateWithFlags(&c->ev_start, hipEventDisableTiming));
    auto t0 = clk::now();
    // the start on the network's stream, overlapping the set-up below
    const double *U0d = nullptr, *P0d = nullptr;
    m3::gnn_start_async(g, t, order, c->device, c->ev_start, &U0d, &P0d);
    Timer ta(c->stream);
    do_assemble(c, nullptr, nullptr, phys);
    const double t_as = ta.stop();
    Timer tr(c->stream);
    do_restrict(c);
    const double t_re = tr.stop();
    Timer tf(c->stream);
    do_factor(c);
    const double t_fa = tf.stop();
    HIPCHECK(hipStreamWaitEvent(c->stream, c->ev_start, 0));
    do_patera(c, U, P, opts, info, U0d, P0d);
    if (info) {
      info->t_assemble = t_as;
      info->t_restrict = t_re;
      info->t_factor = t_fa;
      info->t_total = secs(t0, clk::now());
    }
  });
}

int m3_solution_device(m3_ctx *c, const double **U_dev, const double **P_dev) {
  return guard(c, [&] {
    M3_REQUIRE(U_dev && P_dev, M3_E_ARG, "null argument");
    M3_REQUIRE(c->have_solution, M3_E_STATE, "no Stokes solution on the device yet");
    *U_dev = c->Usol.p;
    *P_dev = c->Psol.p;
  });
}

int m3_get_solution(m3_ctx *c, double *U, double *P) {
  return guard(c, [&] {
    M3_REQUIRE(c->have_solution, M3_E_STATE, "no Stokes solution on the device yet");
    if (U) HIPCHECK(hipMemcpyAsync(U, c->Usol.p, sizeof(double) * c->Usol.n, hipMemcpyDeviceToHost, c->stream));
    if (P) HIPCHECK(hipMemcpyAsync(P, c->Psol.p, sizeof(double) * c->Psol.n, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

int m3_set_fields(m3_ctx *c, const double *Visc, const double *Dens) {
  return guard(c, [&] {
    M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_set_mesh must be called first");
    M3_REQUIRE(Visc && Dens, M3_E_ARG, "null argument");
    const int64_t n = c->L[0].nnod;
    HIPCHECK(hipMemcpyAsync(c->visc.p, Visc, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    HIPCHECK(hipMemcpyAsync(c->dens.p, Dens, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    c->have_fields = true;
  });
}

int m3_apply(m3_ctx *c, int32_t which, int32_t level, const double *x, double *y) {
  return guard(c, [&] {
    M3_REQUIRE(c->assembled, M3_E_STATE, "m3_assemble must be called first");
    M3_REQUIRE(level >= 0 && level < c->nmg, M3_E_ARG, "bad level");
    hipStream_t s = c->stream;
    DBuf<double> dx, dy;
    LevelDev &lv = c->L[level];
    int64_t nx = 0, ny = 0;
    switch (which) {
      case 0: nx = ny = 3 * lv.nnod; break;
      case 1: nx = c->nV; ny = 3 * c->nnod; break;
      case 2: nx = 3 * c->nnod; ny = c->nV; break;
      case 3: nx = ny = c->nV; break;
      case 4: M3_REQUIRE(level < c->nmg - 1, M3_E_ARG, "bad level");
        nx = 3 * c->L[level + 1].nnod; ny = 3 * lv.nnod; break;
      case 5: M3_REQUIRE(level < c->nmg - 1, M3_E_ARG, "bad level");
        nx = 3 * lv.nnod; ny = 3 * c->L[level + 1].nnod; break;
      default: throw M3Error(M3_E_ARG, "bad operator id");
    }
    M3_REQUIRE(which != 0 || level == 0 || c->restricted, M3_E_STATE, "coarse operators not built");
    dx.upload(x, nx);
    dy.alloc(ny);
    switch (which) {
      case 0: m3::spmv_K(s, lv, dx.p, dy.p); break;
      case 1: m3::spmv_G(s, c->G, dx.p, dy.p, nullptr); break;
      case 2: m3::spmv_GT(s, c->GT, dx.p, dy.p); break;
      case 3: m3::spmv_M(s, c->M, dx.p, dy.p); break;
      case 4:  // the transfers act on vector-ordered ones
        m3::to_places(s, c->L[level + 1], dx.p, c->L[level + 1].r0.p);
        m3::prolong(s, lv, c->L[level + 1].r0.p, nullptr, lv.r0.p);
        m3::to_nodes(s, lv, lv.r0.p, dy.p);
        break;
      case 5:
        m3::to_places(s, lv, dx.p, lv.r0.p);
        m3::restrict_(s, lv, c->L[level + 1], lv.r0.p, c->L[level + 1].r0.p);
        m3::to_nodes(s, c->L[level + 1], c->L[level + 1].r0.p, dy.p);
        break;
    }
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(s));
    dy.download(y, ny);
  });
}

int m3_get_vector(m3_ctx *c, int32_t which, int32_t level, double *out) {
  return guard(c, [&] {
    M3_REQUIRE(level >= 0 && level < c->nmg, M3_E_ARG, "bad level");
    HIPCHECK(hipStreamSynchronize(c->stream));
    LevelDev &lv = c->L[level];
    switch (which) {
      case 0: c->Fb.download(out, 3 * c->nnod); break;
      case 1: c->bc_rhs.download(out, 3 * c->nnod); break;
      case 2: {
        M3_REQUIRE(lv.dinv.n == (size_t)(3 * lv.nnod), M3_E_STATE, "m3_set_mesh has not been completed");
        const std::vector<double> di = lv.dinv.to_host();
        for (int64_t q = 0; q < lv.nnod; ++q) {
          const int64_t r = lv.K.h_vperm.empty() ? q : (int64_t)lv.K.h_vperm[q];
          for (int k = 0; k < 3; ++k) out[3 * r + k] = 1.0 / di[3 * q + k];
        }
        break;
      }
      case 3: lv.mask.download(out, 3 * lv.nnod); break;
      case 4: c->LiMM.download(out, c->nV);
        for (int64_t i = 0; i < c->nV; ++i) out[i] = 1.0 / out[i];
        break;
      default: throw M3Error(M3_E_ARG, "bad vector id");
    }
  });
}

int m3_residual(m3_ctx *c, const double *U, const double *P, double *out) {
  return guard(c, [&] {
    M3_REQUIRE(c->assembled, M3_E_STATE, "m3_assemble must be called first");
    hipStream_t s = c->stream;
    LevelDev &f = c->L[0];
    const int64_t n3 = 3 * f.nnod, nV = f.nV;
    DBuf<double> u, uf, p, fU, KU, rP;
    u.upload(U, n3);
    p.upload(P, nV);
    uf.alloc(n3);
    fU.alloc(n3);
    KU.alloc(n3);
    rP.alloc(nV);
    // f_U = mask (Fb + GG P - bc_rhs)
    m3::spmv_G(s, c->G, p.p, fU.p, f.mask.p);
    m3::copy(s, c->Fb.p, KU.p, n3);
    m3::axpy(s, -1.0, c->bc_rhs.p, KU.p, n3);
    m3::scale_mask(s, KU.p, f.mask.p, KU.p, n3);
    m3::axpy(s, 1.0, KU.p, fU.p, n3);
    const double nf = (double)f.nfree;
    const double normf = std::sqrt(m3::dot(c, fU.p, fU.p, n3) / nf);
    // r_U = f_U - K1 (mask U)
    m3::scale_mask(s, u.p, f.mask.p, uf.p, n3);
    m3::spmv_K(s, f, uf.p, KU.p);
    m3::scale_mask(s, KU.p, f.mask.p, KU.p, n3);
    m3::axpy(s, -1.0, KU.p, fU.p, n3);
    const double normr = std::sqrt(m3::dot(c, fU.p, fU.p, n3) / nf);
    // r_P = -GG' U, mean removed
    m3::spmv_GT(s, c->GT, u.p, rP.p);
    m3::add_scalar(s, rP.p, -m3::mean(c, rP.p, nV), nV);
    out[0] = normr;
    out[1] = normf;
    out[2] = std::sqrt(m3::dot(c, rP.p, rP.p, nV) / (double)nV);
  });
}

int m3_profile(m3_ctx *c, int32_t enable) {
  return guard(c, [&] {
    c->prof = enable != 0;
    if (enable) {
      for (int k = 0; k < 3; ++k) {
        for (auto &ev : c->prof_ev[k]) {
          (void)hipEventDestroy(ev.a);
          (void)hipEventDestroy(ev.b);
        }
        c->prof_ev[k].clear();
        c->prof_acc[k] = c->prof_bytes[k] = 0;
        c->prof_n[k] = 0;
      }
    }
  });
}

int m3_profile_read(m3_ctx *c, double *out, int32_t nout) {
  return guard(c, [&] {
    HIPCHECK(hipStreamSynchronize(c->stream));
    for (int k = 0; k < 3; ++k) {
      for (auto &ev : c->prof_ev[k]) {
        float ms = 0;
        HIPCHECK(hipEventElapsedTime(&ms, ev.a, ev.b));
        c->prof_acc[k] += ms * 1e-3;
        c->prof_bytes[k] += ev.bytes;
        c->prof_n[k] += 1;
        (void)hipEventDestroy(ev.a);
        (void)hipEventDestroy(ev.b);
      }
      c->prof_ev[k].clear();
    }
    const double v[9] = {(double)c->prof_n[0], c->prof_acc[0], c->prof_bytes[0],
                         (double)c->prof_n[1], c->prof_acc[1], c->prof_bytes[1],
                         (double)c->prof_n[2], c->prof_acc[2], c->prof_bytes[2]};
    for (int i = 0; i < nout && i < 9; ++i) out[i] = v[i];
  });
}

int m3_rock_prop(m3_ctx *c, const double *T, const m3_rock_params *rp, double *Visc, double *Dens) {
  return guard(c, [&] { m3::rock_prop(c, T, rp, Visc, Dens); });
}

int m3_calculate_dt(m3_ctx *c, const double *U, double dt_adv_limit, double dtmax, double *dt) {
  return guard(c, [&] { *dt = m3::calculate_dt(c, U, dt_adv_limit, dtmax); });
}

int m3_sl_advect(m3_ctx *c, const double *T, const double *U, double dt, double T_cmb, double T_surf,
                 double *T_out) {
  return guard(c, [&] { m3::sl_advect(c, T, U, dt, T_cmb, T_surf, T_out); });
}

int m3_advect3d_slm_p_sph(m3_ctx *c, const double *Ux, const double *Uy, const double *Uz, double *T, double dt,
                          const m3_slm_opts *opts, m3_slm_info *info) {
  return guard(c, [&] { m3::slm_advect(c, Ux, Uy, Uz, T, dt, opts, info); });
}

int m3_diffusion_mesh(m3_ctx *c, const uint32_t *EL2NOD, int64_t nel, int64_t nnodT, double theta_cone) {
  return guard(c, [&] { m3::diffusion_mesh(c, EL2NOD, nel, nnodT, theta_cone); });
}

int m3_diffusion3d(m3_ctx *c, double *T, double kappa, double dt, const int64_t *ifix, const double *vfix,
                   int64_t nfix, const m3_diffusion_opts *opts, m3_diffusion_info *info) {
  return guard(c, [&] { m3::diffusion3d(c, T, kappa, dt, ifix, vfix, nfix, opts, info); });
}

int m3_diffusion_apply(m3_ctx *c, int32_t which, const double *x, double *y) {
  return guard(c, [&] { m3::diffusion_apply(c, which, x, y); });
}

int m3_get_operator(m3_ctx *c, int32_t level, int64_t *rowptr, int32_t *col, double *val) {
  return guard(c, [&] {
    M3_REQUIRE(level >= 0 && level < c->nmg, M3_E_ARG, "bad level");
    M3_REQUIRE(level == 0 ? c->assembled : c->restricted, M3_E_STATE, "operator not built");
    Sell &K = c->L[level].K;
    HIPCHECK(hipStreamSynchronize(c->stream));
    const std::vector<double> v = K.val.to_host();
    int64_t q = 0;
    rowptr[0] = 0;
    for (int64_t r = 0; r < K.nrow; ++r) {
      const int64_t base = K.base_of(r);
      for (int k = 0; k < K.h_rowlen[r]; ++k, ++q) {
        const int64_t slot = base + (int64_t)k * 64;
        col[q] = K.h_col[slot];
        for (int e = 0; e < 9; ++e) val[9 * q + e] = v[(size_t)kval(slot, e)];
      }
      rowptr[r + 1] = q;
    }
  });
}

int m3_stats(m3_ctx *c, int64_t *out, int32_t nout) {
  return guard(c, [&] {
    std::vector<int64_t> v;
    v.push_back(c->nmg);
    for (int l = 0; l < c->nmg; ++l) v.push_back(c->L[l].K.nnz);
    v.push_back(c->chol.n);
    v.push_back(c->chol.T);
    v.push_back(c->chol.ntile);
    v.push_back(c->chol.nlev);
    v.push_back(c->chol.H);
    for (int l = 0; l < c->nmg; ++l) v.push_back(c->L[l].K.nslot);
    for (int l = 0; l < c->nmg; ++l) v.push_back(c->L[l].K.nwin);
    for (int l = 0; l < c->nmg; ++l) v.push_back(c->L[l].K.nwin ? c->L[l].K.umax : 0);
    for (int i = 0; i < nout && i < (int)v.size(); ++i) out[i] = v[i];
  });
}

}  // extern "C"
