// bl_tiles.hip -- the element tiling of the tile step (host side).
//
// The tile step fuses the fused step's F2, F3 and F4, for a Lagrangian step
// of pure cells and for the Lagrangian part of an ALE step with unsplit
// advection, mixed cells included (whose remap then runs on the same tiles,
// k_remap_tile in bl_fused.hip): one workgroup owns a tile of elements.  It computes
// the predictor and the corrector corner terms (F2's work, kept in LDS) of
// its own elements and of the ring of elements around their nodes, sums
// them for every node of its own elements in the reference's scatter order
// (F3's work), and then the corrector state of its own elements (F4's
// work), whose nodes it now holds.  Every element is completed by the one
// tile that owns it, so the F2->F3->F4 corner terms never reach HBM and no
// second pass is needed.  A node that belongs to several tiles is computed
// by each of them from the same inputs (the same bits) and written by one:
// the tile owning the node's first incident element.
//
// The reference sums a node's corner terms in (corner jj, element in
// ielsort1 order) order (hydro_kn_getacceleration.f90:53-72).  When no node
// is corner jj of two elements, that order is simply jj = 1..4 over the
// node's incident corners, which a tile reproduces from one LDS slot per
// (node, jj).  A mesh where some node is corner jj of two elements keeps the
// three-kernel step.
//
// Tiles come from recursive coordinate bisection of the element centroids
// when the tiling is built (setup_rcb.f90 cuts the reference's partitions
// the same way; see Rcb below).  The positions only shape the tiles: any
// tiling gives the same results.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <exception>
#include <memory>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "bl_grow.h"
#include "bl_internal.h"
#include "bl_tiles.h"

namespace bl {

namespace {

// The set-up is host work over every element, shared by up to kThreads
// threads: a first run call of 524288 elements with mixed cells and the
// remap took 110 ms with one and 45 to 55 with eight (13 of either are its
// steps).  A share is at least 32768 elements or 256 tiles: at 16384 and 64
// the relaxation on 414x173 was ready after 93 ms, at these after 76, as a
// thread that has to wait for a core costs more than it saves.  The result
// does not depend on their number.
constexpr int kThreads = 8;

// a and b at once, each to its end; what either throws is thrown here
template <typename F, typename G>
void both(F&& a, G&& b) {
  std::exception_ptr ea, eb;
  auto run_b = [&] {
    try { b(); } catch (...) { eb = std::current_exception(); }
  };
  std::thread t;
  try {
    t = std::thread(run_b);
  } catch (const std::system_error&) {  // no thread to be had
  }
  try { a(); } catch (...) { ea = std::current_exception(); }
  if (t.joinable()) t.join();
  else run_b();
  if (ea) std::rethrow_exception(ea);
  if (eb) std::rethrow_exception(eb);
}

// f(p) for every part p in [lo, hi), each on a thread of its own
template <typename F>
void each_part(int lo, int hi, F& f) {
  if (hi - lo < 2) {
    if (lo < hi) f(lo);
    return;
  }
  const int mid = (lo + hi) / 2;
  both([&] { each_part(lo, mid, f); }, [&] { each_part(mid, hi, f); });
}
// the shares of n pieces of work, at least `least` each
int parts_of(int64_t n, int64_t least) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(kThreads, n / least));
}

// zeros, whose pages a thread takes as it touches them
struct Zeros {
  std::unique_ptr<int32_t, void (*)(void*)> p;
  explicit Zeros(size_t n)
      : p(static_cast<int32_t*>(std::calloc(std::max<size_t>(n, 1), sizeof(int32_t))), std::free) {
    if (!p) throw std::bad_alloc();
  }
  int32_t& operator[](size_t k) { return p.get()[k]; }
};

// Recursive coordinate bisection of the elements by their centroids: each
// cut along the longer side of the element set's bounding box, at the share
// that keeps the tile counts of the two sides proportional, down to about
// kTileTarget elements; a leaf whose nodes or the elements around them do
// not fit one workgroup is cut again.
struct Centroid {
  double x, y;
  int32_t e;
};
using Leaves = std::vector<std::pair<int, int>>;
struct Rcb {
  const std::vector<int32_t>& ielnd;  // 4 per element, 1-based
  const std::vector<int32_t>& inc;    // 4 per node: the element whose corner j it is, or -1
  std::vector<Centroid>& el;          // cut in place

  struct Scratch {
    Zeros nstamp, estamp;  // per node and element: the last count that saw it
    int counter = 0;
    Scratch(size_t nnd, size_t nel) : nstamp(nnd), estamp(nel) {}
  };

  // the nodes of el[lo, hi) fit the tile's node slots and the elements
  // around them one workgroup
  bool fits(int lo, int hi, Scratch& s) const {
    ++s.counter;
    int nn = 0, ne = 0;
    for (int k = lo; k < hi; ++k)
      for (int j = 0; j < 4; ++j) {
        const int v = ielnd[4 * (size_t)el[k].e + j] - 1;
        if (s.nstamp[v] == s.counter) continue;
        s.nstamp[v] = s.counter;
        if (++nn > kTileNodes) return false;
        for (int q = 0; q < 4; ++q) {
          const int32_t b = inc[4 * (size_t)v + q];
          if (b < 0 || s.estamp[b] == s.counter) continue;
          s.estamp[b] = s.counter;
          if (++ne > kTileEls) return false;
        }
      }
    return true;
  }

  // cuts [lo, hi) at el[m]; returns m
  int halve(int lo, int hi, int k, int k1) {
    double x0 = el[lo].x, x1 = x0, y0 = el[lo].y, y1 = y0;
    for (int q = lo + 1; q < hi; ++q) {
      x0 = std::min(x0, el[q].x); x1 = std::max(x1, el[q].x);
      y0 = std::min(y0, el[q].y); y1 = std::max(y1, el[q].y);
    }
    int m = lo + (int)((int64_t)(hi - lo) * k1 / k);
    m = std::max(lo + 1, std::min(hi - 1, m));
    auto at = [&](int q) { return el.begin() + q; };
    if (x1 - x0 >= y1 - y0)
      std::nth_element(at(lo), at(m), at(hi), [](const Centroid& a, const Centroid& b) {
        return a.x < b.x || (a.x == b.x && a.e < b.e);
      });
    else
      std::nth_element(at(lo), at(m), at(hi), [](const Centroid& a, const Centroid& b) {
        return a.y < b.y || (a.y == b.y && a.e < b.e);
      });
    return m;
  }

  void cut(int lo, int hi, int k, Leaves& out, Scratch& s) {
    if (k <= 1) {
      if (hi - lo < 2 || fits(lo, hi, s)) {
        out.emplace_back(lo, hi);
        return;
      }
      k = 2;
    }
    const int k1 = k / 2, m = halve(lo, hi, k, k1);
    cut(lo, m, k1, out, s);
    cut(m, hi, k - k1, out, s);
  }

  // the same by `threads` threads
  void cut_by(int threads, int lo, int hi, int k, Leaves& out) {
    if (threads < 2 || k < 256) {
      Scratch s(inc.size() / 4, el.size());
      cut(lo, hi, k, out, s);
      return;
    }
    const int k1 = k / 2, m = halve(lo, hi, k, k1);
    Leaves right;
    both([&] { cut_by(threads / 2, lo, m, k1, out); },
         [&] { cut_by(threads - threads / 2, m, hi, k - k1, right); });
    out.insert(out.end(), right.begin(), right.end());
  }
};

template <typename T>
int upload_vec(T** d, const std::vector<T>& v) {
  if (*d) { hipFree(*d); *d = nullptr; }
  BL_HIP(hipMalloc(d, sizeof(T) * std::max<size_t>(v.size(), 1)));
  if (!v.empty()) BL_HIP(hipMemcpy(*d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
  return BL_SUCCESS;
}

// four partials for each of n workgroups
template <typename T>
T* slots_of(int64_t n) {
  T* p = nullptr;
  if (hipMalloc(&p, sizeof(T) * 4 * (size_t)n) == hipSuccess) return p;
  (void)hipGetLastError();
  return nullptr;
}

}  // namespace

void free_tiles(Handle* h) {
  void* bufs[] = {h->d_tile_eptr, h->d_tile_nptr, h->d_tile_bounds, h->d_tile_nodes,
                  h->d_tile_ncm,  h->d_tile_el,   h->d_tile_nd,     h->d_rest8,
                  h->d_ens_toff,  h->d_tile_nbr,  h->d_tile_nbfc,   h->d_tile_ninc};
  for (void* p : bufs)
    if (p) hipFree(p);
  h->d_tile_eptr = h->d_tile_nptr = h->d_tile_nodes = nullptr;
  h->d_tile_ncm = nullptr;
  h->d_tile_bounds = nullptr;
  h->d_tile_el = nullptr;
  h->d_tile_nd = nullptr;
  h->d_ens_toff = nullptr;
  h->d_tile_nbr = nullptr;
  h->d_tile_nbfc = nullptr;
  h->d_tile_ninc = nullptr;
  h->ale_tables = false;
  h->d_rest8 = nullptr;
  h->ntile = h->nentries = 0;
  h->tile_state = 0;
}

namespace {

// one thread's tiles
struct TilePart {
  std::vector<int32_t> nodes;
  std::vector<uint8_t> ncm;
  std::vector<int2> ents;
  std::vector<int4> ent_nd;
  bool fits = true;
};

// a table on the device from the parts' own, one after another
template <typename T>
int upload_parts(T** d, const std::vector<TilePart>& parts, std::vector<T> TilePart::*v) {
  size_t n = 0;
  for (const TilePart& p : parts) n += (p.*v).size();
  if (*d) { hipFree(*d); *d = nullptr; }
  BL_HIP(hipMalloc(d, sizeof(T) * std::max<size_t>(n, 1)));
  size_t at = 0;
  for (const TilePart& p : parts) {
    const std::vector<T>& q = p.*v;
    if (!q.empty())
      BL_HIP(hipMemcpy(*d + at, q.data(), sizeof(T) * q.size(), hipMemcpyHostToDevice));
    at += q.size();
  }
  return BL_SUCCESS;
}

int cut_tiles(Handle* h) {
  free_tiles(h);
  const int nel = h->sz.nel, nnd = h->sz.nnd;
  std::vector<int32_t> ielnd(4 * (size_t)nel);
  std::vector<double> x(nnd), y(nnd);
  bl_handle_t* hh = static_cast<bl_handle_t*>(h);
  if (bl_download(hh, BL_IELND, ielnd.data(), 4 * (int64_t)nel) ||
      bl_download(hh, BL_NDX, x.data(), nnd) || bl_download(hh, BL_NDY, y.data(), nnd))
    return BL_FAILURE;
  // every node is corner jj of at most one element, for each jj, and of one
  // element at least (a node no element uses would be written by no tile);
  // an element with a repeated node is there once per corner
  std::vector<int32_t> inc(4 * (size_t)nnd, -1);
  for (int e = 0; e < nel; ++e)
    for (int j = 0; j < 4; ++j) {
      const int v = ielnd[4 * (size_t)e + j] - 1;
      if (v < 0 || v >= nnd || inc[4 * (size_t)v + j] >= 0) {
        h->tile_state = -1;  // not a tiling this step can use
        return BL_SUCCESS;
      }
      inc[4 * (size_t)v + j] = e;
    }
  // the node's first incident element
  auto first_of = [&](int v) {
    int e = nel;
    for (int j = 0; j < 4; ++j)
      if (inc[4 * (size_t)v + j] >= 0) e = std::min(e, inc[4 * (size_t)v + j]);
    return e;
  };
  for (int v = 0; v < nnd; ++v)
    if (first_of(v) == nel) {
      h->tile_state = -1;
      return BL_SUCCESS;
    }
  if (nel >= (1 << 30) || nnd >= (1 << 31) - 1) { h->tile_state = -1; return BL_SUCCESS; }
  std::vector<Centroid> el(nel);
  const int npart = parts_of(nel, 32768);
  auto share = [](int64_t n, int p, int np) { return (int)(n * p / np); };
  auto centroids = [&](int p) {
    for (int e = share(nel, p, npart), e1 = share(nel, p + 1, npart); e < e1; ++e) {
      const int32_t* q = &ielnd[4 * (size_t)e];
      el[e] = Centroid{0.25 * (x[q[0] - 1] + x[q[1] - 1] + x[q[2] - 1] + x[q[3] - 1]),
                       0.25 * (y[q[0] - 1] + y[q[1] - 1] + y[q[2] - 1] + y[q[3] - 1]), e};
    }
  };
  each_part(0, npart, centroids);
  Rcb r{ielnd, inc, el};
  Leaves leaves;
  // an ensemble's instances own contiguous element ranges: each is cut on
  // its own, so that a tile lies in one instance (one dt)
  std::vector<int32_t> toff;
  auto tiles_for = [](int n) { return std::max(1, (n + kTileTarget - 1) / kTileTarget); };
  if (h->ens_n > 0) {
    const int ninst = h->ens_n, np = parts_of(std::min<int64_t>(nel / 32768, ninst), 1);
    std::vector<Leaves> out(ninst);
    auto cut_some = [&](int p) {
      Rcb::Scratch s(nnd, nel);
      for (int k = share(ninst, p, np); k < share(ninst, p + 1, np); ++k) {
        const int lo = h->ens_eoff[k], hi = h->ens_eoff[k + 1];
        r.cut(lo, hi, tiles_for(hi - lo), out[k], s);
      }
    };
    each_part(0, np, cut_some);
    toff.push_back(0);
    for (const Leaves& o : out) {
      leaves.insert(leaves.end(), o.begin(), o.end());
      toff.push_back((int)leaves.size());
    }
  } else {
    r.cut_by(kThreads, 0, nel, tiles_for(nel), leaves);
  }

  const int ntile = (int)leaves.size();
  std::vector<int32_t> tile_of(nel);
  for (int t = 0; t < ntile; ++t)
    for (int k = leaves[t].first; k < leaves[t].second; ++k) tile_of[el[k].e] = t;
  // per tile: its nodes (ascending; the high bit marks the tile that writes
  // the node, the one holding the node's first incident element), then the
  // entries: its own elements ascending, then the ring around them
  const int nasm = parts_of(ntile, 256);
  std::vector<TilePart> parts(nasm);
  std::vector<int32_t> nptr(ntile + 1, 0), eptr(ntile + 1, 0);  // of the part, then of the whole
  auto assemble = [&](int p) {
    TilePart& o = parts[p];
    Zeros nstamp(nnd), slot_of(nnd), estamp(nel);
    std::vector<int32_t> tn, own, ring;
    const int t0 = share(ntile, p, nasm), t1 = share(ntile, p + 1, nasm);
    if (t0 < t1) {
      const size_t n = (size_t)(leaves[t1 - 1].second - leaves[t0].first);
      o.nodes.reserve(n + n / 3);
      o.ncm.reserve(n + n / 3);
      o.ents.reserve(n + n / 2);
      o.ent_nd.reserve(n + n / 2);
    }
    for (int t = t0; t < t1; ++t) {
      const int stamp = t - t0 + 1;
      own.clear();
      for (int k = leaves[t].first; k < leaves[t].second; ++k) own.push_back(el[k].e);
      std::sort(own.begin(), own.end());
      tn.clear();
      for (int e : own) {
        estamp[e] = stamp;
        for (int j = 0; j < 4; ++j) {
          const int v = ielnd[4 * (size_t)e + j] - 1;
          if (nstamp[v] != stamp) { nstamp[v] = stamp; tn.push_back(v); }
        }
      }
      std::sort(tn.begin(), tn.end());
      ring.clear();
      for (int v : tn)
        for (int j = 0; j < 4; ++j) {
          const int32_t e = inc[4 * (size_t)v + j];
          if (e >= 0 && estamp[e] != stamp) { estamp[e] = stamp; ring.push_back(e); }
        }
      std::sort(ring.begin(), ring.end());
      if ((int)tn.size() > kTileNodes || own.size() + ring.size() > (size_t)kTileEls) {
        o.fits = false;
        return;
      }
      nptr[t] = (int)o.nodes.size();
      for (size_t k = 0; k < tn.size(); ++k) {
        const int v = tn[k];
        slot_of[v] = (int)k;
        const bool writes = tile_of[first_of(v)] == t;
        o.nodes.push_back((int32_t)((uint32_t)v | (writes ? 0x80000000u : 0u)));
        // the corners jj the node is (every element around it is an entry
        // of this tile, own or ring)
        uint8_t cm = 0;
        for (int j = 0; j < 4; ++j) cm |= inc[4 * (size_t)v + j] >= 0 ? (uint8_t)(1u << j) : 0u;
        o.ncm.push_back(cm);
      }
      eptr[t] = (int)o.ents.size();
      for (int pass = 0; pass < 2; ++pass)
        for (int e : pass == 0 ? own : ring) {
          uint32_t slots = 0;
          for (int j = 0; j < 4; ++j) {
            const int v = ielnd[4 * (size_t)e + j] - 1;
            slots |= (uint32_t)(nstamp[v] == stamp ? (uint32_t)slot_of[v] : kNoSlot) << (8 * j);
          }
          // an own element: this tile completes and writes it
          const uint32_t flags = pass == 0 ? kTileOwn : 0u;
          o.ents.push_back(make_int2((int)((uint32_t)e | (flags << 30)), (int)slots));
          const int32_t* q = &ielnd[4 * (size_t)e];
          o.ent_nd.push_back(make_int4(q[0] - 1, q[1] - 1, q[2] - 1, q[3] - 1));
        }
    }
  };
  each_part(0, nasm, assemble);
  int nn = 0, ne = 0;
  for (int p = 0; p < nasm; ++p) {
    if (!parts[p].fits) {
      h->tile_state = -1;
      return BL_SUCCESS;
    }
    for (int t = share(ntile, p, nasm); t < share(ntile, p + 1, nasm); ++t) {
      nptr[t] += nn;
      eptr[t] += ne;
    }
    nn += (int)parts[p].nodes.size();
    ne += (int)parts[p].ents.size();
  }
  nptr[ntile] = nn;
  eptr[ntile] = ne;
  std::vector<int4> bounds(ntile);
  for (int t = 0; t < ntile; ++t) bounds[t] = make_int4(eptr[t], eptr[t + 1], nptr[t], nptr[t + 1]);
  if (upload_vec(&h->d_tile_eptr, eptr) || upload_vec(&h->d_tile_nptr, nptr) ||
      upload_vec(&h->d_tile_bounds, bounds) ||
      upload_parts(&h->d_tile_nodes, parts, &TilePart::nodes) ||
      upload_parts(&h->d_tile_ncm, parts, &TilePart::ncm) ||
      upload_parts(&h->d_tile_el, parts, &TilePart::ents) ||
      upload_parts(&h->d_tile_nd, parts, &TilePart::ent_nd) ||
      (!toff.empty() && upload_vec(&h->d_ens_toff, toff)))
    return BL_FAILURE;
  BL_HIP(hipMalloc(&h->d_rest8, 2 * (size_t)std::max(nel, 1)));
  BL_HIP(hipMemset(h->d_rest8, 0, 2 * (size_t)std::max(nel, 1)));
  h->ntile = ntile;
  h->nentries = ne;
  // the partial slots of the tile step: one per tile
  const int64_t need = ntile + 16;
  int64_t have = h->npart, have_i = h->npart;
  if (!grow(&h->d_part, &have, need, slots_of<double>, hipFree) ||
      !grow(&h->d_parti, &have_i, need, slots_of<int32_t>, hipFree)) {
    set_error("tiles: out of device memory");
    return BL_FAILURE;
  }
  h->npart = std::max(h->npart, need);
  // the second element set
  if (!h->elset[0][0]) {
    const int ids[4] = {BL_ELDENSITY, BL_ELENERGY, BL_ELPRESSURE, BL_ELCS2};
    for (int k = 0; k < 4; ++k) {
      h->elset[h->cur_set][k] = h->R(ids[k]);
      BL_HIP(hipMalloc(&h->elset[1 - h->cur_set][k],
                       sizeof(double) * std::max<int64_t>(h->count[ids[k]], 1)));
    }
    h->el_cur = h->cur_set;
  }
  h->tile_state = 1;
  return BL_SUCCESS;
}

int build_ale_tables(Handle* h) {
  if (h->d_tile_nbr) hipFree(h->d_tile_nbr);
  if (h->d_tile_nbfc) hipFree(h->d_tile_nbfc);
  if (h->d_tile_ninc) hipFree(h->d_tile_ninc);
  h->d_tile_nbr = nullptr;
  h->d_tile_nbfc = nullptr;
  h->d_tile_ninc = nullptr;
  const int nel = h->sz.nel, ntile = h->ntile;
  bl_handle_t* hh = static_cast<bl_handle_t*>(h);
  std::vector<int32_t> el(4 * (size_t)nel), fc(4 * (size_t)nel), sort2(nel), pos2(nel);
  std::vector<int32_t> eptr(ntile + 1), nptr(ntile + 1);
  if (bl_download(hh, BL_IELEL, el.data(), 4 * (int64_t)nel) ||
      bl_download(hh, BL_IELFC, fc.data(), 4 * (int64_t)nel) ||
      bl_download(hh, BL_IELSORT2, sort2.data(), nel))
    return BL_FAILURE;
  BL_HIP(hipMemcpy(eptr.data(), h->d_tile_eptr, sizeof(int32_t) * (ntile + 1),
                   hipMemcpyDeviceToHost));
  BL_HIP(hipMemcpy(nptr.data(), h->d_tile_nptr, sizeof(int32_t) * (ntile + 1),
                   hipMemcpyDeviceToHost));
  std::vector<int2> ents(eptr[ntile]);
  BL_HIP(hipMemcpy(ents.data(), h->d_tile_el, sizeof(int2) * ents.size(),
                   hipMemcpyDeviceToHost));
  // the place of each element in the ALE sums (unset ielsort2: identity)
  for (int k = 0; k < nel; ++k) pos2[k] = k;
  for (int k = 0; k < nel; ++k) {
    const int e = (sort2[k] < 1 || sort2[k] > nel) ? k : sort2[k] - 1;
    pos2[e] = k;
  }
  std::vector<int32_t> nbr(ents.size(), 0);
  std::vector<int2> ninc(nptr[ntile], make_int2(0, 0));
  std::vector<int4> nbfc(ents.size());
  auto packed = [&](int e, int i) {
    return ((el[4 * (size_t)e + i] - 1) << 2) | ((fc[4 * (size_t)e + i] - 1) & 3);
  };
  struct Inc { int32_t e, j; };
  const int npart = parts_of(ntile, 256);
  std::atomic<bool> runs{true};
  auto some = [&](int p) {
    Zeros local(nel), stamp(nel);
    std::vector<Inc> inc(4 * (kTileNodes + 1));
    std::vector<int> cnt(kTileNodes + 1);
    const int t0 = (int)((int64_t)ntile * p / npart), t1 = (int)((int64_t)ntile * (p + 1) / npart);
    for (int t = t0; t < t1; ++t) {
      const int eb = eptr[t], ne = eptr[t + 1] - eb, nb = nptr[t], nn = nptr[t + 1] - nb;
      std::fill(cnt.begin(), cnt.begin() + nn, 0);
      for (int k = 0; k < ne; ++k) {
        const int e = ents[eb + k].x & 0x3fffffff;
        local[e] = k;
        stamp[e] = t + 1;
        nbfc[eb + k] = make_int4(packed(e, 0), packed(e, 1), packed(e, 2), packed(e, 3));
        for (int j = 0; j < 4; ++j) {
          const uint32_t sl = ((uint32_t)ents[eb + k].y >> (8 * j)) & 0xFFu;
          if (sl == kNoSlot) continue;
          // (at most four: no node is corner jj of two elements)
          int2& q = ninc[nb + sl];
          q.x = (int)((uint32_t)q.x | ((uint32_t)k << (8 * j)));
          inc[4 * sl + cnt[sl]++] = Inc{e, j};
        }
      }
      for (int k = 0; k < ne; ++k) {
        const uint32_t w = (uint32_t)ents[eb + k].x;
        if (!((w >> 30) & kTileOwn)) continue;
        const int e = (int)(w & 0x3fffffffu);
        uint32_t bytes = 0;
        for (int i = 0; i < 4; ++i) {
          const int b = el[4 * (size_t)e + i] - 1, g = fc[4 * (size_t)e + i] - 1;
          if (b < 0 || b >= nel || g < 0 || g > 3 || stamp[b] != t + 1 ||
              (b == e && g != ((i + 2) & 3))) {
            runs = false;  // not a mesh the tiled remap runs on
            return;
          }
          bytes |= (uint32_t)local[b] << (8 * i);
        }
        nbr[eb + k] = (int32_t)bytes;
      }
      for (int v = 0; v < nn; ++v) {
        Inc* q = &inc[4 * (size_t)v];
        const int n = cnt[v];
        uint32_t code = (uint32_t)n << 16;
        std::sort(q, q + n, [&](const Inc& a, const Inc& b) {
          return a.e != b.e ? pos2[a.e] < pos2[b.e] : a.j < b.j;
        });
        for (int k = 0; k < n; ++k) code |= (uint32_t)q[k].j << (2 * k);
        std::sort(q, q + n, [](const Inc& a, const Inc& b) {
          return a.e != b.e ? a.e < b.e : a.j < b.j;
        });
        for (int k = 0; k < n; ++k) code |= (uint32_t)q[k].j << (8 + 2 * k);
        ninc[nb + v].y = (int)code;
      }
    }
  };
  each_part(0, npart, some);
  if (runs && (upload_vec(&h->d_tile_ninc, ninc) || upload_vec(&h->d_tile_nbfc, nbfc) ||
               upload_vec(&h->d_tile_nbr, nbr)))
    return BL_FAILURE;
  h->ale_tables = true;
  return BL_SUCCESS;
}

// no exception passes the C entries
template <typename F>
int no_throw(F f, Handle* h) {
  try {
    return f(h);
  } catch (const std::exception& e) {
    set_error(std::string("tiles: ") + e.what());
    return BL_FAILURE;
  }
}

}  // namespace

int build_tiles(Handle* h) { return no_throw(cut_tiles, h); }

int build_ale_tiles(Handle* h) { return no_throw(build_ale_tables, h); }

}  // namespace bl
