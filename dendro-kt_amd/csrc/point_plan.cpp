// Host construction of the point tiles (point_plan.h).
//
// Reference semantics (fem::matvec_rec, FEM/include/matvec.h:380-522), p = 1.
// Write c for a hanging leaf's child index, M for its missing ranks and
// P(s) for the parent's node at rank s.  With ranks counted by their
// difference from c (r' = r xor c), the interpolated value at a missing rank is
// the mean of P over the subsets of r', and the transposed interpolation gives
// 2^-|r'| v(r) to P(s) for every s' in r' with s in M.
//   * A missing rank is a hanging point, the mean of the two points with one
//     bit of r' less on either side: midpoints of edges from nodes, of faces
//     from midpoints of edges, and so on.  Leaves that miss the same position
//     share the point, and its accumulator passes halves back the same way.
//   * That reaches every P(s) behind the point.  What the leaf's own ranks
//     exclude is usually the parent's node c alone (rank c of the child is that
//     node, and is present): the leaf takes sum_r 2^-|r'| v(r) back from it
//     through its correction slot.
//   * Where other ranks behind the point are present too, it is an odd point,
//     with the list of the nodes it reaches.
//   * A rank that interpolates from an absent P(s) reads the stale parent
//     buffer (its leaf is a reader): a point of its own, written by the replay.
#include "point_plan.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <stdexcept>

#include "threads.h"

namespace dkt {

namespace {

constexpr uint16_t kAbsent = 0xFFFF;
constexpr int kMaxTileReaders = 32;  // stale-buffer readers per tile (6 bits of a chain word)

// A tile that does not fit the layout.  smaller: one of fewer leaves may.
struct Misfit : std::runtime_error {
  bool smaller;
  explicit Misfit(const char *what, bool smaller = true) : std::runtime_error(what), smaller(smaller) {}
};

// Tile-local numbering of global ids (first touch): open addressing, cleared
// in time proportional to its use.
struct LocalIds {
  std::vector<int32_t> key, val;
  std::vector<uint32_t> used;
  LocalIds() : key(1 << 14, -1), val(1 << 14, 0) {}
  void clear() {
    for (uint32_t u : used) key[u] = -1;
    used.clear();
  }
  int32_t get(int32_t n, bool *fresh) {
    const uint32_t mask = (uint32_t)key.size() - 1;
    uint32_t h = ((uint32_t)n * 2654435761u >> 7) & mask;
    while (key[h] != -1 && key[h] != n) h = (h + 1) & mask;
    *fresh = key[h] == -1;
    if (*fresh) {
      if (used.size() * 2 >= key.size()) throw Misfit("tile has too many nodes");
      key[h] = n;
      val[h] = (int32_t)used.size();
      used.push_back(h);
    }
    return val[h];
  }
};

enum { kRow = 0, kOdd = 1, kReader = 2 };

// A point of a tile under construction.  Ends of a row and leaf ranks are
// references: a tile-local node n >= 0, or the point -1 - ref.
struct Point {
  int32_t a, b;        // the two points it is the mean of (rows and odd points)
  uint32_t off;        // in the pool: the nodes behind it, then (odd, reader) the nodes it reaches
  uint16_t nrow, ntgt;
  uint8_t kind, cls;   // cls: |r'|
  bool live;           // its accumulator is used: a leaf rank, or behind one (not only the end of an odd point)
};

// The points of one tile, with a hash of (nodes behind, nodes reached).
struct PointSet {
  std::vector<Point> pts;
  std::vector<uint16_t> pool;
  std::vector<int32_t> table;
  std::vector<uint32_t> used;
  PointSet() : table(1 << 14, -1) {}
  void clear() {
    for (uint32_t u : used) table[u] = -1;
    used.clear();
    pts.clear();
    pool.clear();
  }
  // Table slot of the point with these (sorted) nodes; table[slot] < 0: new.
  uint32_t find(const uint16_t *row, int nrow, const uint16_t *tgt, int ntgt) {
    uint64_t h = (uint64_t)nrow * 31 + ntgt + 0x9E3779B97F4A7C15ull;
    for (int i = 0; i < nrow; i++) h = (h ^ row[i]) * 0xBF58476D1CE4E5B9ull;
    for (int i = 0; i < ntgt; i++) h = (h ^ (tgt[i] + 0x10000u)) * 0xBF58476D1CE4E5B9ull;
    const uint32_t mask = (uint32_t)table.size() - 1;
    uint32_t k = (uint32_t)(h >> 33) & mask;
    while (table[k] >= 0) {
      const Point &p = pts[table[k]];
      if (p.nrow == nrow && p.ntgt == ntgt && !std::memcmp(&pool[p.off], row, nrow * sizeof(uint16_t)) &&
          !std::memcmp(&pool[p.off + nrow], tgt, ntgt * sizeof(uint16_t)))
        return k;
      k = (k + 1) & mask;
    }
    if (used.size() * 2 >= table.size()) throw Misfit("tile has too many points");
    used.push_back(k);
    return k;
  }
  int add(int kind, int cls, int32_t a, int32_t b, const uint16_t *row, int nrow, const uint16_t *tgt, int ntgt) {
    pts.push_back(Point{a, b, (uint32_t)pool.size(), (uint16_t)nrow, (uint16_t)ntgt, (uint8_t)kind, (uint8_t)cls,
                        kind != kRow});
    pool.insert(pool.end(), row, row + nrow);
    pool.insert(pool.end(), tgt, tgt + ntgt);
    return (int)pts.size() - 1;
  }
};

// What one tile contributes to the plan's arrays.
struct TileOut {
  PtTile h{};
  std::vector<int32_t> nodes, out;  // global id and output slot per local node
  std::vector<uint8_t> is_target;
  std::vector<uint16_t> gploc;
  std::vector<uint32_t> rows, pairs, step, ckey, chain;
  std::vector<uint64_t> quads, blk, rdr;
  std::vector<double> cw;
  size_t entries = 0;
  double cone_sum = 0, cone_n = 0, span = -1, groups = 0, hang = 0, carry = 0;
};

// Final local indexes of a tile's nodes (by first touch) and points.
struct Renumber {
  std::vector<uint16_t> node, point;
  uint16_t operator()(int32_t ref) const { return ref >= 0 ? node[ref] : point[-1 - ref]; }
};

// Orders a tile's nodes and points and writes its rows and sums.  In: nodes by
// first touch, the points, corr: the node of each correction slot.
void finish_tile(TileOut &to, PointSet &ps, const std::vector<uint16_t> &corr, Renumber &rn) {
  const size_t nn = to.nodes.size(), np = ps.pts.size(), nc = corr.size();
  if (nn + np + nc + 1 > (size_t)kPtMaxPoints) throw Misfit("tile has too many points");
  // Levels: a row's level is one more than its higher end's (ends come first).
  std::vector<uint8_t> lev(np, 0);
  int nlev = 0;
  for (size_t i = 0; i < np; i++) {
    const Point &p = ps.pts[i];
    if (p.kind != kRow) continue;
    const int la = p.a >= 0 ? 0 : lev[-1 - p.a], lb = p.b >= 0 ? 0 : lev[-1 - p.b];
    lev[i] = (uint8_t)(1 + std::max(la, lb));
    nlev = std::max(nlev, (int)lev[i]);
  }
  if (nlev > kPtLevels) throw Misfit("tile has too many row levels", false);  // a leaf's chain, whatever the tile
  for (size_t i = np; i-- > 0;) {  // the ends of a live row are live
    const Point &p = ps.pts[i];
    if (p.kind == kRow && p.live)
      for (int32_t end : {p.a, p.b}) {
        if (end < 0) ps.pts[-1 - end].live = true;
        else to.is_target[end] = 1;
      }
  }
  // Sums onto every node and row: sources as references (-1 - point, or
  // nn + slot for a correction slot).
  std::vector<uint32_t> cnt(nn + np + 1, 0);
  auto at = [&](int32_t ref) { return ref >= 0 ? (size_t)ref : nn + (size_t)(-1 - ref); };
  auto each = [&](auto &&f) {  // f(target, source)
    for (size_t k = 0; k < nc; k++) f((size_t)corr[k], (int32_t)k);
    for (size_t i = 0; i < np; i++) {
      const Point &p = ps.pts[i];
      const int32_t me = -1 - (int32_t)i;
      if (p.kind == kRow) {
        if (!p.live) continue;
        f(at(p.a), me);
        f(at(p.b), me);
      } else {
        for (int t = 0; t < p.ntgt; t++) f((size_t)ps.pool[p.off + p.nrow + t], me);
      }
    }
  };
  each([&](size_t t, int32_t) { cnt[t]++; });
  // Nodes by their number of quads, descending, then by global id: a step of
  // the sums then covers a prefix of the nodes.  Rows by level, then by their
  // number of pairs; odd points; readers in order.
  std::vector<uint32_t> nord(nn), pord(np);
  for (size_t i = 0; i < nn; i++) nord[i] = (uint32_t)i;
  std::sort(nord.begin(), nord.end(), [&](uint32_t a, uint32_t b) {
    const uint32_t qa = (cnt[a] + 3) / 4, qb = (cnt[b] + 3) / 4;
    return qa != qb ? qa > qb : to.nodes[a] < to.nodes[b];
  });
  for (size_t i = 0; i < np; i++) pord[i] = (uint32_t)i;
  std::stable_sort(pord.begin(), pord.end(), [&](uint32_t a, uint32_t b) {
    const Point &p = ps.pts[a], &q = ps.pts[b];
    if (p.kind != q.kind) return p.kind < q.kind;
    if (p.kind != kRow) return false;
    if (lev[a] != lev[b]) return lev[a] < lev[b];
    return (cnt[nn + a] + 1) / 2 > (cnt[nn + b] + 1) / 2;
  });
  rn.node.resize(nn);
  rn.point.resize(np);
  for (size_t i = 0; i < nn; i++) rn.node[nord[i]] = (uint16_t)i;
  for (size_t i = 0; i < np; i++) rn.point[pord[i]] = (uint16_t)(nn + i);
  {
    std::vector<int32_t> n2(nn);
    std::vector<uint8_t> t2(nn);
    for (size_t i = 0; i < nn; i++) {
      n2[i] = to.nodes[nord[i]];
      t2[i] = to.is_target[nord[i]];
    }
    to.nodes.swap(n2);
    to.is_target.swap(t2);
  }
  PtTile &h = to.h;
  h.nnode = (int32_t)nn;
  h.nlev = nlev;
  h.ncor = (int32_t)nc;
  for (int k = 0; k <= kPtLevels; k++) h.lv[k] = (uint32_t)nn;
  for (size_t i = 0; i < np; i++) {
    const Point &p = ps.pts[i];
    if (p.kind == kRow)
      for (int k = lev[i]; k <= kPtLevels; k++) h.lv[k]++;
    else
      (p.kind == kOdd ? h.nodd : h.nrdp)++;
  }
  h.nrow = h.past(nlev);
  // Terms of every target in final order (correction slots, then points by
  // first touch).
  const size_t nt = (size_t)h.past(nlev);  // nodes and rows
  auto fin = [&](size_t t) { return t < nn ? (size_t)rn.node[t] : (size_t)rn.point[t - nn]; };
  std::vector<uint32_t> off(nt + 1, 0);
  for (size_t t = 0; t < nn + np; t++)
    if (cnt[t]) off[fin(t) + 1] = cnt[t];
  for (size_t t = 0; t < nt; t++) off[t + 1] += off[t];
  std::vector<uint16_t> term(off[nt]);
  std::vector<uint32_t> fill(off.begin(), off.end() - 1);
  each([&](size_t t, int32_t src) {
    term[fill[fin(t)]++] = src >= 0 ? (uint16_t)(nn + np + src) : rn.point[-1 - src];
  });
  to.entries = term.size();
  const uint16_t zero = (uint16_t)(nn + np + nc);
  // Groups of steps of the sums onto targets [t0, t1), `per` terms to a word.
  auto sums = [&](size_t t0, size_t t1, size_t per, auto &words) {
    size_t steps = 0;
    for (size_t t = t0; t < t1; t++) steps = std::max<size_t>(steps, (off[t + 1] - off[t] + per - 1) / per);
    for (size_t s = 0; s < steps; s++) {
      const size_t first = words.size();
      size_t t = t0;
      for (; t < t1 && off[t + 1] - off[t] > per * s; t++) {
        typename std::decay<decltype(words)>::type::value_type w = 0;
        for (size_t b = 0; b < per; b++) {
          const size_t k = off[t] + per * s + b;
          w |= (decltype(w))(k < off[t + 1] ? term[k] : zero) << (16 * b);
        }
        words.push_back(w);
      }
      if (first > 0xFFFF) throw Misfit("tile has too many transposed terms");
      to.step.push_back((uint32_t)first | (uint32_t)(t - t0) << 16);
    }
    for (; steps % per; steps++) to.step.push_back(0);  // groups of four quads, two pairs
    return steps / per;
  };
  h.nqs = (int32_t)sums(0, nn, 4, to.quads);
  for (int k = nlev - 1; k >= 1; k--) h.lv[k] |= (uint32_t)sums(h.past(k - 1), h.past(k), 2, to.pairs) << 16;
  for (size_t i = 0; i < np; i++) {
    const Point &p = ps.pts[pord[i]];
    if (p.kind == kReader) to.rows.push_back((uint32_t)(p.cls - 1) << 26);
    else to.rows.push_back((uint32_t)rn(p.a) | (uint32_t)rn(p.b) << 13 | (uint32_t)(p.kind == kOdd ? p.cls - 1 : 0) << 26);
  }
}

// Runs work(t, scratch) for every tile on up to 16 threads, one per kGrain tiles
// at most (a thread costs more than a small mesh's tiles).
constexpr size_t kGrain = 6;
template <typename Scratch, typename F>
void for_tiles(size_t ntiles, F &&work) {
  const int nthreads = (int)std::min<size_t>(host_threads(), (ntiles + kGrain - 1) / kGrain);
  std::atomic<size_t> next{0};
  on_threads(nthreads, [&]() {
    try {
      Scratch sc;
      while (true) {
        const size_t t0 = next.fetch_add(kGrain);
        if (t0 >= ntiles) break;
        for (size_t t = t0; t < std::min(ntiles, t0 + kGrain); t++) work(t, sc);
      }
    } catch (...) {
      next.store(ntiles);
      throw;
    }
  });
}

// Partial slots of the nodes that several tiles write (consecutive per node,
// in tile order) and the tiles' blocks.
void concatenate(PointHost &o, std::vector<TileOut> &outs, size_t N, int T, int npe) {
  const int carry_log = __builtin_ctz((unsigned)(T / npe));
  std::vector<int32_t> ntarget(N, 0);
  for (const TileOut &to : outs)
    for (size_t j = 0; j < to.nodes.size(); j++)
      if (to.is_target[j]) ntarget[to.nodes[j]]++;
  std::vector<int32_t> slot(N, -1);
  o.soff.push_back(0);
  int64_t np = 0;
  for (size_t n = 0; n < N; n++)
    if (ntarget[n] > 1) {
      slot[n] = (int32_t)np;
      np += ntarget[n];
      o.snode.push_back((int32_t)n);
      o.soff.push_back((int32_t)np);
      if (np >= INT32_MAX) throw std::runtime_error("too many partial sums");
    }
  o.npartial = (size_t)np;
  const size_t nt = outs.size();
  o.tiles.resize(nt);
  std::vector<double> st(10, 0.0);
  double n_cone = 0, n_rt = 0;
  size_t units = 0;
  for (size_t t = 0; t < nt; t++) {
    TileOut &to = outs[t];
    PtTile &h = to.h;
    h.nstep = (int32_t)to.step.size();
    h.nquad = (int32_t)to.quads.size();
    h.nrd = (int32_t)to.rdr.size();
    h.rep = (int32_t)to.blk.size() | carry_log << 16;
    h.ncr = (int32_t)to.ckey.size();
    h.ngrp = (int32_t)(to.gploc.size() / npe);
    h.nch = (int32_t)to.chain.size();
    h.na = (h.gploc_at() + 2 * npe * h.ngrp + 15) / 16;
    h.nb = (h.pairs_at() + 4 * (int32_t)to.pairs.size() + 15) / 16;
    h.a0 = (int32_t)units;
    h.b0 = (int32_t)(units + h.na);
    units += (size_t)h.na + h.nb;
    if (units >= INT32_MAX) throw std::runtime_error("mesh too large for 32-bit tile offsets");
    o.tiles[t] = h;
    o.max_nodes = std::max(o.max_nodes, h.nnode);
    o.max_slots = std::max(o.max_slots, h.npts() + h.ncor + 1);
    o.max_units = std::max(o.max_units, std::max(h.na, h.nb));
    o.max_hang = std::max(o.max_hang, (int)to.hang);
    o.max_terms = std::max(o.max_terms, 2 * (h.nrow - h.nnode));
    o.max_grp = std::max(o.max_grp, h.ngrp);
    o.entries += to.entries;
    st[0] += h.nrd;
    st[1] = std::max<double>(st[1], h.nrd);
    st[2] += to.carry;
    st[3] = std::max(st[3], to.carry);
    st[4] += to.groups;
    st[5] += h.nnode;
    st[7] += to.cone_sum;
    n_cone += to.cone_n;
    if (to.span >= 0) {
      n_rt += 1;
      st[8] += to.span;
      st[9] = std::max(st[9], to.span);
    }
    to.out.resize(to.nodes.size());  // a shared node's slots in tile order
    for (size_t j = 0; j < to.nodes.size(); j++) {
      const int32_t g = to.nodes[j];
      to.out[j] = !to.is_target[j] ? INT32_MIN : ntarget[g] == 1 ? g : -(slot[g]++) - 1;
    }
  }
  const double n = std::max<double>(1, (double)nt);
  o.stats = {st[0] / n, st[1], st[2] / n, st[3], st[4] / n, st[5] / n, (double)o.entries,
             n_cone > 0 ? st[7] / n_cone : 0.0, n_rt > 0 ? st[8] / n_rt : 0.0, st[9]};
  o.blocks.resize(units * 4);
  struct None {};
  for_tiles<None>(nt, [&](size_t t, None &) {
    TileOut &to = outs[t];
    const PtTile &h = to.h;
    char *a = reinterpret_cast<char *>(&o.blocks[(size_t)h.a0 * 4]);
    char *b = reinterpret_cast<char *>(&o.blocks[(size_t)h.b0 * 4]);
    std::memset(a, 0, (size_t)(h.na + h.nb) * 16);
    auto put = [](char *to, const auto &v) {
      if (!v.empty()) std::memcpy(to, v.data(), v.size() * sizeof(v[0]));
    };
    put(a, to.nodes);
    put(a + 4 * h.nnode, to.out);
    put(a + h.rows_at(), to.rows);
    put(a + h.readers_at(), to.rdr);
    put(a + h.blocks_at(), to.blk);
    put(a + h.carry_w_at(), to.cw);
    put(a + h.carry_key_at(), to.ckey);
    put(a + h.gploc_at(), to.gploc);
    put(a + h.chain_at(), to.chain);
    put(b, to.step);
    put(b + h.quads_at(), to.quads);
    put(b + h.pairs_at(), to.pairs);
    to = TileOut();  // release as we go
  });
}

// Builds every tile (build_tile fills outs) and, where all fit, the plan's arrays.
template <typename Scratch, typename F>
PtFit finish(PointHost &o, std::vector<TileOut> &outs, size_t N, int T, int npe, F &&build_tile, PointHost &out) {
  try {
    for_tiles<Scratch>(outs.size(), build_tile);
  } catch (const Misfit &m) {
    return m.smaller ? PtFit::smaller : PtFit::none;
  }
  concatenate(o, outs, N, T, npe);
  out = std::move(o);
  return PtFit::yes;
}

}  // namespace

size_t PointHost::bytes() const {
  return tiles.size() * sizeof(PtTile) + snode.size() * 8 + lloc.size() * 2 + (laux.size() + blocks.size()) * 4;
}

PtFit build_points_reference(const MeshParams &mp, const Traversal &tr, size_t N, int &T, int min_leaves, PointHost &out) {
  const int dim = mp.dim, npe = tr.nPe;
  const size_t L = tr.leaves.size();
  StaleBuffer sb(mp, tr);
  auto parent_of = [&](size_t e) {
    Oct par = tr.leaves[e];
    par.lev -= 1;
    const uint32_t pmask = ~(uint32_t)(((uint64_t)1 << (mp.maxd - (int)par.lev)) - 1);
    for (int d = 0; d < dim; d++) par.x[d] &= pmask;
    return par;
  };
  auto same_oct = [&](const Oct &a, const Oct &b) {
    bool same = a.lev == b.lev;
    for (int d = 0; same && d < dim; d++) same = a.x[d] == b.x[d];
    return same;
  };
  // need[c * nPe + r]: the parent ranks that rank r of child c interpolates
  // from (s' in r'), a bit mask.
  std::vector<uint32_t> need((size_t)npe * npe, 0);
  for (int c = 0; c < npe; c++)
    for (int r = 0; r < npe; r++)
      for (int s = 0; s < npe; s++)
        if (((s ^ c) & ~(r ^ c)) == 0) need[(size_t)c * npe + r] |= 1u << s;
  auto masks = [&](size_t e, uint32_t *missing, uint32_t *absent) {
    const int32_t *sl = &tr.slot[e * npe], *ps = &tr.pslot[(size_t)tr.hang_of[e] * npe];
    uint32_t m = 0, a = 0;
    for (int r = 0; r < npe; r++) {
      m |= (uint32_t)(sl[r] < 0) << r;
      a |= (uint32_t)(ps[r] < 0) << r;
    }
    *missing = m;
    *absent = a;
  };
  auto needed = [&](int c, uint32_t missing) {
    uint32_t n = 0;
    for (uint32_t m = missing; m; m &= m - 1) n |= need[(size_t)c * npe + __builtin_ctz(m)];
    return n;
  };
  // What the tile bounds depend on, per leaf.
  enum { kHangs = 1, kReads = 2, kSibling = 4 };  // kSibling: the leaf before hangs, too, and has the same parent
  std::vector<uint8_t> leaf(L);
  constexpr size_t kLeaves = 2048;  // per unit of work
  struct None {};
  for_tiles<None>((L + kLeaves - 1) / kLeaves, [&](size_t u, None &) {
    for (size_t e = u * kLeaves; e < std::min(L, (u + 1) * kLeaves); e++) {
      if (tr.hang_of[e] < 0) continue;
      uint32_t m, a;
      masks(e, &m, &a);
      leaf[e] = kHangs | ((needed(tr.child[e], m) & a) ? kReads : 0);
      if (e > 0 && tr.hang_of[e - 1] >= 0 && same_oct(parent_of(e), parent_of(e - 1))) leaf[e] |= kSibling;
    }
  });
  // Tiles: runs of at most T leaves, kMaxTileReaders readers and T / 4 sibling
  // groups (a group: consecutive hanging leaves of one parent, cut at 64 leaves).
  std::vector<size_t> bounds;
  auto cut_tiles = [&]() {
    bounds.assign(1, 0);
    const int max_groups = std::max(1, T / 4);
    int nrd = 0, ngrp = 0;
    for (size_t e = 0; e < L; e++) {
      const bool hang = leaf[e] & kHangs, reader = leaf[e] & kReads;
      bool new_group = hang && !((leaf[e] & kSibling) && (e - bounds.back()) % 64 != 0);
      if (e - bounds.back() == (size_t)T || (reader && nrd == kMaxTileReaders) || (new_group && ngrp == max_groups)) {
        bounds.push_back(e);
        nrd = 0;
        ngrp = 0;
        new_group = hang;  // of the new tile, also where the last one ended inside the group
      }
      nrd += reader ? 1 : 0;
      ngrp += new_group ? 1 : 0;
    }
    if (bounds.back() != L) bounds.push_back(L);
  };
  cut_tiles();
  if (bounds.size() > 2 && L < (size_t)min_leaves * (bounds.size() - 2)) {
    T /= 2;
    cut_tiles();
  }
  const int n_groups = std::max(1, T / npe);  // replay blocks per tile, a lane group each
  const size_t ntiles = bounds.size() - 1;
  PointHost o;
  o.lloc.resize(L * (size_t)npe);
  o.laux.resize(L);
  struct Scratch {
    LocalIds ids;
    PointSet ps;
    Renumber rn;
    std::vector<uint16_t> corr;
    std::vector<int32_t> ref;    // per leaf rank: first-touch node, or -1 - point
    std::vector<int32_t> slots;  // per leaf: correction slot or -1
    std::vector<int32_t> lat;    // per lattice position of the current group: reference, or INT32_MAX
    std::vector<size_t> hang;    // the tile's hanging leaves
    std::unordered_map<uint64_t, Combo> memo;
  };
  std::vector<TileOut> outs(ntiles);
  int nlat = 1;
  for (int d = 0; d < dim; d++) nlat *= 3;
  // The row point of the parent's lattice at node c with free axes rx (a
  // reference; rx = 0: the node itself): the mean of the points on either side
  // along the last free axis.
  auto row_point = [&](auto &&self, Scratch &sc, const int32_t *ps, int c, uint32_t rx, auto &node) -> int32_t {
    if (!rx) return (int32_t)node(ps[c], false);
    int lat = 0;
    for (int d = dim - 1; d >= 0; d--) lat = lat * 3 + ((rx >> d) & 1 ? 1 : 2 * ((c >> d) & 1));
    if (sc.lat[lat] < INT32_MAX) return sc.lat[lat];
    const uint32_t top = 31 - __builtin_clz(rx), rest = rx ^ (1u << top);
    const int32_t a = self(self, sc, ps, c, rest, node), b = self(self, sc, ps, c ^ (1 << top), rest, node);
    uint16_t row[16];
    int nr = 0;
    for (uint32_t s = need[(size_t)c * npe + (c ^ (int)rx)]; s; s &= s - 1)
      row[nr++] = node(ps[__builtin_ctz(s)], false);
    std::sort(row, row + nr);
    const uint32_t k = sc.ps.find(row, nr, row, 0);
    if (sc.ps.table[k] < 0) sc.ps.table[k] = sc.ps.add(kRow, __builtin_popcount(rx), a, b, row, nr, row, 0);
    return sc.lat[lat] = -1 - sc.ps.table[k];
  };
  auto build_tile = [&](size_t t, Scratch &sc) {
    TileOut &to = outs[t];
    const size_t l0 = bounds[t], l1 = bounds[t + 1];
    to.h.leaf0 = (int32_t)l0;
    to.h.nleaf = (int32_t)(l1 - l0);
    sc.ids.clear();
    sc.ps.clear();
    sc.corr.clear();
    sc.ref.assign((l1 - l0) * npe, 0);
    sc.slots.assign(l1 - l0, -1);
    sc.hang.clear();
    if (sc.memo.size() > (1u << 20)) sc.memo.clear();
    auto node = [&](int32_t n, bool target) -> uint16_t {
      bool fresh;
      const int32_t l = sc.ids.get(n, &fresh);
      if (fresh) {
        to.nodes.push_back(n);
        to.is_target.push_back(0);
      }
      if (target) to.is_target[l] = 1;
      return (uint16_t)l;
    };
    struct Rd {
      int start, own;  // cone start (hanging index, -1: before the tile), own hanging index
      int point;       // first reader point
      uint32_t mask;
    };
    std::vector<Rd> rd;
    bool open = false;  // a sibling group is open
    Oct gpar{};
    for (size_t e = l0; e < l1; e++) {
      const int32_t *sl = &tr.slot[e * npe];
      int32_t *ref = &sc.ref[(e - l0) * npe];
      for (int r = 0; r < npe; r++)
        if (sl[r] >= 0) ref[r] = node(sl[r], true);
      if (tr.hang_of[e] < 0) {
        open = false;
        continue;
      }
      const Oct par = parent_of(e);
      if (!open || !same_oct(par, gpar)) {
        open = true;
        gpar = par;
        to.groups += 1;
        sc.lat.assign(nlat, INT32_MAX);
      }
      const int c = tr.child[e];
      const int32_t *ps = &tr.pslot[(size_t)tr.hang_of[e] * npe];
      uint32_t missing, absent;
      masks(e, &missing, &absent);
      const bool reader = (needed(c, missing) & absent) != 0;
      if (reader) rd.push_back(Rd{-1, (int)sc.hang.size(), (int)sc.ps.pts.size(), 0});
      sc.hang.push_back(e);
      // The leaf takes its own part back from the parent's node c, which its
      // missing ranks' points include (rank c of the leaf is that node).
      const bool corrected = missing && !(missing >> c & 1) && !(absent >> c & 1);
      if (corrected) {
        sc.slots[e - l0] = (int32_t)sc.corr.size();
        sc.corr.push_back(node(ps[c], true));
      }
      if (reader)  // points of their own, in rank order
        for (uint32_t m = missing; m; m &= m - 1) {
          const int r = __builtin_ctz(m);
          const uint32_t nd = need[(size_t)c * npe + r];
          if (!(nd & absent)) continue;
          uint16_t tgt[16];
          int nt = 0;
          for (uint32_t b = nd & ~absent & (missing | (1u << c)); b; b &= b - 1)
            tgt[nt++] = node(ps[__builtin_ctz(b)], true);
          ref[r] = -1 - sc.ps.add(kReader, __builtin_popcount((uint32_t)(r ^ c)), 0, 0, tgt, 0, tgt, nt);
          rd.back().mask |= 1u << r;
        }
      for (uint32_t m = missing & ~(reader ? rd.back().mask : 0u); m; m &= m - 1) {
        const int r = __builtin_ctz(m);
        const uint32_t nd = need[(size_t)c * npe + r];
        const uint32_t tg = nd & (missing | (1u << c));
        if (tg == nd) {
          ref[r] = row_point(row_point, sc, ps, c, (uint32_t)(r ^ c), node);
          sc.ps.pts[-1 - ref[r]].live = true;
          continue;
        }
        uint16_t row[16], tgt[16];
        int nr = 0, nt = 0;
        const uint32_t rx = (uint32_t)(r ^ c), top = 31 - __builtin_clz(rx);
        const int32_t a = row_point(row_point, sc, ps, c, rx ^ (1u << top), node);
        const int32_t b = row_point(row_point, sc, ps, c ^ (1 << top), rx ^ (1u << top), node);
        for (uint32_t q = nd; q; q &= q - 1) row[nr++] = node(ps[__builtin_ctz(q)], false);
        for (uint32_t q = tg; q; q &= q - 1) tgt[nt++] = node(ps[__builtin_ctz(q)], true);
        std::sort(row, row + nr);
        std::sort(tgt, tgt + nt);
        const uint32_t k = sc.ps.find(row, nr, tgt, nt);
        if (sc.ps.table[k] < 0) sc.ps.table[k] = sc.ps.add(kOdd, __builtin_popcount(rx), a, b, row, nr, tgt, nt);
        ref[r] = -1 - sc.ps.table[k];
      }
    }
    to.hang = (double)sc.hang.size();
    // Readers: the cone of a reader starts at the last hanging leaf whose own
    // parent values alone fix the slots the reader needs, or before the tile
    // (carry: the buffer state at the tile start, from host-expanded terms).
    // Replaying from any earlier start is exact as well, so readers are grouped
    // into blocks, one replay per block.
    uint32_t entry = 0;
    for (Rd &q : rd) {
      const size_t e = sc.hang[q.own];
      uint32_t missing, absent;
      masks(e, &missing, &absent);
      uint32_t cur = needed(tr.child[e], missing) & absent;
      int k = q.own - 1;
      while (true) {
        if (k < 0) {
          entry |= cur;
          break;
        }
        masks(sc.hang[k], &missing, &absent);
        uint32_t nxt = needed(tr.child[sc.hang[k]], cur) & absent;
        if (!nxt) {
          q.start = k;
          break;
        }
        cur = nxt;
        k--;
      }
      to.cone_sum += (double)q.own - q.start;
      to.cone_n += 1;
    }
    size_t carry_hdr = 0;
    if (entry) {
      const int before = tr.hang_of[sc.hang[0]] - 1;  // last hanging leaf before the tile
      std::vector<uint32_t> ck;
      std::vector<double> cwl;
      if (before >= 0)
        for (uint32_t m = entry; m; m &= m - 1) {
          const int s = __builtin_ctz(m);
          for (const auto &e2 : sb.after((size_t)before, s, sc.memo)) {
            if (e2.second == 0.0) continue;
            ck.push_back(((uint32_t)s << 16) | node(e2.first, false));
            cwl.push_back(e2.second);
          }
        }
      if (!ck.empty()) {
        std::vector<uint32_t> hdr(npe + 1, 0);
        for (uint32_t k : ck) hdr[(k >> 16) + 1]++;
        for (int s = 0; s < npe; s++) hdr[s + 1] += hdr[s];
        for (int s = 0; s <= npe; s++) {
          to.ckey.push_back(hdr[s] + (uint32_t)npe + 1);
          to.cw.push_back(0.0);
        }
        carry_hdr = to.ckey.size();
        to.carry = (double)ck.size();
        to.ckey.insert(to.ckey.end(), ck.begin(), ck.end());
        to.cw.insert(to.cw.end(), cwl.begin(), cwl.end());
      }
    }
    if (!rd.empty()) {
      // Blocks of consecutive readers with the smallest maximum replay length,
      // at most one block per lane group.
      auto cut = [&](int span, std::vector<std::pair<size_t, size_t>> *out) {
        size_t i = 0, blocks = 0;
        while (i < rd.size()) {
          int mn = rd[i].start;
          size_t j = i + 1;
          while (j < rd.size() && rd[j].own - std::min(mn, rd[j].start) <= span) mn = std::min(mn, rd[j++].start);
          if (out) out->push_back({i, j});
          blocks++;
          i = j;
        }
        return blocks;
      };
      int lo = 0, hi = T + 1;
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if ((int)cut(mid, nullptr) <= n_groups) hi = mid;
        else lo = mid + 1;
      }
      std::vector<std::pair<size_t, size_t>> blocks;
      cut(lo, &blocks);
      int first = (int)sc.hang.size(), last = 0, mspan = 0;
      for (const auto &b : blocks) {
        int mn = rd[b.first].start, mx = 0;
        for (size_t r = b.first; r < b.second; r++) {
          mn = std::min(mn, rd[r].start);
          mx = std::max(mx, rd[r].own);
        }
        mspan = std::max(mspan, mx - mn);
        first = std::min(first, std::max(mn, 0));
        last = std::max(last, mx);
      }
      to.span = mspan;
      // Chain words and parent maps of the hanging leaves the replay passes,
      // numbered from the first of them.
      int g = -1;
      Oct cpar{};
      for (int k = first; k <= last; k++) {
        const size_t e = sc.hang[k];
        const Oct par = parent_of(e);
        if (g < 0 || !same_oct(par, cpar)) {
          g++;
          cpar = par;
          const int32_t *ps = &tr.pslot[(size_t)tr.hang_of[e] * npe];
          for (int s = 0; s < npe; s++) to.gploc.push_back(ps[s] >= 0 ? node(ps[s], false) : kAbsent);
          if (g > 63) throw Misfit("tile has too many sibling groups");
        }
        uint32_t missing, absent;
        masks(e, &missing, &absent);
        to.chain.push_back((uint32_t)tr.child[e] | (uint32_t)g << 10 | absent << 16);
      }
      for (const auto &b : blocks) {
        int mn = rd[b.first].start, mx = 0;
        for (size_t r = b.first; r < b.second; r++) {
          mn = std::min(mn, rd[r].start);
          mx = std::max(mx, rd[r].own);
        }
        const uint64_t S = mn < 0 ? 0xFFFFu : (uint64_t)(mn - first);
        to.blk.push_back(S | ((uint64_t)(mx - first) << 16) | ((uint64_t)b.first << 32) |
                         ((uint64_t)(b.second - b.first) << 48));
      }
      for (size_t r = 0; r < rd.size(); r++) to.chain[rd[r].own - first] |= (uint32_t)(r + 1) << 4;
    }
    finish_tile(to, sc.ps, sc.corr, sc.rn);
    for (size_t e = l0; e < l1; e++) {
      for (int r = 0; r < npe; r++) {
        const int32_t v = sc.ref[(e - l0) * npe + r];
        o.lloc[e * npe + r] = sc.rn(v);
      }
      const int32_t s = sc.slots[e - l0];
      uint32_t aux = (tr.leaves[e].lev & 31u) | ((uint32_t)tr.child[e] << 5);
      if (s >= 0) aux |= 1u << 9 | (uint32_t)(to.h.npts() + s) << 16;
      o.laux[e] = aux;
    }
    for (uint16_t &g : to.gploc)
      if (g != kAbsent) g = sc.rn.node[g];
    for (size_t i = carry_hdr; i < to.ckey.size(); i++)
      to.ckey[i] = (to.ckey[i] & 0xFFFF0000u) | sc.rn.node[to.ckey[i] & 0xFFFFu];
    for (const Rd &q : rd)
      to.rdr.push_back((uint64_t)sc.rn.point[q.point] | (uint64_t)q.mask << 32);
  };
  return finish<Scratch>(o, outs, N, T, npe, build_tile, out);
}

PtFit build_points_conforming(const MeshParams &mp, const Traversal &tr, const std::vector<Oct> &nodes, int T,
                             int max_terms, PointHost &out) {
  const int dim = mp.dim, npe = tr.nPe;
  const size_t E = tr.leaves.size(), N = nodes.size();
  // Node ids by position: open addressing, filled in parallel (positions are
  // distinct; a node claims the first free slot of its probe sequence).
  size_t cap = 16;
  while (cap < 2 * N) cap <<= 1;
  std::vector<int32_t> table(cap, -1);
  auto hash = [&](const u32 *x) {
    u64 h = 0x9E3779B97F4A7C15ull;
    for (int d = 0; d < dim; d++) h = (h ^ x[d]) * 0xBF58476D1CE4E5B9ull;
    return (size_t)(h ^ (h >> 31)) & (cap - 1);
  };
  constexpr size_t kFill = 2048;  // nodes per unit of work
  struct None {};
  for_tiles<None>((N + kFill - 1) / kFill, [&](size_t c, None &) {
    for (size_t n = c * kFill; n < std::min(N, (c + 1) * kFill); n++)
      for (size_t i = hash(nodes[n].x);; i = (i + 1) & (cap - 1)) {
        int32_t free = -1;
        if (__atomic_compare_exchange_n(&table[i], &free, (int32_t)n, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) break;
      }
  });
  auto find_node = [&](const u32 *x) -> int32_t {
    for (size_t i = hash(x);; i = (i + 1) & (cap - 1)) {
      const int32_t n = table[i];
      if (n < 0) return -1;
      bool same = true;
      for (int d = 0; same && d < dim; d++) same = nodes[n].x[d] == x[d];
      if (same) return n;
    }
  };
  const size_t ntiles = (E + T - 1) / T;
  PointHost o;
  o.lloc.resize(E * (size_t)npe);
  o.laux.resize(E);
  // A position and the level it is resolved from, to its reference.
  struct Known {
    struct Key {
      u32 x[4], lev;
    };
    std::vector<Key> key;
    std::vector<int32_t> ref;
    std::vector<uint32_t> used;
    std::vector<uint8_t> full;
    Known() : key(1 << 14), ref(1 << 14), full(1 << 14, 0) {}
    void clear() {
      for (uint32_t u : used) full[u] = 0;
      used.clear();
    }
    // Slot of the key, free or not.
    uint32_t slot(const Key &k) {
      u64 h = 0x9E3779B97F4A7C15ull;
      for (u32 v : {k.x[0], k.x[1], k.x[2], k.x[3], k.lev}) h = (h ^ v) * 0xBF58476D1CE4E5B9ull;
      uint32_t i = (uint32_t)(h >> 33) & ((1 << 14) - 1);
      while (full[i] && std::memcmp(&key[i], &k, sizeof k)) i = (i + 1) & ((1 << 14) - 1);
      return i;
    }
    void put(const Key &k, int32_t r) {
      const uint32_t i = slot(k);
      if (full[i]) return;
      if (used.size() * 2 >= full.size()) throw Misfit("tile has too many points");
      full[i] = 1;
      key[i] = k;
      ref[i] = r;
      used.push_back(i);
    }
  };
  struct Scratch {
    LocalIds ids;
    PointSet ps;
    Renumber rn;
    Known corner, inside;
    std::vector<int32_t> ref;
  };
  std::vector<TileOut> outs(ntiles);
  auto build_tile = [&](size_t t, Scratch &sc) {
    TileOut &to = outs[t];
    const size_t l0 = t * T, l1 = std::min(E, l0 + T);
    to.h.leaf0 = (int32_t)l0;
    to.h.nleaf = (int32_t)(l1 - l0);
    sc.ids.clear();
    sc.ps.clear();
    sc.corner.clear();
    sc.inside.clear();
    sc.ref.assign((l1 - l0) * npe, 0);
    auto node = [&](int32_t n) -> int32_t {
      bool fresh;
      const int32_t l = sc.ids.get(n, &fresh);
      if (fresh) {
        to.nodes.push_back(n);
        to.is_target.push_back(1);
      }
      return l;
    };
    // interpolant: the value at x of the cell (anchor a, level lev); cornered: at
    // a corner of that cell, a node or the interpolant of its parent.
    auto cornered = [&](auto &&self, auto &&inside, const u32 *x, const u32 *a, u32 lev) -> int32_t {
      typename Known::Key k{{x[0], x[1], x[2], x[3]}, lev};
      const uint32_t i = sc.corner.slot(k);
      if (sc.corner.full[i]) return sc.corner.ref[i];
      int32_t r;
      if (const int32_t n = find_node(x); n >= 0) {
        r = node(n);
      } else {
        if (lev == 0) throw std::runtime_error("conforming constraint: a root node is missing");
        const u32 plen = 2u << (mp.maxd - lev);
        u32 pa[4] = {0, 0, 0, 0};
        for (int d = 0; d < dim; d++) pa[d] = a[d] & ~(plen - 1);
        r = inside(self, inside, x, pa, lev - 1);
      }
      sc.corner.put(k, r);
      return r;
    };
    auto inside = [&](auto &&cornered, auto &&self, const u32 *x, const u32 *a, u32 lev) -> int32_t {
      const u32 len = 1u << (mp.maxd - lev);
      int d = dim - 1;  // the last axis on which x is no end of the cell
      while (d >= 0 && (x[d] == a[d] || x[d] == a[d] + len)) d--;
      if (d < 0) return cornered(cornered, self, x, a, lev);
      // Known by position and level: cells of one level that share the position
      // share the face behind it.
      typename Known::Key k{{x[0], x[1], x[2], x[3]}, lev};
      const uint32_t i = sc.inside.slot(k);
      if (sc.inside.full[i]) return sc.inside.ref[i];
      u32 xa[4] = {x[0], x[1], x[2], x[3]}, xb[4] = {x[0], x[1], x[2], x[3]};
      xa[d] = a[d];
      xb[d] = a[d] + len;
      const int32_t ra = self(cornered, self, xa, a, lev), rb = self(cornered, self, xb, a, lev);
      const uint16_t none = 0;
      const int32_t r = -1 - sc.ps.add(kRow, 1, ra, rb, &none, 0, &none, 0);
      sc.inside.put(k, r);
      return r;
    };
    for (size_t e = l0; e < l1; e++) {
      const Oct &c = tr.leaves[e];
      const u32 len = 1u << (mp.maxd - c.lev);
      for (int r = 0; r < npe; r++) {
        const int32_t n = tr.slot[e * npe + r];
        int32_t &ref = sc.ref[(e - l0) * npe + r];
        if (n >= 0) {
          ref = node(n);
          continue;
        }
        u32 x[4] = {0, 0, 0, 0}, pa[4] = {0, 0, 0, 0};
        for (int d = 0; d < dim; d++) {
          x[d] = c.x[d] + ((r >> d) & 1) * len;
          pa[d] = c.x[d] & ~(2 * len - 1);
        }
        ref = inside(cornered, inside, x, pa, c.lev - 1);
        if (ref < 0) sc.ps.pts[-1 - ref].live = true;
      }
      o.laux[e] = (c.lev & 31u) | ((uint32_t)tr.child[e] << 5);
    }
    finish_tile(to, sc.ps, {}, sc.rn);
    if (2 * (to.h.nrow - to.h.nnode) > max_terms) throw Misfit("tile has too many row ends");
    for (size_t i = 0; i < (l1 - l0) * npe; i++) o.lloc[l0 * npe + i] = sc.rn(sc.ref[i]);
  };
  return finish<Scratch>(o, outs, N, T, npe, build_tile, out);
}

}  // namespace dkt
