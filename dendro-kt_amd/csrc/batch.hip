// Batched matvec over many independent meshes (no counterpart in the
// reference, which runs one fem::matvec per call, FEM/include/matvec.h:231).
//
// Plans of the same (dim, p) run as one launch: workgroup b finds its record
// by a binary search over the records' tile offsets and runs that tile with
// the record's maps and vectors (a device table with one record per plan and
// chunk of right-hand sides, each with partial slots of its own; a chunk's
// columns are workgroups of their own), and one fix-up launch sums the shared
// nodes of all groups.  With DKT_BATCH_GRAPH the launches are captured once into a
// hipGraph and replayed.  Each plan's result is bitwise the same as its own
// dkt_plan_matvec: the tile work and the fix-up order are the plan's, whatever
// the work-items of the launch.
#include <algorithm>
#include <map>
#include <memory>
#include <tuple>
#include <vector>

#include "../../include/dkt.h"
#include "capi_common.h"
#include "plan_common.h"
#include "plan_impl.h"
#include "tile_kernel.h"
#include "conf_kernel.h"

using namespace dkt;

namespace {

struct GroupBase {
  virtual ~GroupBase() = default;
  virtual void launch(hipStream_t st) = 0;
  double ranks = 0;  // leaf ranks of the group's items: its work, to order launches by
};

// launch(first, count) over the items of a group, in as many launches as their
// work-items need.
template <typename F>
void launch_items(int nitems, int threads, const F &launch) {
  const int most = (int)std::min<size_t>(INT32_MAX, max_groups_of(std::max(1, threads)));
  for (int first = 0; first < nitems;) {
    const int count = std::min(most, nitems - first);
    launch(first, count);
    HIP_OK(hipGetLastError());
    first += count;
  }
}

// First items of a group's records: adds a record's items to their sum, which
// must stay a 32-bit index.
inline void push_items(std::vector<int> &start, size_t items) {
  if (start.back() + items > (size_t)INT32_MAX) throw std::invalid_argument("too many tiles and columns in a batch");
  start.push_back(start.back() + (int)items);
}

// Device copies of a group's tables: in the caller's arena when there is one,
// else in buffers the group owns.
struct GroupMem {
  DevArena *arena = nullptr;
  std::vector<std::unique_ptr<DevBuf<unsigned char>>> own;
  template <typename T>
  T *upload(const std::vector<T> &v) {
    if (arena) return arena->upload(v);
    own.emplace_back(new DevBuf<unsigned char>());
    own.back()->alloc(std::max<size_t>(1, v.size() * sizeof(T)));
    if (!v.empty()) HIP_OK(hipMemcpy(own.back()->p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return (T *)own.back()->p;
  }
  template <typename T>
  T *alloc(size_t count) {
    if (arena) return (T *)arena->take(count * sizeof(T));
    own.emplace_back(new DevBuf<unsigned char>());
    own.back()->alloc(std::max<size_t>(1, count * sizeof(T)));
    return (T *)own.back()->p;
  }
};

// Shared nodes of one plan of a batch (the fix-up of either kind of tile).
template <typename T>
struct FixRec {
  const int32_t *snode, *soff;
  const T *partial;
  T *y;
  const uint8_t *dir_out;
  const int *cancel;
  int nq, ld, nshared;
};

// Shared nodes of a batch: workgroup b sums block b - block_start[k] of plan k.
template <typename T>
__global__ void __launch_bounds__(256) fixup_kernel_rec(const FixRec<T> *__restrict__ recs,
                                                        const int *__restrict__ block_start, int nplans) {
  const int k = find_range(block_start, nplans, blockIdx.x);
  const FixRec<T> &fr = recs[k];
  const int i = (blockIdx.x - block_start[k]) * 256 + threadIdx.x;
  if (i >= fr.nshared || (fr.cancel && *fr.cancel)) return;
  const int n = fr.snode[i];
  const int a = fr.soff[i], b = fr.soff[i + 1];
  const bool z = fr.dir_out && fr.dir_out[n];
  for (int q = 0; q < fr.nq; q++) fr.y[(size_t)n * fr.ld + q] = z ? T(0) : sum_partials(fr.partial, a, b, fr.nq, q);
}

// The fix-up records of a group (one per tile record, host copies): a batch
// sums the shared nodes of all its groups in one launch after their tiles.
template <typename T>
struct FixSource {
  virtual ~FixSource() = default;
  std::vector<FixRec<T>> fix;
};

struct FixLaunchBase {
  virtual ~FixLaunchBase() = default;
  virtual void launch(hipStream_t st) = 0;
};

template <typename T>
struct FixAll : FixLaunchBase {
  GroupMem mem;
  FixRec<T> *table = nullptr;
  int *block_start = nullptr;
  int nrec = 0, nblocks = 0;
  FixAll(const std::vector<FixRec<T>> &recs, DevArena *arena) {
    mem.arena = arena;
    std::vector<int> bs{0};
    for (const FixRec<T> &r : recs) bs.push_back(bs.back() + (r.nshared + 255) / 256);
    nrec = (int)recs.size();
    nblocks = bs.back();
    table = mem.upload(recs);
    block_start = mem.upload(bs);
  }
  void launch(hipStream_t st) override {
    if (!nblocks) return;
    hipLaunchKernelGGL((fixup_kernel_rec<T>), dim3(nblocks), dim3(256), 0, st, table, block_start, nrec);
    HIP_OK(hipGetLastError());
  }
};

template <typename T, int DIM, int P>
struct Group : GroupBase, FixSource<T> {
  GroupMem mem;
  // One record per (column chunk, plan): columns [q0, q0 + nq) of the plan,
  // every chunk in the same launch with partial slots of its own.
  BatchPlan<T> *table = nullptr;
  int *tile_start = nullptr;
  T *partial = nullptr;
  int nrec = 0, ntiles = 0, threads = 0;
  size_t lds = 0;
  bool one = false;  // every record has one column

  Group(const std::vector<dkt_plan *> &pls, const std::vector<const void *> &xs, const std::vector<void *> &ys,
        int nrhs, int masked, const std::vector<const int *> &cancel, DevArena *arena = nullptr, int max_cols = 0,
        bool colmajor = false) {
    mem.arena = arena;
    constexpr int NPE = Pow<P + 1, DIM>::v;
    const bool f64 = sizeof(T) == 8;
    auto dims_of = [](const dkt_plan *pl) {
      return TileDims{pl->max_nodes, pl->max_grp, pl->max_he, pl->max_rd, pl->max_cr, pl->tile_leaves, pl->max_hang};
    };
    // Columns of a record, separate items of the launch; column-major vectors
    // ([nrhs][N]) take one record per column.
    const int chunk = colmajor ? 1 : (max_cols > 0 ? std::min(nrhs, max_cols) : nrhs);
    for (dkt_plan *pl : pls)
      if (tile_lds_bytes<T, NPE>(dims_of(pl)) > kLdsLimit) throw std::invalid_argument("tile does not fit in LDS");
    const int nchunks = (nrhs + chunk - 1) / chunk;
    std::vector<int> ts{0};
    std::vector<size_t> poff;
    size_t ptot = 0;
    for (int c = 0; c < nchunks; c++)
      for (dkt_plan *pl : pls) {
        threads = std::max(threads, pl->tile_leaves);
        poff.push_back(ptot);
        ptot += pl->npartial * (size_t)chunk;
        push_items(ts, pl->ntiles * (size_t)std::min(chunk, nrhs - c * chunk));
        ranks += (double)pl->L * NPE * std::min(chunk, nrhs - c * chunk);
      }
    partial = mem.alloc<T>(std::max<size_t>(1, ptot));
    one = chunk == 1;
    std::vector<BatchPlan<T>> hp(pls.size() * nchunks);
    for (int c = 0; c < nchunks; c++) {
      const int q0 = c * chunk, nq = std::min(chunk, nrhs - q0);
      for (size_t k = 0; k < pls.size(); k++) {
        dkt_plan *pl = pls[k];
        BatchPlan<T> &r = hp[c * pls.size() + k];
        lds = std::max(lds, tile_lds_bytes<T, NPE>(dims_of(pl)));
        TileArgs &A = r.A;
        A.tiles = pl->tiles.p;
        A.tile_nodes = pl->tile_nodes.p;
        A.tile_out = pl->tile_out.p;
        A.leaf_loc = pl->leaf_loc.p;
        A.leaf_aux = pl->leaf_aux.p;
        A.group_ploc = pl->group_ploc.p;
        A.hentries = pl->hentries.p;
        A.readers = pl->readers.p;
        A.blocks = pl->blocks.p;
        A.carry_key = pl->carry_key.p;
        A.dir_in = masked == 1 ? pl->dirichlet.p : nullptr;
        A.dir_out = masked ? pl->dirichlet.p : nullptr;
        A.cancel = cancel.empty() ? nullptr : cancel[k];
        A.op = pl->op;
        A.hp = pl->hp;
        A.nq = nq;
        A.ld = colmajor ? 1 : nrhs;
        A.dims = dims_of(pl);
        r.kref = P == 2 ? (f64 ? (const T *)pl->kfac64.p : (const T *)pl->kfac32.p)
                        : (f64 ? (const T *)pl->kmat64.p : (const T *)pl->kmat32.p);
        r.carry_w = f64 ? (const T *)pl->carry_w64.p : (const T *)pl->carry_w32.p;
        const size_t coff = colmajor ? (size_t)q0 * pl->N : (size_t)q0;
        r.x = (const T *)xs[k] + coff;
        r.y = (T *)ys[k] + coff;
        r.partial = partial + poff[c * pls.size() + k];
        r.snode = pl->snode.p;
        r.soff = pl->soff.p;
        r.nshared = (int)pl->nshared;
        this->fix.push_back(FixRec<T>{pl->snode.p, pl->soff.p, r.partial, r.y, A.dir_out, A.cancel, nq, A.ld,
                                      (int)pl->nshared});
      }
    }
    table = mem.upload(hp);
    nrec = (int)hp.size();
    ntiles = ts.back();
    tile_start = mem.upload(ts);
  }

  void launch(hipStream_t st) override {
    auto kernel = one ? tile_kernel_batch<T, DIM, P, true> : tile_kernel_batch<T, DIM, P, false>;
    launch_items(ntiles, threads, [&](int first, int count) {
      hipLaunchKernelGGL(kernel, dim3(count), dim3(threads), lds, st, table, tile_start, nrec, first);
    });
  }
};

// A plan of a batch over point tiles.
template <typename T>
struct PointBatchPlan {
  PtArgs A;
  const T *kref, *x;
  T *y, *partial;
};

// All tiles and columns of a batch of point plans of one dim in one launch.
template <typename T, int DIM, bool CAP>
__global__ void __launch_bounds__(kTileThreads) point_kernel_batch(const PointBatchPlan<T> *__restrict__ plans,
                                                                   const int *__restrict__ item_start, int nplans,
                                                                   int first) {
  const int t = first + xcd_tile(blockIdx.x, gridDim.x);
  const int k = find_range(item_start, nplans, t);
  const PointBatchPlan<T> bp = plans[k];  // a copy: its fields live in scalar registers
  if (bp.A.cancel && *bp.A.cancel) return;
  point_body<T, DIM, CAP>(bp.A, t - item_start[k], bp.kref, bp.x, bp.y, bp.partial);
}

// Point plans of one dim: one tile launch with one record per (column chunk,
// plan).  A chunk's columns are separate work items of the launch; column-major
// vectors take one record per column.
template <typename T, int DIM, bool CAP>
struct PointGroup : GroupBase, FixSource<T> {
  GroupMem mem;
  PointBatchPlan<T> *table = nullptr;
  int *item_start = nullptr;
  T *partial = nullptr;
  int nrec = 0, nitems = 0, threads = 0;
  size_t lds = 0;

  PointGroup(const std::vector<dkt_plan *> &pls, const std::vector<const void *> &xs, const std::vector<void *> &ys,
             int nrhs, int masked, const std::vector<const int *> &cancel, DevArena *arena = nullptr, int max_cols = 0,
             bool colmajor = false) {
    mem.arena = arena;
    const bool f64 = sizeof(T) == 8;
    const int chunk = colmajor ? 1 : (max_cols > 0 ? std::min(nrhs, max_cols) : nrhs);
    std::vector<int> is{0};
    std::vector<PointBatchPlan<T>> hp;
    std::vector<size_t> poff;
    size_t ptot = 0;
    for (int q0 = 0; q0 < nrhs; q0 += chunk) {
      const int nq = std::min(chunk, nrhs - q0);
      for (size_t k = 0; k < pls.size(); k++) {
        dkt_plan *pl = pls[k];
        threads = std::max(threads, pl->tile_leaves);
        lds = std::max(lds, point_lds_bytes<T>(pl->max_slots, pl->max_units, pl->max_grp * pl->npe));
        const PtArgs A = pl->point_args(masked, cancel.empty() ? nullptr : cancel[k], nq, colmajor ? 1 : nrhs);
        const size_t coff = colmajor ? (size_t)q0 * pl->N : (size_t)q0;
        hp.push_back(PointBatchPlan<T>{A, f64 ? (const T *)pl->kmat64.p : (const T *)pl->kmat32.p,
                                       (const T *)xs[k] + coff, (T *)ys[k] + coff, nullptr});
        poff.push_back(ptot);
        ptot += pl->npartial * (size_t)nq;
        push_items(is, pl->ntiles * (size_t)nq);
        ranks += (double)pl->L * pl->npe * nq;
      }
    }
    partial = mem.alloc<T>(std::max<size_t>(1, ptot));
    for (size_t i = 0; i < hp.size(); i++) {
      dkt_plan *pl = pls[i % pls.size()];
      hp[i].partial = partial + poff[i];
      this->fix.push_back(FixRec<T>{pl->snode.p, pl->soff.p, hp[i].partial, hp[i].y, hp[i].A.dir_out, hp[i].A.cancel,
                                    hp[i].A.nq, hp[i].A.ld, (int)pl->nshared});
    }
    table = mem.upload(hp);
    nrec = (int)hp.size();
    nitems = is.back();
    item_start = mem.upload(is);
  }

  void launch(hipStream_t st) override {
    launch_items(nitems, threads, [&](int first, int count) {
      hipLaunchKernelGGL((point_kernel_batch<T, DIM, CAP>), dim3(count), dim3(threads), lds, st, table, item_start, nrec,
                         first);
    });
  }
};

// A conforming plan of a batch.
template <typename T>
struct ConfBatchPlan {
  ConfArgs A;
  const T *kref, *term_w, *x;
  T *y, *partial;
};

// All tiles of a batch of same-(dim, p) conforming plans in one launch.
template <typename T, int DIM, int P, bool CAP>
__global__ void __launch_bounds__(kTileThreads) conf_tile_kernel_batch(const ConfBatchPlan<T> *__restrict__ plans,
                                                                       const int *__restrict__ tile_start,
                                                                       int nplans, int first) {
  const int t = first + xcd_tile(blockIdx.x, gridDim.x);
  const int k = find_range(tile_start, nplans, t);
  const ConfBatchPlan<T> bp = plans[k];  // a copy: its fields live in scalar registers
  if (bp.A.cancel && *bp.A.cancel) return;
  conf_tile_body<T, DIM, P, CAP>(bp.A, t - tile_start[k], bp.kref, bp.term_w, bp.x, bp.y, bp.partial);
}

// Conforming plans of one (dim, p) (CAP: with per-level captured matrices):
// one tile launch and one fix-up launch, with one record per (column chunk,
// plan).  Each result is bitwise the plan's own
// matvec (same tile work, same fix-up order).
template <typename T, int DIM, int P, bool CAP>
struct ConfGroup : GroupBase, FixSource<T> {
  GroupMem mem;
  ConfBatchPlan<T> *table = nullptr;
  int *tile_start = nullptr;
  T *partial = nullptr;
  int nrec = 0, ntiles = 0, threads = 0;
  size_t lds = 0;

  ConfGroup(const std::vector<dkt_plan *> &pls, const std::vector<const void *> &xs, const std::vector<void *> &ys,
            int nrhs, int masked, const std::vector<const int *> &cancel, DevArena *arena = nullptr,
            int max_cols = 0, bool colmajor = false) {
    mem.arena = arena;
    constexpr int NPE = Pow<P + 1, DIM>::v;
    const bool f64 = sizeof(T) == 8;
    auto lds_of = [](const dkt_plan *pl) { return conf_lds_bytes<T, NPE>(pl->max_nodes, pl->nw); };
    const int chunk = colmajor ? 1 : (max_cols > 0 ? std::min(nrhs, max_cols) : nrhs);
    for (dkt_plan *pl : pls)
      if (lds_of(pl) > kLdsLimit) throw std::invalid_argument("tile does not fit in LDS");
    const int nchunks = (nrhs + chunk - 1) / chunk;
    std::vector<int> ts{0};
    std::vector<size_t> poff;
    size_t ptot = 0;
    for (int c = 0; c < nchunks; c++)
      for (dkt_plan *pl : pls) {
        threads = std::max(threads, pl->tile_leaves);
        poff.push_back(ptot);
        ptot += pl->npartial * (size_t)chunk;
        push_items(ts, pl->ntiles * (size_t)std::min(chunk, nrhs - c * chunk));
        ranks += (double)pl->L * NPE * std::min(chunk, nrhs - c * chunk);
      }
    partial = mem.alloc<T>(std::max<size_t>(1, ptot));
    std::vector<ConfBatchPlan<T>> hp(pls.size() * nchunks);
    std::vector<FixRec<T>> &hf = this->fix;
    hf.resize(pls.size() * nchunks);
    for (int c = 0; c < nchunks; c++) {
      const int q0 = c * chunk, nq = std::min(chunk, nrhs - q0);
      for (size_t k = 0; k < pls.size(); k++) {
        dkt_plan *pl = pls[k];
        const size_t ri = c * pls.size() + k;
        lds = std::max(lds, lds_of(pl));
        ConfArgs &A = hp[ri].A;
        A.tiles = pl->ctiles.p;
        A.tile_nodes = pl->tile_nodes.p;
        A.tile_out = pl->tile_out.p;
        A.leaf_loc = pl->leaf_loc.p;
        A.leaf_lev = pl->leaf_lev.p;
        A.virt_off = pl->virt_off.p;
        A.term_pk = pl->term_pk.p;
        A.term_spk = pl->term_spk.p;
        A.seg = pl->seg.p;
        A.nw = pl->nw;
        A.dir_in = masked == 1 ? pl->dirichlet.p : nullptr;
        A.dir_out = masked ? pl->dirichlet.p : nullptr;
        A.cancel = cancel.empty() ? nullptr : cancel[k];
        A.op = pl->op;
        A.hp = pl->hp;
        A.nq = nq;
        A.ld = colmajor ? 1 : nrhs;
        A.max_points = pl->max_nodes;
        A.tile_leaves = pl->tile_leaves;
        hp[ri].kref = P == 2 && !pl->per_level ? (f64 ? (const T *)pl->kfac64.p : (const T *)pl->kfac32.p)
                                               : (f64 ? (const T *)pl->kmat64.p : (const T *)pl->kmat32.p);
        hp[ri].term_w = f64 ? (const T *)pl->term_w64.p : (const T *)pl->term_w32.p;
        const size_t coff = colmajor ? (size_t)q0 * pl->N : (size_t)q0;
        hp[ri].x = (const T *)xs[k] + coff;
        hp[ri].y = (T *)ys[k] + coff;
        hp[ri].partial = partial + poff[ri];
        hf[ri] = FixRec<T>{pl->snode.p, pl->soff.p, partial + poff[ri], (T *)ys[k] + coff, A.dir_out, A.cancel,
                           nq, A.ld, (int)pl->nshared};
      }
    }
    table = mem.upload(hp);
    nrec = (int)hp.size();
    ntiles = ts.back();
    tile_start = mem.upload(ts);
  }

  void launch(hipStream_t st) override {
    launch_items(ntiles, threads, [&](int first, int count) {
      hipLaunchKernelGGL((conf_tile_kernel_batch<T, DIM, P, CAP>), dim3(count), dim3(threads), lds, st, table,
                         tile_start, nrec, first);
    });
  }
};

template <typename T>
// kind: 0 reference-semantics tiles, 1 conforming tiles, 3 point tiles; 2 and 4
// those of 1 and 3 with per-level captured element matrices.
GroupBase *make_group(int kind, int dim, int p, const std::vector<dkt_plan *> &pls,
                      const std::vector<const void *> &xs, const std::vector<void *> &ys, int nrhs, int masked,
                      const std::vector<const int *> &cancel = {}, DevArena *arena = nullptr, int max_cols = 0,
                      bool colmajor = false) {
#define DKT_GROUP(D, PP)                                                                                     \
  if (dim == D && p == PP) {                                                                                 \
    if (kind == 2)                                                                                           \
      return new ConfGroup<T, D, PP, true>(pls, xs, ys, nrhs, masked, cancel, arena, max_cols, colmajor);    \
    if (kind == 1)                                                                                           \
      return new ConfGroup<T, D, PP, false>(pls, xs, ys, nrhs, masked, cancel, arena, max_cols, colmajor);   \
    if constexpr (PP == 1) {                                                                                 \
      if (kind == 3)                                                                                         \
        return new PointGroup<T, D, false>(pls, xs, ys, nrhs, masked, cancel, arena, max_cols, colmajor);    \
      if (kind == 4)                                                                                         \
        return new PointGroup<T, D, true>(pls, xs, ys, nrhs, masked, cancel, arena, max_cols, colmajor);     \
    }                                                                                                        \
    if constexpr (!point_tiles(D, PP))                                                                       \
      return new Group<T, D, PP>(pls, xs, ys, nrhs, masked, cancel, arena, max_cols, colmajor);              \
  }
  DKT_GROUP(2, 1)
  DKT_GROUP(3, 1)
  DKT_GROUP(4, 1)
  DKT_GROUP(2, 2)
  DKT_GROUP(3, 2)
#undef DKT_GROUP
  throw std::invalid_argument("unsupported (dim, order)");
}

// Plans grouped by (kind as make_group's, dim, p): indices into the caller's list.
std::map<std::tuple<int, int, int>, std::vector<int>> by_kind_of(dkt_plan *const *plans, int nplans) {
  std::map<std::tuple<int, int, int>, std::vector<int>> by_kind;
  for (int k = 0; k < nplans; k++) {
    dkt_plan *pl = plans[k];
    if (pl->dry || pl->simple || (pl->per_level && !pl->conforming))
      throw std::invalid_argument("batch plans must be tiled device plans (reference or conforming)");
    by_kind[{(pl->points ? 3 : pl->conforming ? 1 : 0) + (pl->per_level ? 1 : 0), pl->dim, pl->order}].push_back(k);
  }
  return by_kind;
}

// One fix-up launch for the shared nodes of every group (the groups' tiles
// have all run before it; their partial slots and outputs are disjoint).
template <typename T>
std::unique_ptr<FixLaunchBase> fix_all(const std::vector<std::unique_ptr<GroupBase>> &groups, DevArena *arena) {
  std::vector<FixRec<T>> recs;
  for (const auto &g : groups)
    if (auto *fs = dynamic_cast<FixSource<T> *>(g.get())) recs.insert(recs.end(), fs->fix.begin(), fs->fix.end());
  return std::make_unique<FixAll<T>>(recs, arena);
}

struct GroupsLauncher : MatvecLauncher {
  std::vector<std::unique_ptr<GroupBase>> groups;
  std::unique_ptr<FixLaunchBase> fixes;
  void launch(hipStream_t st) override {
    for (auto &g : groups) g->launch(st);
    if (fixes) fixes->launch(st);
  }
};

}  // namespace

std::unique_ptr<MatvecLauncher> dkt::batch_matvec(int dtype, const std::vector<dkt_plan *> &plans,
                                                  const std::vector<const void *> &x, const std::vector<void *> &y,
                                                  int mask, const std::vector<const int *> &cancel, DevArena *arena) {
  auto out = std::make_unique<GroupsLauncher>();
  for (const auto &kv : by_kind_of(plans.data(), (int)plans.size())) {
    std::vector<dkt_plan *> pls;
    std::vector<const void *> xs;
    std::vector<void *> ys;
    std::vector<const int *> cs;
    for (int k : kv.second) {
      pls.push_back(plans[k]);
      xs.push_back(x[k]);
      ys.push_back(y[k]);
      cs.push_back(cancel[k]);
    }
    const auto [conf, dim, p] = kv.first;
    out->groups.emplace_back(dtype == 0 ? make_group<double>(conf, dim, p, pls, xs, ys, 1, mask, cs, arena)
                                        : make_group<float>(conf, dim, p, pls, xs, ys, 1, mask, cs, arena));
  }
  out->fixes = dtype == 0 ? fix_all<double>(out->groups, arena) : fix_all<float>(out->groups, arena);
  return out;
}

struct dkt_batch {
  std::vector<std::unique_ptr<GroupBase>> groups;  // the most work first
  std::unique_ptr<FixLaunchBase> fixes;  // the shared nodes of every group, after their tiles
  void launch(hipStream_t st) {
    for (auto &g : groups) g->launch(st);
    if (fixes) fixes->launch(st);
  }
  // Graph capture: the groups' tile launches are independent (their records,
  // partial slots and outputs are disjoint), so each goes on a branch of its
  // own, forked from and joined back to the caller's stream before the
  // fix-up; the replayed graph may then run them side by side.  The branch
  // streams have the default priority.  The group with the most work is recorded
  // first: in a replay a branch starts 9 to 20 us behind the one recorded before
  // it, which a long launch hides and a short one does not (24 trees of up to 35k
  // elements, p = 1 and 2 in turn, one FP32 column: 34.0 us, with the p = 1 group
  // first 46.2, with both on one stream 44.6; 8 FP64 columns on 18 trees of up to
  // 11k: 79.4, 88.3 and 90.5).
  // Large FP32 batches stay on one stream: side by side the launches slow each
  // other down by more than the overlap of their ends gains (182M leaf ranks: 535 us
  // against 522, 122M 374 and 369, 102M 318 and 317, but 68M 202 and 208; in FP64 182M
  // 976 and 994).
  static constexpr double kBranchRanks32 = 1e8;
  bool branches = false;
  std::vector<hipStream_t> branch;
  std::vector<hipEvent_t> done;
  hipEvent_t fork = nullptr;
  // Streams and events of the branches, made before the capture starts.
  void prepare_branches() {
    if (fork || !branches) return;
    HIP_OK(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
    for (size_t g = 1; g < groups.size(); g++) {
      hipStream_t s2 = nullptr;
      HIP_OK(hipStreamCreateWithFlags(&s2, hipStreamNonBlocking));
      branch.push_back(s2);
      hipEvent_t e = nullptr;
      HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      done.push_back(e);
    }
  }
  void capture(hipStream_t st) {
    if (!branches || done.size() + 1 != groups.size()) {
      launch(st);
      return;
    }
    HIP_OK(hipEventRecord(fork, st));
    for (size_t g = 0; g < done.size(); g++) {
      HIP_OK(hipStreamWaitEvent(branch[g], fork, 0));
      groups[g]->launch(branch[g]);
      HIP_OK(hipEventRecord(done[g], branch[g]));
    }
    groups.back()->launch(st);
    for (hipEvent_t e : done) HIP_OK(hipStreamWaitEvent(st, e, 0));
    if (fixes) fixes->launch(st);
  }
  bool use_graph = false;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~dkt_batch() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    for (hipEvent_t e : done) (void)hipEventDestroy(e);
    for (hipStream_t s2 : branch) (void)hipStreamDestroy(s2);
    if (fork) (void)hipEventDestroy(fork);
  }
};

extern "C" int dkt_batch_create(dkt_plan *const *plans, int nplans, int dtype, int nrhs, const void *const *x,
                                void *const *y, int masked, int flags, dkt_batch **out) {
  return guarded([&] {
    if (!plans || !x || !y || !out || nplans < 1) throw std::invalid_argument("null pointer or empty batch");
    if (dtype != 0 && dtype != 1) throw std::invalid_argument("dtype must be 0 (f64) or 1 (f32)");
    if (nrhs < 1 || nrhs > 64) throw std::invalid_argument("nrhs must be 1..64");
    if (masked < 0 || masked > 2) throw std::invalid_argument("masked must be 0, 1 or 2");
    for (int k = 0; k < nplans; k++) {
      if (!plans[k] || !x[k] || !y[k]) throw std::invalid_argument("null plan or vector");
      if (x[k] == (const void *)y[k]) throw std::invalid_argument("x and y must not alias");
    }
    const int cbits = (flags >> DKT_BATCH_COLUMNS_SHIFT) & 15;
    if (cbits > 7) throw std::invalid_argument("columns per launch must be 1, 2, 4, ..., 64");
    const int max_cols = cbits ? 1 << (cbits - 1) : 0;
    auto b = std::make_unique<dkt_batch>();
    if (flags & DKT_BATCH_PERSISTENT)
      throw std::invalid_argument(
          "DKT_BATCH_PERSISTENT is reserved: its kernel did not finish on the device and was removed; use the "
          "per-(dim, p) launches (with DKT_BATCH_GRAPH for a replayed graph)");
    for (const auto &kv : by_kind_of(plans, nplans)) {
      std::vector<dkt_plan *> pls;
      std::vector<const void *> xs;
      std::vector<void *> ys;
      for (int k : kv.second) {
        pls.push_back(plans[k]);
        xs.push_back(x[k]);
        ys.push_back(y[k]);
      }
      const auto [conf, dim, p] = kv.first;
      const bool cm = (flags & DKT_BATCH_COLUMN_MAJOR) != 0;
      GroupBase *g = dtype == 0
                         ? make_group<double>(conf, dim, p, pls, xs, ys, nrhs, masked, {}, nullptr, max_cols, cm)
                         : make_group<float>(conf, dim, p, pls, xs, ys, nrhs, masked, {}, nullptr, max_cols, cm);
      b->groups.emplace_back(g);
    }
    std::stable_sort(b->groups.begin(), b->groups.end(),
                     [](const auto &a, const auto &c) { return a->ranks > c->ranks; });
    double ranks = 0;
    for (const auto &g : b->groups) ranks += g->ranks;
    b->branches = b->groups.size() > 1 && (dtype == 0 || ranks <= dkt_batch::kBranchRanks32);
    b->fixes = dtype == 0 ? fix_all<double>(b->groups, nullptr) : fix_all<float>(b->groups, nullptr);
    b->use_graph = (flags & DKT_BATCH_GRAPH) != 0;
    *out = b.release();
  });
}

extern "C" int dkt_batch_run(dkt_batch *b, void *stream) {
  return guarded([&] {
    if (!b) throw std::invalid_argument("null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (!b->use_graph) {
      b->launch(st);
      return;
    }
    if (!st) throw std::invalid_argument("graph replay needs a non-default stream");
    if (!b->exec) {
      b->prepare_branches();
      HIP_OK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      try {
        b->capture(st);
      } catch (...) {
        hipGraph_t dropped = nullptr;
        (void)hipStreamEndCapture(st, &dropped);
        if (dropped) (void)hipGraphDestroy(dropped);
        throw;
      }
      HIP_OK(hipStreamEndCapture(st, &b->graph));
      HIP_OK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    HIP_OK(hipGraphLaunch(b->exec, st));
  });
}

extern "C" int dkt_batch_destroy(dkt_batch *b) {
  delete b;
  return 0;
}

extern "C" int dkt_batch_status(dkt_batch *b, int *err) {
  return guarded([&] {
    if (!b || !err) throw std::invalid_argument("null pointer");
    *err = 0;  // no launch of a batch waits on another
  });
}
