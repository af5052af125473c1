// Matvec over point tiles (p = 1; layout in point_plan.h): one tile and one
// column per workgroup, one leaf per work-item.
//
// The reference interpolates and transposes per leaf (FEM/include/matvec.h:
// 403-522).  128 leaves of a 3D sphere tree miss 340 ranks but only 112 different
// positions (256: 680 and 210), so here that work is done once per position:
//   1. stage the tile's nodes from x;
//   2. rows: each hanging point is the mean of two earlier points, level by
//      level; stale-buffer readers' points come from the replay (replay());
//   3. per leaf: gather its ranks' points, apply v = 2^(-level hp) K_ref u (p = 1:
//      in the Walsh-Hadamard basis that diagonalises K_ref), and form its
//      correction;
//   4. the points become accumulators: v is added rank by rank (two disjoint
//      leaves never share a point at the same rank, so a phase has no conflicts);
//   5. transposed sums: levels pass half of their accumulators to the points
//      behind them, each target summing its sources in plan order;
//   6. nodes touched by this tile only are written to y; nodes shared with
//      other tiles go to partial slots, summed in tile order by fixup_kernel.
// All reductions run in an order fixed by the plan: bitwise reproducible.
//
// What bounds it is the chain of round trips of a tile, not bandwidth: the maps
// come as two blocks copied straight to LDS (one trip each; loaded where they
// are used they cost 25 trips, 1.39 ms against 0.93 ms on the 4D workload of
// 15.3M elements), the header is read once into scalar registers (read in the
// level loops, each level waited 1,500 cycles for it), and every group of reads of
// a sum is issued before any is used.  LDS adds without a returned value
// (ds_add_f64, ds_add_f32) in place of the rank phases were no faster in FP64 and
// twice as slow in FP32.
#pragma once
#include "plan_common.h"
#include "point_plan.h"
#include "tile_kernel.h"

namespace dkt {

struct PtArgs {
  const PtTile *tiles;
  const uint32_t *blocks;
  const uint16_t *leaf_loc;
  const uint32_t *leaf_aux;
  const uint8_t *dir_in, *dir_out;
  const int *cancel;
  int op, hp, nq, ld;
  int max_slots, max_units;  // per-tile maxima that size the LDS carve
};

// LDS bytes of a point tile: the points, one block of maps, and for the replay
// the parent values of its sibling groups (nvalue = groups * nPe) and the buffer
// state.
template <typename T>
__host__ __device__ inline size_t point_lds_bytes(int max_slots, int max_units, int nvalue) {
  return (((size_t)max_slots * sizeof(T) + 15) & ~(size_t)15) + (size_t)max_units * 16 +
         (nvalue ? ((size_t)nvalue + 16) * sizeof(T) : 0);
}

// Copies n 16-byte units from global memory to LDS without passing through
// registers; the copy is complete after block_wait() and a barrier.
__device__ __forceinline__ void block_copy(unsigned char *lds, const uint32_t *__restrict__ src, int n) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  for (int u = wave * 64; u < n; u += nw * 64)
    if (u + lane < n)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void *)(src + (size_t)(u + lane) * 4),
          (__attribute__((address_space(3))) void *)(lds + (size_t)u * 16), 16, 0, 0);
}
__device__ __forceinline__ void block_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Parent-to-child interpolation (p = 1) with the buffer spread over a group of
// 2^DIM lanes: one axis at a time, a lane whose bit differs from the child's
// takes the mean of its value and its neighbour's.  differs: lane xor child.
template <int D, int DIM, typename T>
__device__ __forceinline__ T child_value(T a, uint32_t differs) {
  if constexpr (D == DIM) {
    return a;
  } else {
    const T b = xor_lane<D>(a);
    const T m = fma(b, T(0.5), T(0.5) * a);
    return child_value<D + 1, DIM>((differs >> D) & 1u ? m : a, differs);
  }
}

// Stale parent-buffer reads of a tile: a group of lanes (one per buffer slot)
// per replay block runs B_k = W_ck (parent nodes where present, else B_(k-1))
// over the block's hanging leaves and writes B_k at the missing ranks of each
// reader it passes.  P: the staged nodes; reader points are written to it.
// block: the tile's block A in LDS.  cst: 16 values, then the parent values.
template <typename T, int DIM>
__device__ __forceinline__ void replay(const PtTile &th, T *P, const unsigned char *block, T *cst) {
  constexpr int NPE = 1 << DIM;
  constexpr int G = NPE;
  const uint64_t *rd = reinterpret_cast<const uint64_t *>(block + th.readers_at());
  const uint64_t *blocks = reinterpret_cast<const uint64_t *>(block + th.blocks_at());
  const uint32_t *chn = reinterpret_cast<const uint32_t *>(block + th.chain_at());
  const uint16_t *gp = reinterpret_cast<const uint16_t *>(block + th.gploc_at());
  T *pval = cst + 16;
  const int tid = threadIdx.x, nthr = blockDim.x;
  for (int i = tid; i < th.ngrp * NPE; i += nthr) pval[i] = P[gp[i] != kNone ? gp[i] : 0];  // absent: not used
  // Buffer state at the tile start: slot s sums its terms (a header of slot
  // offsets, then the terms by slot), dealt to the R lanes of the slot.  R is
  // the plan's, not the workgroup's, so that the order of the sum does not
  // depend on the launch: a batch's workgroups have the work-items of its
  // largest tiles, NPE * R or more (those past them do the last slot again).
  if (th.ncr > 0) {
    const int lg = th.carry_log(), R = 1 << lg, slot = min(tid >> lg, NPE - 1), sub = tid & (R - 1);  // R = 4 .. 64
    const double *cw = reinterpret_cast<const double *>(block + th.carry_w_at());
    const uint32_t *ck = reinterpret_cast<const uint32_t *>(block + th.carry_key_at());
    const int lo = (int)ck[slot], hi = (int)ck[slot + 1];
    T acc = T(0);
    for (int c = lo + sub; c < hi; c += R) acc += (T)cw[c] * P[ck[c] & 0xFFFFu];
    for (int d = R >> 1; d; d >>= 1) acc += __shfl_xor(acc, d, 64);
    if (!sub) cst[slot] = acc;
  } else if (tid < NPE) {
    cst[tid] = T(0);
  }
  __syncthreads();
  const int lane = tid % G, ngroups = nthr / G;
  for (int bi = tid / G; bi < th.nbk(); bi += ngroups) {
    const uint64_t blk = blocks[bi];
    const int S = (int)(blk & 0xFFFFu), E = (int)((blk >> 16) & 0xFFFFu);
    const uint32_t r0 = ((uint32_t)(blk >> 32) & 0xFFFFu) + 1, nr = (uint32_t)(blk >> 48);  // the block's readers (+ 1)
    // Chain words and parent values do not depend on B: read ahead of their use.
    auto word = [&](int k) -> uint32_t { return chn[min(k, E)]; };
    auto value = [&](uint32_t w) -> T { return pval[((w >> 10) & 63u) * NPE + lane]; };
    int k = S == 0xFFFF ? 0 : S;
    T B = S == 0xFFFF ? cst[lane] : T(0);  // the cone start's missing slots are not read further on
    uint32_t w0 = word(k), w1 = word(k + 1);
    T x0 = value(w0);
    for (; k <= E; k++) {
      const uint32_t w2 = word(k + 2);
      const T x1 = value(w1);
      B = child_value<0, DIM>((w0 >> (16 + lane)) & 1u ? B : x0, w0 ^ (uint32_t)lane);
      const uint32_t r = (w0 >> 4) & 63u;
      if (r - r0 < nr) {
        const uint64_t rec = rd[r - 1];
        const uint32_t mask = (uint32_t)(rec >> 32);
        if (mask >> lane & 1u) P[(uint32_t)rec + __popc(mask & ((1u << lane) - 1u))] = B;
      }
      w0 = w1, w1 = w2;
      x0 = x1;
    }
  }
}

// f(Level<K>) for K = FIRST, FIRST + STEP, ... before END: compile-time indexes
// keep a copied header in registers.
template <int K>
struct Level {
  static constexpr int v = K;
};
template <int FIRST, int END, int STEP, typename F>
__device__ __forceinline__ void each_level(F &&f) {
  if constexpr (FIRST != END) {
    f(Level<FIRST>());
    each_level<FIRST + STEP, END, STEP>(f);
  }
}

// Item `item` of one plan: column item % nq of tile item / nq, so that the
// columns of a tile run next to each other and share its maps and the lines of
// the node-major vectors in L2 (the workgroup may have more work-items than
// the plan's tiles have leaves; they idle in the leaf phases and help in the
// loops).  CAP: per-level captured element matrices, kref pointing to
// [level][nPe][nPe].
template <typename T, int DIM, bool CAP>
__device__ __forceinline__ void point_body(const PtArgs &A, int item, const T *__restrict__ kref,
                                          const T *__restrict__ x, T *__restrict__ y, T *__restrict__ partial) {
  constexpr int NPE = 1 << DIM, NW = NPE / 2;
  constexpr int kLev = DIM;  // row levels of the reference's tiles: read with the header, not in the loop
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *P = reinterpret_cast<T *>(smem_raw);
  unsigned char *block = smem_raw + (((size_t)A.max_slots * sizeof(T) + 15) & ~(size_t)15);
  const int tile = A.nq == 1 ? item : item / A.nq, q = item - tile * A.nq;
  const PtTile th = A.tiles[tile];  // a copy: every field is loaded at once
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int nn = th.nnode, nlev = th.nlev, nrow = th.nrow, nlist = th.nodd + th.nrdp, nslot = nrow + nlist + th.ncor + 1;

  // Block A, and the leaf's ranks.
  block_copy(block, A.blocks + (size_t)th.a0 * 4, th.na);
  const bool active = tid < th.nleaf;
  uint32_t lw[NW];
  uint32_t aux = 0;
  if (active) {
    const uint32_t *lp = reinterpret_cast<const uint32_t *>(A.leaf_loc + (size_t)(th.leaf0 + tid) * NPE);
#pragma unroll
    for (int w = 0; w < NW; w++) lw[w] = lp[w];
    aux = A.leaf_aux[th.leaf0 + tid];
  } else {
#pragma unroll
    for (int w = 0; w < NW; w++) lw[w] = 0u;
  }
  auto loc_of = [&](int r) -> int { return (int)((lw[r >> 1] >> ((r & 1) * 16)) & 0xFFFFu); };
  block_wait();
  __syncthreads();

  // 1. Stage the nodes, a batch's values and Dirichlet flags loaded together.
  constexpr int kB = 2;
  const int32_t *nodes = reinterpret_cast<const int32_t *>(block);
  int o0[kB];  // output slots of the first batch: block A does not last until the write-out
  for (int j0 = tid, b0 = 0; j0 < nn; j0 += kB * nthr, b0 = 1) {
    int g[kB];
    T xv[kB];
    uint32_t d[kB];
#pragma unroll
    for (int b = 0; b < kB; b++) {
      const int j = min(j0 + b * nthr, nn - 1);
      g[b] = nodes[j];
      if (!b0) o0[b] = nodes[nn + j];
      d[b] = 0u;
    }
#pragma unroll
    for (int b = 0; b < kB; b++) xv[b] = x[(size_t)g[b] * A.ld + q];
    if (A.dir_in)
#pragma unroll
      for (int b = 0; b < kB; b++) d[b] = A.dir_in[g[b]];
#pragma unroll
    for (int b = 0; b < kB; b++)
      if (j0 + b * nthr < nn) P[j0 + b * nthr] = d[b] ? T(0) : xv[b];
  }
  __syncthreads();
  // 2. Rows by level, then the odd points and the readers'.
  const uint32_t *rows = reinterpret_cast<const uint32_t *>(block + th.rows_at()) - nn;  // by point
  auto row = [&](int p) {
    const uint32_t w = rows[p];
    P[p] = T(0.5) * (P[w & 0x1FFFu] + P[(w >> 13) & 0x1FFFu]);
  };
  auto level = [&](int p0, int p1) {
    for (int p = p0 + tid; p < p1; p += nthr) row(p);
    __syncthreads();
  };
  each_level<0, kLev, 1>([&](auto k) {
    if (k.v < nlev) level(th.past(k.v), th.past(k.v + 1));
  });
  for (int k = kLev; k < nlev; k++) level(A.tiles[tile].past(k), A.tiles[tile].past(k + 1));
  const uint32_t rw_odd = tid < nlist ? rows[nrow + tid] : 0u;
  if (nlist) {
    for (int i = tid; i < th.nodd; i += nthr) row(nrow + i);
    if (th.nbk()) replay<T, DIM>(th, P, block, reinterpret_cast<T *>(block + (size_t)A.max_units * 16));
    __syncthreads();
  }
  block_copy(block, A.blocks + (size_t)th.b0 * 4, th.nb);
  // 3. Elements.
  T v[NPE];
  T corr = T(0);
  if (active) {
    T u[NPE];
#pragma unroll
    for (int r = 0; r < NPE; r++) u[r] = P[loc_of(r)];
    if constexpr (CAP) {
      const T *K = kref + (size_t)aux_level(aux) * NPE * NPE;
#pragma unroll
      for (int i = 0; i < NPE; i++) {
        T acc = T(0);
#pragma unroll
        for (int j = 0; j < NPE; j++) acc += K[i * NPE + j] * u[j];
        v[i] = acc;
      }
    } else {
      const T scale = (T)ldexp(1.0, -aux_level(aux) * A.hp);
      if (A.op == 0)
        q1_apply<T, DIM, 0>(u, v, scale);
      else if (A.op == 1)
        q1_apply<T, DIM, 1>(u, v, scale);
      else
#pragma unroll
        for (int i = 0; i < NPE; i++) v[i] = scale * u[i];
    }
  }
  // The packed indices are opaque from here on, so the adds unpack them again
  // instead of keeping the gather's copies alive.
#pragma unroll
  for (int w = 0; w < NW; w++) asm volatile("" : "+v"(lw[w]));
  // Correction: sum over the missing ranks of 2^-|r xor c| v[r], folded one
  // axis at a time (a rank is missing when its point is no node).
  const bool corrected = (aux >> 9) & 1u;
  if (__ballot(corrected)) {
    T t[NPE];
#pragma unroll
    for (int r = 0; r < NPE; r++) t[r] = loc_of(r) >= nn ? v[r] : T(0);
    const int c = aux_child(aux);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      const bool cb = (c >> d) & 1;
      const T wa = cb ? T(0.5) : T(1), wb = cb ? T(1) : T(0.5);
#pragma unroll
      for (int i = 0; i < NPE >> (d + 1); i++) t[i] = fma(wb, t[2 * i + 1], wa * t[2 * i]);
    }
    corr = T(-2) * t[0];
  }
  block_wait();
  __syncthreads();
  // 4. The points become accumulators.
  {
    uint4 *z = reinterpret_cast<uint4 *>(P);
    for (int i = tid; i < (int)((nslot * sizeof(T) + 15) / 16); i += nthr) z[i] = uint4{0, 0, 0, 0};
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NPE; r++) {
    if (active) P[loc_of(r)] += v[r];
    if (r == 0 && corrected) P[aux >> 16] = corr;
    __syncthreads();
  }
  // 5. Transposed sums: onto the rows from the highest level down (the odd and
  //    reader points are scaled meanwhile), then onto the nodes.
  const uint32_t *block_a = A.blocks + (size_t)th.a0 * 4;  // in global memory
  for (int i = tid; i < nlist; i += nthr) {
    const uint32_t w = i < nthr ? rw_odd : block_a[th.rows_at() / 4 + nrow - nn + i];
    P[nrow + i] = ldexp(P[nrow + i], -(int)(w >> 26));
  }
  const uint4 *steps4 = reinterpret_cast<const uint4 *>(block);
  const uint2 *steps2 = reinterpret_cast<const uint2 *>(block) + 2 * th.nqs;
  uint64_t *quads = reinterpret_cast<uint64_t *>(block + th.quads_at());
  const uint32_t *pairs = reinterpret_cast<const uint32_t *>(block + th.pairs_at());
  // Onto the rows: a step that does not reach a target reads the zero slot, so
  // that every read of a group is issued before any is used.
  const uint32_t zero2 = (uint32_t)(nslot - 1) * 0x10001u;
  auto sums = [&](int t0, int t1, int ns) {
    for (int t = t0 + tid; t < t1; t += nthr) {
      T acc = T(0);
      for (int s = 0; s < ns; s++) {
        const uint2 st = steps2[s];
        const bool in0 = t - t0 < (int)(st.x >> 16), in1 = t - t0 < (int)(st.y >> 16);
        uint32_t w0 = pairs[in0 ? (int)(st.x & 0xFFFFu) + t - t0 : 0], w1 = pairs[in1 ? (int)(st.y & 0xFFFFu) + t - t0 : 0];
        w0 = in0 ? w0 : zero2;
        w1 = in1 ? w1 : zero2;
        acc += (P[w0 & 0xFFFFu] + P[w0 >> 16]) + (P[w1 & 0xFFFFu] + P[w1 >> 16]);
      }
      if (ns) P[t] += T(0.5) * acc;
    }
    steps2 += ns;
    __syncthreads();
  };
  for (int k = nlev - 1; k >= kLev; k--)
    sums(A.tiles[tile].past(k - 1), A.tiles[tile].past(k), (int)(A.tiles[tile].lv[k] >> 16));
  each_level<kLev - 1, 0, -1>([&](auto k) {
    if (k.v < nlev) sums(th.past(k.v - 1), th.past(k.v), (int)(th.lv[k.v] >> 16));
  });
  if (nlev < 2) __syncthreads();
  // Onto the nodes: first every quad's sum, in the quad's place (a node's list is
  // up to ten times the mean: dealt out by quad, no lane waits for another's
  // list), then each node adds its quads up.  In FP64 for FP32 too, at no cost in
  // time (24.8 and 24.7 us at 1.33M elements): a leaf's correction cancels its part of
  // these sums, and summed in FP32 the matvec's error was 1 to 2 % (stiffness) and up to
  // 14 % (mass) above that of interpolating per leaf; so it is the same.
  auto quad = [&](int i) -> double & { return *reinterpret_cast<double *>(quads + i); };
  for (int i = tid; i < th.nquad; i += nthr) {
    const uint64_t w = quads[i];
    quad(i) = ((double)P[w & 0xFFFFu] + (double)P[(w >> 16) & 0xFFFFu]) +
              ((double)P[(w >> 32) & 0xFFFFu] + (double)P[w >> 48]);
  }
  __syncthreads();
  // 6. Write-out.
  for (int j = tid, b = 0; j < nn; j += nthr, b++) {
    const int o = b == 0 ? o0[0] : b == 1 ? o0[1] : (int)block_a[nn + j];
    const bool zero = A.dir_out && A.dir_out[o >= 0 ? o : 0];
    double acc = 0.0;
    for (int s = 0; s < th.nqs; s++) {
      const uint4 st = steps4[s];
      if (j >= (int)(st.x >> 16)) break;  // steps cover ever fewer nodes
      const uint32_t sw[4] = {st.x, st.y, st.z, st.w};
      double v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool in = j < (int)(sw[i] >> 16);
        v[i] = quad(in ? (int)(sw[i] & 0xFFFFu) + j : 0);
        v[i] = in ? v[i] : 0.0;
      }
      acc += (v[0] + v[1]) + (v[2] + v[3]);
    }
    if (o == INT32_MIN) continue;
    const T r = (T)fma(0.5, acc, (double)P[j]);
    if (o >= 0)
      y[(size_t)o * A.ld + q] = zero ? T(0) : r;
    else
      partial[(size_t)(-o - 1) * A.nq + q] = r;
  }
}

template <typename T, int DIM, bool CAP>
__global__ void __launch_bounds__(kTileThreads) point_kernel(PtArgs A, const T *__restrict__ kref,
                                                             const T *__restrict__ x, T *__restrict__ y,
                                                             T *__restrict__ partial) {
  if (A.cancel && *A.cancel) return;
  point_body<T, DIM, CAP>(A, xcd_tile(blockIdx.x, gridDim.x), kref, x, y, partial);
}

}  // namespace dkt
