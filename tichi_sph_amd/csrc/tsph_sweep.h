// Neighbour iteration shared by the step and adjoint sweeps.
//
// Storage is in cell order.  The 27 (3D) / 9 (2D) cells of a particle's
// neighbourhood are visited as 9 / 3 contiguous row runs: cells (x-R .. x+R)
// of one (y, z) row have consecutive codes and therefore consecutive slots,
// in the reference's template order (x fastest, sph_config.py:219-224) and
// in-cell order.
#pragma once

#include "tsph_host.h"

namespace tsph {

// Visit the row runs [j0, j1) of `cstart`'s object in the cells around c[]:
// one run per (dy, dz) row, in template order.
template <class T, class F>
__device__ __forceinline__ void walk_runs(const KP<T>& k, const int* __restrict__ cstart,
                                          const int* c, F&& f) {
  const int R = k.R;
  const int zr = k.dim == 3 ? R : 0;
#pragma unroll 1
  for (int dz = -zr; dz <= zr; ++dz) {
#pragma unroll 1
    for (int dy = -R; dy <= R; ++dy) {
      int c0 = dim_encode(k, wadd(c[0], -R), wadd(c[1], dy), wadd(c[2], dz));
      long lo = c0 < 1 ? 1 : (long)c0;
      long hi = (long)c0 + 2 * R;
      if (hi > k.node_num - 1) hi = k.node_num - 1;
      if (lo > hi) continue;
      f(cstart[lo], cstart[hi + 1]);
    }
  }
}

// Visit every candidate slot of `cstart`'s object in the cells around c[].
template <class T, class F>
__device__ __forceinline__ void walk_cells(const KP<T>& k, const int* __restrict__ cstart,
                                           const int* c, F&& f) {
  walk_runs(k, cstart, c, [&](int j0, int j1) {
    for (int j = j0; j < j1; ++j) f(j);
  });
}

// Candidate walk with prefetch: the records load(j) of a run's candidates are
// gathered U at a time, all U in flight together, then f(j, record) runs for
// each in walk order.  Cell walks are bound by the latency of these gathers
// (a one-candidate-at-a-time loop waits a full round trip per candidate),
// not by their number.
template <int U, class T, class Load, class F>
__device__ __forceinline__ void walk_cells_prefetch(const KP<T>& k, const int* __restrict__ cstart,
                                                    const int* c, Load&& load, F&& f) {
  walk_runs(k, cstart, c, [&](int j0, int j1) {
    for (int j = j0; j < j1; j += U) {
      decltype(load(j0)) rec[U];
#pragma unroll
      for (int u = 0; u < U; ++u) rec[u] = load(j + u < j1 ? j + u : j);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j + u < j1) f(j + u, rec[u]);
    }
  });
}

// The pass A form: the prefetched record is the candidate's position.
template <int U, class T, class F>
__device__ __forceinline__ void walk_cells_batched(const KP<T>& k, const int* __restrict__ cstart,
                                                   const int* c, const V4<T>* __restrict__ pos,
                                                   F&& f) {
  walk_cells_prefetch<U>(k, cstart, c, [&](int j) { return pos[j]; }, f);
}
constexpr int kPassAU = 4;

template <class T>
__device__ __forceinline__ T rest_psi_of(const KP<T>& k, const T* rdens, int i) {
  return k.solver == TSPH_VFSPH ? T(1) : rdens[i];
}

// Iterate a particle's fluid neighbours: the recorded list, or, when the list
// overflowed, the cell walk with the same in-range test.
template <class T, class L, class F>
__device__ __forceinline__ void for_fluid_nbrs(const KP<T>& k, int i, int cap, int nf,
                                               const L& list,
                                               const int* __restrict__ cstart,
                                               const V4<T>* __restrict__ pos, V4<T> p, F&& f) {
  if (nf <= k.list_cap_f) {
    for (int s = 0; s < nf; ++s) f(list[(long)s * cap + i]);
  } else {
    int c[3];
    node_encode(k, p.x, p.y, p.z, c);
    walk_cells(k, cstart, c, [&](int j) {
      V4<T> q = pos[j];
      T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
      if (r2 > T(0) && r2 <= k.r2max) f(j);
    });
  }
}
template <class T, class F>
__device__ __forceinline__ void for_bound_nbrs(const KP<T>& k, int i, int cap, int nbb,
                                               const int* __restrict__ list,
                                               const int* __restrict__ cstart,
                                               const V4<T>* __restrict__ bpos, V4<T> p, F&& f) {
  if (nbb <= k.list_cap_b) {
    for (int s = 0; s < nbb; ++s) f(list[(long)s * cap + i]);
  } else {
    int c[3];
    node_encode(k, p.x, p.y, p.z, c);
    walk_cells(k, cstart, c, [&](int j) {
      V4<T> q = bpos[j];
      T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
      if (r2 > T(0) && r2 <= k.r2max) f(j);
    });
  }
}

template <class T>
struct Rec2 {
  V4<T> a, b;
};
template <class T>
struct Rec3 {
  V4<T> a, b, c;
};

// ---------------------------------------------------------------------------
// Cooperative list sweeps.  A group of kCoop adjacent lanes shares one
// particle; lane c of the group takes list slots c, c + kCoop, c + 2 kCoop,
// ...  At each step the group's lanes gather kCoop consecutive neighbours of
// the same particle, which lie in one or two cells, and the 64 lanes of a
// wave gather from about half as many cache sectors as with one lane per
// particle (whose lanes drift apart through their lists).  The sweeps are
// bound by the number of L1 sectors their gathers touch, not by the number
// of gathers.  The group's partial sums are combined by a butterfly, which
// leaves the same value in every lane of the group.
// ---------------------------------------------------------------------------
constexpr int kCoop = 4;    // lanes per particle of the gather-heavy sweeps
constexpr int kCoopU = 2;   // lanes per particle of the update sweep (one gather per pair)
constexpr int kCoopNb = 4;  // gathers in flight per lane
// In a grouped launch the scenes' constants take registers besides: fewer in flight in
// FP64, for the waves, and in 2D, where the 12 neighbours (32 in 3D) take three slots
// of each of four lanes.  (How many does not change a sum.)
// us with 4 / 3 in flight, 24 2D scenes of 25-35k: psi 35.3 / 33.5, update 23.9 / 23.2,
// advection (and velocity update) 43.6 / 41.2; 3D FP32 psi, 3 x 180k, 43.7 / 47.5.  FP64
// with 4 / 3 / 2: psi 2D 901 tiles 27.1 / 23.8 / 23.0, 3D 908 tiles 40.8 / 38.2 / 35.1,
// 2024 80.6 / 76.0 / 69.7, 19404 (R = 4) 742 / 787 / 784; advection 3D 908 44.5 / 46.0 /
// 42.0, 2799 118 / 122 / 113, 19404 842 / 885 / 874; update with 4 / 3 2D 2798 36.7 / 34.9,
// 3D 2799 66.9 / 62.1, 19404 472 / 491.
template <class T, class Rec, int R>
constexpr int group_nb(int dim) {
  const bool two = sizeof(Rec) > sizeof(V4<T>);  // psi, advection; the update: one vector
  return dim == 2 ? 3 : sizeof(T) == 4 ? 4 : !two ? 3 : R == 1 ? 2 : 4;
}

// A block covers kBlock / C particles, one per group: C rounds of as many
// particles in a C-th of the blocks leave a small launch short of blocks and
// a large one with long last blocks, and hold more registers.  In us, C rounds
// and one: psi, update, advection at 1M 74.0, 49.6, 74.4 and 68.9, 46.6,
// 66.1; at 4M 370, 250, 370 and 335, 243, 340.
//
// Blocks of a sweep over n particles: C per kBlock particles, so that they are
// also the sub-tiles of a grouped launch's fluid tiles and a scene's block
// partials are the same in both.
template <int C>
__host__ __device__ __forceinline__ int coop_blocks(int n) {
  return (int)(((long)(n > 0 ? n : 1) + kBlock - 1) / kBlock) * C;
}
// Round r of the R rounds of block blk: the sub-tile of the particles it
// takes, and the particle of this thread's group in a sub-tile (n or more:
// none).  R = 1 except in grouped launches (for_coop_tiles).
template <int R = 1>
__device__ __forceinline__ int coop_sub(Blk blk, int r = 0) {
  return xcd_block(blk.b, blk.nb) * R + r;
}
template <int C>
__device__ __forceinline__ int coop_particle(int sub) {
  return sub * (kBlock / C) + (int)(threadIdx.x / C);
}
// Every scene's sweep in a grouped launch; f(entry, blk).  A block takes R of
// a fluid tile's C sub-tiles: finding a tile's scene and its constants is a
// chain of dependent loads, which R = C pays once per tile, while split tiles
// (R = 1, as in a single scene's launch) leave no block waiting for its last round.
//   Advection is split always, us with the velocity update, split / whole: 2D 2798
// tiles 40.9 / 41.7, FP64 72.0 / 78.0, 19150 tiles FP64 531 / 579; 3D 2799 tiles 58.1 /
// 61.3, FP64 117 / 126.
//   Psi up to 2048 tiles, us split / whole: 3D 56 tiles 5.3 / 10.9, 908 20.8 / 21.5, 1440
// 29.2 / 32.6, 2024 38.5 / 38.6, 2799 50.3 / 51.6, 19404 394 / 403; but 2D 1135 17.4 /
// 15.8, 1428 21.0 / 22.3, 2026 27.6 / 25.5, 2360 31.1 / 27.3, 19150 256 / 228.  In FP64 up
// to 3072: 3D 2338 83.6 / 92.1, 2799 99.6 / 104, 5555 223 / 220, 19404 767 / 740; 2D 2360
// 52.7 / 54.5, 2798 61.0 / 61.2, 3471 76.0 / 75.0, 19150 455 / 428.
//   The update while its blocks are about all on the chip at once: a scene's first block
// sends the host the stop signal, and a block that waits for a place sends it late, so
// that the next kernel comes late.  Steps, us split / whole: 3D 449 tiles 269 / 285, 602
// 298 / 322, 908 358 / 348, 1440 445 / 437; FP64 218 291 / 294, 449 371 / 372, 676 445 /
// 438, 760 462 / 449, 908 556 / 539, 2D 598 263 / 262, 671 274 / 271, 756 286 / 283 (the
// kernel alone is the faster for being split: 760 tiles 20.2 / 20.5, 602 17.6 / 20.1).
template <class T, int C, int R, class F>
__device__ __forceinline__ void for_coop_tiles(const char* __restrict__ tab, int ns, F&& f) {
  constexpr int split = C / R;
  const int total = tile_prefix<T, kTileFluid>(tab, ns)[ns] * split;
  for (int t = blockIdx.x; t < total; t += gridDim.x)
    on_tile<T, kTileFluid>(tab, ns, t / split, [&](const SceneEntry<T>& e, int, Blk tile) {
      f(e, Blk{tile.b * split + t % split, tile.nb * split});
    });
}
template <class T>
inline bool psi_split(int tiles) { return tiles < (sizeof(T) == 8 ? 3072 : 2048); }
template <class T>
inline bool update_split(int tiles) { return tiles < (sizeof(T) == 8 ? 512 : 896); }
template <int C>
__device__ __forceinline__ int coop_lane() {
  return threadIdx.x & (C - 1);
}
template <int C, class T>
__device__ __forceinline__ T group_sum(T v) {
#pragma unroll
  for (int o = 1; o < C; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One list, lane c's share of it, NB gathers in flight per lane; the next trip's
// list entries are loaded right after this one's records are requested, so that a
// trip costs one round trip to memory instead of two (index, then record).  Every
// trip gathers NB records without a branch: a slot past the list's end reads the last slot again (a line the
// group holds already) and pair(record, false) leaves it out of the sums, so
// that the loads of a trip issue back to back.  With a branch around each
// load instead, a trip's loads went out one exec-mask change at a time: where
// few waves are in flight (8,000 particles in 3D, four rounds a block then)
// psi took 12.3 us with it and 10.2 without, update 8.8 and 7.2, advection
// 12.8 and 10.5.  From 200k particles on the sweeps are bound by their cache
// accesses and take the same time (1M: psi 75.6 and 74.0 us); fewer registers
// hold the same loads (psi 93 -> 78).
template <int C, class Rec, int NB = kCoopNb, class Load, class Pair>
__device__ __forceinline__ void sweep_one_list_coop(int cap, int i, int c,
                                                    const int* __restrict__ list, int n,
                                                    Load&& load, Pair&& pair) {
  if (c >= n) return;
  const int last = n - 1;
  int j[NB];
#pragma unroll
  for (int u = 0; u < NB; ++u) j[u] = list[(long)min(c + C * u, last) * cap + i];
  for (int s0 = c;;) {
    Rec d[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) d[u] = load(j[u]);
    const int s1 = s0 + C * NB;
    if (s1 < n) {
#pragma unroll
      for (int u = 0; u < NB; ++u) j[u] = list[(long)min(s1 + C * u, last) * cap + i];
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) pair(d[u], s0 + C * u < n);
    if (s1 >= n) break;
    s0 = s1;
  }
}

// A particle's fluid list, then its boundary list, for lane c of its group.  A
// particle whose list overflowed is swept by lane 0 alone, walking the cells with
// the lists' in-range test.
template <int C, class T, class Rec, int NB = kCoopNb, int NB2D = NB, class LoadF, class LoadB,
          class PairF, class PairB>
__device__ __forceinline__ void sweep_lists_coop(const KP<T>& k, int cap, int i, int c, V4<T> p,
                                                 const int* __restrict__ fstart,
                                                 const int* __restrict__ bstart,
                                                 const V4<T>* __restrict__ fpos,
                                                 const V4<T>* __restrict__ bpos,
                                                 const int* __restrict__ nbr_f,
                                                 const int* __restrict__ nbr_b, int nf, int nbb,
                                                 LoadF&& load_f, LoadB&& load_b, PairF&& pair_f,
                                                 PairB&& pair_b) {
  if (nf <= k.list_cap_f && nbb <= k.list_cap_b) {
    if (NB2D != NB && k.dim == 2)
      sweep_one_list_coop<C, Rec, NB2D>(cap, i, c, nbr_f, nf, load_f, pair_f);
    else
      sweep_one_list_coop<C, Rec, NB>(cap, i, c, nbr_f, nf, load_f, pair_f);
    if (nbb > 0) sweep_one_list_coop<C, Rec, NB>(cap, i, c, nbr_b, nbb, load_b, pair_b);
    return;
  }
  if (c != 0) return;
  int cc[3];
  node_encode(k, p.x, p.y, p.z, cc);
  walk_cells(k, fstart, cc, [&](int j) {
    V4<T> q = fpos[j];
    T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
    if (r2 > T(0) && r2 <= k.r2max) pair_f(load_f(j), true);
  });
  if (nbr_b == nullptr) return;
  walk_cells(k, bstart, cc, [&](int j) {
    V4<T> q = bpos[j];
    T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
    if (r2 > T(0) && r2 <= k.r2max) pair_b(load_b(j), true);
  });
}

// ---------------------------------------------------------------------------
// Cooperative cell walk.  A quad of lanes shares one particle.  The quad reads
// four consecutive candidates of a row run at once, tests them, and appends
// those in range to a list in LDS, in walk order (a candidate's slot is the
// quad's count so far plus the hits among the lanes before it); whenever the
// list fills, and at the end, the quad works the list off, each lane taking
// every fourth slot, so that the pair math runs on full quads.  The runs of a
// particle's rows are looked up once, side by side, and only the rows that
// hold particles are walked.
// ---------------------------------------------------------------------------
constexpr int kQuad = 4;
constexpr int kQuads = kBlock / kQuad;  // particles per block
constexpr int kWalkRows = 9;            // row runs looked up at a time
constexpr int kWalkS = 48;              // list slots per particle
// Candidates and list slots in flight per lane.  Pass A at 64k / 195k: 2 and 2
// 51 / 102 us, 2 and 1 40 / 88, 1 and 1 45 / 95, 3 and 1 39 / 85.
constexpr int kWalkU = 3;
constexpr int kWalkNb = 1;

struct WalkLds {
  int2 run[kWalkRows][kQuads];
  int list[kWalkS][kQuads];
};

// The value of lane K of the quad, in all its lanes.
template <int K>
__device__ __forceinline__ int quad_lane(int v) {
  return __builtin_amdgcn_update_dpp(0, v, K * 0x55, 0xf, 0xf, true);
}
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(quad_lane<K>(__float_as_int(v)));
}
template <int K>
__device__ __forceinline__ double quad_lane(double v) {
  return __hiloint2double(quad_lane<K>(__double2hiint(v)), quad_lane<K>(__double2loint(v)));
}
// acc + the quad's four values in lane order, one rounding each.
template <class T>
__device__ __forceinline__ T quad_add(T acc, T v) {
  TSPH_STRICT
  acc = acc + quad_lane<0>(v);
  acc = acc + quad_lane<1>(v);
  acc = acc + quad_lane<2>(v);
  return acc + quad_lane<3>(v);
}
// The quad's four votes, lane 0 in bit 0.
__device__ __forceinline__ unsigned quad_vote(bool v) {
  const unsigned long long m = __ballot(v);
  const unsigned lane = threadIdx.x & 63;
  const unsigned half = lane < 32 ? (unsigned)m : (unsigned)(m >> 32);
  return (half >> (lane & 28)) & 15u;
}
// LDS written by lanes of this wave is read by others of it: the wave's LDS
// accesses complete in order, so only the compiler has to keep theirs.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The walk around cell cc[].  bounds(lo, hi, &split) is the range of candidates
// of the cells lo .. hi (one row run).  Where these cells' ranges do not follow
// one another it sets split (SPLITS: it may), and the quad walks the rows from
// there on cell by cell.  fetch(s) is candidate s of a range; take(fetched,
// &apart) says whether it belongs to the list, and apart whether r > 0 (r = 0
// goes to the list with a mark).  load(j) gathers what the pair terms need of
// candidate j; term(record, j, valid, apart) adds one list slot per lane
// (valid: the lane holds one) and runs with the whole quad.
template <class T>
struct Cand {
  V4<T> q;
  int j;  // negative: none
};
// walk_quad_runs: the rows (CELLS: the cells) from run0 on; the row at which it
// stopped for a split one, or -1 when all are done.
template <bool CELLS, bool SPLITS, class T, class Bounds, class Fetch, class Take, class Load,
          class Term>
__device__ __forceinline__ int walk_quad_runs(const KP<T>& k, const int* cc, WalkLds& lds,
                                              int run0, Bounds&& bounds, Fetch&& fetch,
                                              Take&& take, Load&& load, Term&& term) {
  const int c = threadIdx.x & (kQuad - 1), g = threadIdx.x / kQuad;
  const unsigned below = (1u << c) - 1;
  const int R = k.R, side = 2 * R + 1, rows = k.dim == 3 ? side * side : side;
  const int runs = CELLS ? rows * side : rows;
  for (; run0 < runs; run0 += kWalkRows) {
    int nrun = 0;
    bool split = false;
#pragma unroll
    for (int q = 0; q < (kWalkRows + kQuad - 1) / kQuad; ++q) {
      const int r = c + kQuad * q, id = run0 + r;
      int2 run = make_int2(0, 0);
      if (r < kWalkRows && id < runs) {
        const int row = CELLS ? id / side : id, dx = CELLS ? id - row * side - R : -R;
        const int dy = row % side - R, dz = k.dim == 3 ? row / side - R : 0;
        const int c0 = dim_encode(k, wadd(cc[0], dx), wadd(cc[1], dy), wadd(cc[2], dz));
        const long lo = c0 < 1 ? 1 : (long)c0;
        long hi = CELLS ? (long)c0 : (long)c0 + 2 * R;
        if (hi > k.node_num - 1) hi = k.node_num - 1;
        if (lo <= hi) run = bounds((int)lo, (int)hi, &split);
      }
      const unsigned v = quad_vote(run.x < run.y);
      if (run.x < run.y) lds.run[nrun + __popc(v & below)][g] = run;
      nrun += __popc(v);
    }
    if (SPLITS && !CELLS && quad_vote(split)) return run0;
    if (nrun == 0) continue;
    wave_lds_fence();
    int at = 0, j = lds.run[0][g].x, end = lds.run[0][g].y, cnt = 0;
    bool more = true;
    Cand<T> cur[kWalkU];
    auto trip = [&](Cand<T>* d) {
#pragma unroll
      for (int u = 0; u < kWalkU; ++u) {
        const int s = j + c + kQuad * u;
        d[u] = fetch(s < end ? s : end - 1);
        if (s >= end) d[u].j = -1;
      }
    };
    trip(cur);
    while (more) {
      while (more && cnt <= kWalkS - kQuad * kWalkU) {
        // the next trip's candidates are requested before this one's tests
        j += kQuad * kWalkU;
        if (j >= end) {
          ++at;
          more = at < nrun;
          if (more) {
            const int2 run = lds.run[at][g];
            j = run.x;
            end = run.y;
          }
        }
        Cand<T> nxt[kWalkU];
        if (more) trip(nxt);
#pragma unroll
        for (int u = 0; u < kWalkU; ++u) {
          bool apart;
          const bool hit = take(cur[u], &apart) && cur[u].j >= 0;
          const unsigned v = quad_vote(hit);
          // the sign bit marks a candidate at r = 0
          if (hit) lds.list[cnt + __popc(v & below)][g] = apart ? cur[u].j : ~cur[u].j;
          cnt += __popc(v);
        }
        if (more) {
#pragma unroll
          for (int u = 0; u < kWalkU; ++u) cur[u] = nxt[u];
        }
      }
      wave_lds_fence();
      for (int s0 = 0; s0 < cnt; s0 += kQuad * kWalkNb) {
        int e[kWalkNb];
        decltype(load(0)) rec[kWalkNb];
#pragma unroll
        for (int u = 0; u < kWalkNb; ++u) e[u] = lds.list[min(s0 + c + kQuad * u, cnt - 1)][g];
#pragma unroll
        for (int u = 0; u < kWalkNb; ++u) rec[u] = load(e[u] < 0 ? ~e[u] : e[u]);
#pragma unroll
        for (int u = 0; u < kWalkNb; ++u)
          term(rec[u], e[u] < 0 ? ~e[u] : e[u], s0 + c + kQuad * u < cnt, e[u] >= 0);
      }
      wave_lds_fence();
      cnt = 0;
    }
  }
  return -1;
}
template <bool SPLITS, class T, class Bounds, class Fetch, class Take, class Load, class Term>
__device__ __forceinline__ void walk_quad_cells(const KP<T>& k, const int* cc, WalkLds& lds,
                                                Bounds&& bounds, Fetch&& fetch, Take&& take,
                                                Load&& load, Term&& term) {
  const int row = walk_quad_runs<false, SPLITS>(k, cc, lds, 0, bounds, fetch, take, load, term);
  if constexpr (SPLITS)
    if (row >= 0)
      walk_quad_runs<true, SPLITS>(k, cc, lds, row * (2 * k.R + 1), bounds, fetch, take, load, term);
}

// Every candidate of the cells around cc[], a quad per particle, without a
// list: the quad's lanes look the row runs up side by side and take every
// fourth candidate of a run, U gathers in flight per lane; f(j, record, valid).
// Sums are per lane.
template <int U, class T, class Load, class F>
__device__ __forceinline__ void walk_quad_all(const KP<T>& k, const int* __restrict__ cstart,
                                              const int* cc, Load&& load, F&& f) {
  const int c = threadIdx.x & (kQuad - 1);
  const int R = k.R, side = 2 * R + 1, rows = k.dim == 3 ? side * side : side;
  constexpr int kQ = (kWalkRows + kQuad - 1) / kQuad;
  for (int row0 = 0; row0 < rows; row0 += kWalkRows) {
    int lo_[kQ], hi_[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int r = c + kQuad * q, row = row0 + r;
      lo_[q] = hi_[q] = 0;
      if (r < kWalkRows && row < rows) {
        const int dy = row % side - R, dz = k.dim == 3 ? row / side - R : 0;
        const int c0 = dim_encode(k, wadd(cc[0], -R), wadd(cc[1], dy), wadd(cc[2], dz));
        const long lo = c0 < 1 ? 1 : (long)c0;
        long hi = (long)c0 + 2 * R;
        if (hi > k.node_num - 1) hi = k.node_num - 1;
        if (lo <= hi) {
          lo_[q] = cstart[lo];
          hi_[q] = cstart[hi + 1];
        }
      }
    }
    auto run = [&](int j0, int j1) {
      for (int j = j0; j < j1; j += kQuad * U) {
        decltype(load(0)) rec[U];
#pragma unroll
        for (int u = 0; u < U; ++u) rec[u] = load(min(j + c + kQuad * u, j1 - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) f(j + c + kQuad * u, rec[u], j + c + kQuad * u < j1);
      }
    };
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      run(quad_lane<0>(lo_[q]), quad_lane<0>(hi_[q]));
      if (4 * q + 1 < kWalkRows) run(quad_lane<1>(lo_[q]), quad_lane<1>(hi_[q]));
      if (4 * q + 2 < kWalkRows) run(quad_lane<2>(lo_[q]), quad_lane<2>(hi_[q]));
      if (4 * q + 3 < kWalkRows) run(quad_lane<3>(lo_[q]), quad_lane<3>(hi_[q]));
    }
  }
}

// The same by L lanes per particle: a quad, or one lane with U1 gathers in flight.
template <int L, int U4, int U1, class T, class Load, class F>
__device__ __forceinline__ void walk_all(const KP<T>& k, const int* __restrict__ cstart,
                                         const int* cc, Load&& load, F&& f) {
  static_assert(L == kQuad || L == 1, "a quad or one lane");
  if constexpr (L == kQuad)
    walk_quad_all<U4>(k, cstart, cc, load, f);
  else
    walk_cells_prefetch<U1>(k, cstart, cc, load, [&](int j, const auto& d) { f(j, d, true); });
}

// The same candidates, and a list's slots, by one lane in the order of a quad: f and
// pair also get the lane of the quad that would take each, so that sums kept apart
// by it and added as group_sum does are a quad's bit for bit.
template <int U, class T, class Load, class F>
__device__ __forceinline__ void walk_as_quad(const KP<T>& k, const int* __restrict__ cstart,
                                             const int* cc, Load&& load, F&& f) {
  static_assert(U % kQuad == 0, "a trip is whole rounds of a quad");
  walk_runs(k, cstart, cc, [&](int j0, int j1) {
    for (int j = j0; j < j1; j += U) {
      decltype(load(0)) rec[U];
#pragma unroll
      for (int u = 0; u < U; ++u) rec[u] = load(min(j + u, j1 - 1));
#pragma unroll
      for (int u = 0; u < U; ++u) f(u % kQuad, j + u, rec[u], j + u < j1);
    }
  });
}
template <class Rec, int NB, class T, class Load, class Pair>
__device__ __forceinline__ void sweep_list_as_quad(const KP<T>& k, int cap, int i, const V4<T>& p,
                                                   const int* cc, const int* __restrict__ fstart,
                                                   const V4<T>* __restrict__ fpos,
                                                   const int* __restrict__ list, int n,
                                                   Load&& load, Pair&& pair) {
  static_assert(NB % kQuad == 0, "a trip is whole rounds of a quad");
  if (n > k.list_cap_f) {  // overflowed: the quad's first lane walks the cells
    walk_cells(k, fstart, cc, [&](int j) {
      const V4<T> q = fpos[j];
      const T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
      if (r2 > T(0) && r2 <= k.r2max) pair(0, load(j), true);
    });
    return;
  }
  for (int s = 0; s < n; s += NB) {
    int j[NB];
    Rec d[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) j[u] = list[(long)min(s + u, n - 1) * cap + i];
#pragma unroll
    for (int u = 0; u < NB; ++u) d[u] = load(j[u]);
#pragma unroll
    for (int u = 0; u < NB; ++u) pair(u % kQuad, d[u], s + u < n);
  }
}

// The walk of an object in cell order around p, taking the candidates in range
// (r^2 <= r2max).
template <class T, class Load, class Term>
__device__ __forceinline__ void walk_quad(const KP<T>& k, const int* __restrict__ cstart,
                                          const V4<T>* __restrict__ pos, const V4<T>& p,
                                          WalkLds& lds, Load&& load, Term&& term) {
  int cc[3];
  node_encode(k, p.x, p.y, p.z, cc);
  walk_quad_cells<false>(
      k, cc, lds, [&](int lo, int hi, bool*) { return make_int2(cstart[lo], cstart[hi + 1]); },
      [&](int s) { return Cand<T>{pos[s], s}; },
      [&](const Cand<T>& d, bool* apart) {
        const T r2 = s_r2(p.x - d.q.x, p.y - d.q.y, p.z - d.q.z);
        *apart = r2 > T(0);
        return r2 <= k.r2max;
      },
      load, term);
}

}  // namespace tsph
