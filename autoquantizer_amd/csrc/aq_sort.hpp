// Sort of the particles by grid block of their stencil base (device code,
// included by aq_sort.hip and aq_group.hip).
//
// Inside a block the particles go in layers over its 64 cells (stencil
// bases): layer r holds the r-th particle of every cell that has more than
// r, in cell order, so that the 64 lanes of a wavefront of the tiled kernels
// mostly hold particles of distinct cells (their P2G atomics and G2P reads
// then hit distinct LDS slots; in particle order within a cell, ~8 lanes
// would share each slot).
//
// Five launches (four when at most kScanInline blocks):
//   keys     per particle: its cell, and its rank in the cell from a counter
//            per cell; marks the blocks that have particles
//   counts   particles per block from the cell counters of marked blocks, and
//            the layers' tables
//   scan     block offsets, work items, gather list
//   scatter  particles to their place in the workspace's copy
//   finish   ids (and the planes, unless the caller reads the copy) back,
//            cell counters and marks cleared for the next sort
// Counting per cell alone spreads the atomics over 64 counters a block: with
// a counter per block as well, particles in random order serialise on it
// (80,000 particles in 100 blocks: 78 us for the keys of the first sort).
#pragma once
#include "aq_sim.hpp"

// Blocks that one workgroup counts and scans by itself (one launch less: 3
// us); four times as many take it 20 us, two launches 6.
constexpr int kScanInline = 64;
// Layers of a block with a table entry (particles of a cell); particles of
// later layers add the block's cell counts up themselves.
constexpr int kLayers = 32;
// Entries of `part` (64 blocks each) under one entry of `top`.  Every
// workgroup of the scan adds up what lies before it: without the second
// level, reads grow with the square of the blocks (16 (m / 256)^2 bytes).
// Sorts (with the copy of a state before each) of 100,000 particles on 256^3
// nodes: 52 us without, 50 so; of 1,000,000 on 512^3: 328 and 274; of 100,000
// on 800^3: 1384 and 561 (759 with a scan in three launches).  Grids of up to
// 64 kTop blocks have one entry, which nobody reads: they leave it alone.
constexpr int kTop = 256;

// What the sort reads and writes, apart from the positions.
struct SortBuf {
  int64_t n, cap;
  int32_t m, nb, planes;     // grid blocks, blocks per axis, planes of the state
  uint32_t *key, *rank;      // [n] cell (block * 64 + cell), rank in the cell
  uint32_t *cells, *marks;   // [64 m] particles per cell, [m] block has particles: zero between sorts
  uint32_t *counts, *off;    // [m], [m + 1]
  // per block and layer r (marked blocks): the cells that hold more than r
  // particles, and the particles of the layers before
  unsigned long long *lmask; // [kLayers m]
  uint32_t *lpre;            // [kLayers m]
  uint32_t *part;            // [2 ceil(m / 64)] particles and items per 64 blocks
  uint32_t *top;             // [2 ceil(m / (64 kTop))] and per kTop entries of part: zero between sorts
  int32_t *item_off;         // [m + 1]
  int4 *items;
  uint32_t *near, *bm, *gcnt, *listed;
  const uint32_t *act;
  int32_t *glist;
  void *state, *tmp;         // planes, and the workspace's copy
  int32_t *ids, *tmp_ids;    // ids: null when not tracked
};

// Work items of a block with c particles.
__device__ __forceinline__ uint32_t items_of(uint32_t c) { return (c + (uint32_t)kItem - 1u) / (uint32_t)kItem; }

// Cell and rank of particle p of the thread (row: the thread's LDS row).
template <int DIM, int ST, int NW32, class T>
__device__ __forceinline__ void sort_key(const StateK &s, const CodecK &cod, const ParamsT<T> &P, const SortBuf &b,
                                         int64_t p, uint32_t *row) {
  if (p >= b.n) return;
  T x[DIM];
  if constexpr (ST == AQ_STORE_QUANT) {
    const uint64_t *w = (const uint64_t *)s.ptr;
#pragma unroll
    for (int i = 0; i < NW32 / 2; ++i) {
      if (i < s.nw && ((s.x_mask >> i) & 1u)) {
        const uint64_t z = w[(int64_t)i * s.cap + p];
        row[2 * i] = (uint32_t)z;
        row[2 * i + 1] = (uint32_t)(z >> 32);
      }
    }
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      if constexpr (IsF64<T>::value)
        x[a] = decode_row_f64(row, comp_at(cod, a), cod.cd + 4 * a);  // f64 compute
      else
        x[a] = (T)decode_row(row, comp_at(cod, a));
    }
  } else {
    const T *vals = (const T *)s.ptr;
#pragma unroll
    for (int a = 0; a < DIM; ++a) x[a] = vals[(int64_t)a * s.cap + p];
  }
  int base[3] = {0, 0, 0};
  T fx, w3[3];
#pragma unroll
  for (int a = 0; a < DIM; ++a) base[a] = stencil_1d<T>(x[a], P, fx, w3);
  constexpr int E = BlockShape<DIM>::E, LG = BlockShape<DIM>::LOG;
  const uint32_t k = (uint32_t)block_of_base<DIM>(base, P.nb);
  const uint32_t cell = DIM == 3 ? (uint32_t)(((base[0] & (E - 1)) << (2 * LG)) | ((base[1] & (E - 1)) << LG) |
                                              (base[2] & (E - 1)))
                                 : (uint32_t)(((base[0] & (E - 1)) << LG) | (base[1] & (E - 1)));
  const uint32_t id = k * 64u + cell;
  b.key[p] = id;
  b.rank[p] = atomicAdd(b.cells + id, 1u);
  if (b.marks[k] == 0u) b.marks[k] = 1u;  // every writer stores the same value
}

// Particles of the 64 blocks [64 g, 64 g + 64): wavefront w of the
// workgroup's 16 sums the cells of 4 of them, one lane per cell, and the
// totals go to part.  (The layer loops of a wavefront's blocks run one after
// the other: with 16 blocks a wavefront the kernel took 14 us for a million
// 3D particles, with 4 it takes 6.)
constexpr int kCountThreads = 1024;
__device__ __forceinline__ void sort_counts(const SortBuf &b, int32_t g, uint32_t (&tot)[kCountThreads / 64][2]) {
  constexpr int NB = 4, NW = kCountThreads / 64;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int32_t base = g * 64 + wave * NB;
  const uint32_t mk = lane < NB && base + lane < b.m ? b.marks[base + lane] : 0u;
  const unsigned long long set = __ballot(mk != 0u);
  int v[NB];
  // unmarked blocks read the first one's cells (a cached line) instead of
  // branching, so that all loads are in flight together
  const uint32_t *cells = b.cells + (int64_t)base * 64 + lane;
  if (set != 0ull) {
#pragma unroll
    for (int k = 0; k < NB; ++k) v[k] = (int)cells[(set >> k) & 1ull ? k * 64 : 0];
  }
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    v[k] = (set >> k) & 1ull ? v[k] : 0;
    if ((set >> k) & 1ull) {
      unsigned long long mine = 0ull;
      uint32_t pre = 0u, acc = 0u;
      for (uint32_t r = 0; r < (uint32_t)kLayers; ++r) {
        const unsigned long long more = __ballot(v[k] > (int)r);
        if (lane == (int)r) {
          mine = more;
          pre = acc;
        }
        if (more == 0ull) break;
        acc += (uint32_t)__popcll(more);
      }
      if (lane < kLayers) {
        b.lmask[(int64_t)(base + k) * kLayers + lane] = mine;
        b.lpre[(int64_t)(base + k) * kLayers + lane] = pre;
      }
    }
  }
  const uint32_t c = (uint32_t)LaneFold<NB>::fold(v, lane, [](int x, int y) { return x + y; });
  const int32_t mine = base + (lane >> 4);  // the block of the lane's sum
  const bool own = (lane & 15) == 0 && mine < b.m;
  if (own) b.counts[mine] = c;
  uint32_t a = own ? c : 0u, i = own ? items_of(c) : 0u;
  for (int o = 32; o > 0; o >>= 1) {
    a += (uint32_t)__shfl_xor((int)a, o);
    i += (uint32_t)__shfl_xor((int)i, o);
  }
  if (lane == 0) {
    tot[wave][0] = a;
    tot[wave][1] = i;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int t = threadIdx.x;
    uint32_t z = 0u;
#pragma unroll
    for (int w = 0; w < NW; ++w) z += tot[w][t];
    b.part[2 * g + t] = z;
    if (z != 0u && b.m > 64 * kTop) atomicAdd(b.top + 2 * (g / kTop) + t, z);
  }
  if (g == 0 && threadIdx.x < 16) b.gcnt[threadIdx.x] = 0u;  // the gather list's counters, for the scan
}

// Blocks [256 g, 256 g + 256), one per thread: their offsets (the totals
// before them, added up again by every workgroup), work items, near
// flags, cleared drift-margin masks and gather list entries.
// near[b]: some block within one block of b (per axis) holds particles, so
// the gather of b may find tiles.  Gather list: every block with particles
// within one block (near) or a grid left from before (act), once (listed
// marks them), at slots from gcnt[0].
// Threads from 256 on take no part.
template <int DIM>
__device__ __forceinline__ void sort_scan(const SortBuf &b, int32_t g, uint32_t (&sh)[4][2]) {
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int32_t blk = t < 256 ? g * 256 + t : b.m;
  const uint32_t c = blk < b.m ? b.counts[blk] : 0u, ic = items_of(c);
  uint32_t pa = 0u, pi = 0u;
  const int32_t g0 = 4 * g / kTop;  // entries of top before this workgroup's blocks, then of part
  for (int32_t i = t; t < 256 && i < g0; i += 256) {
    pa += b.top[2 * i];
    pi += b.top[2 * i + 1];
  }
  for (int32_t i = g0 * kTop + t; t < 256 && i < 4 * g; i += 256) {
    pa += b.part[2 * i];
    pi += b.part[2 * i + 1];
  }
  // wavefront: inclusive scan of the counts, sums of the chunks before
  uint32_t sa = c, si = ic;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t ya = (uint32_t)__shfl_up((int)sa, o), yi = (uint32_t)__shfl_up((int)si, o);
    if (lane >= o) {
      sa += ya;
      si += yi;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    pa += (uint32_t)__shfl_xor((int)pa, o);
    pi += (uint32_t)__shfl_xor((int)pi, o);
  }
  if (lane == 63 && wave < 4) {
    sh[wave][0] = sa;
    sh[wave][1] = si;
  }
  __shared__ uint32_t pre[4][2];
  if (lane == 0 && wave < 4) {
    pre[wave][0] = pa;
    pre[wave][1] = pi;
  }
  __syncthreads();
  uint32_t oa = sa - c, oi = si - ic;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    oa += pre[w][0];
    oi += pre[w][1];
    if (w < wave) {
      oa += sh[w][0];
      oi += sh[w][1];
    }
  }
  if (blk < b.m) {
    b.off[blk] = oa;
    b.item_off[blk] = (int32_t)oi;
    if (blk == b.m - 1) {
      b.off[b.m] = oa + c;
      b.item_off[b.m] = (int32_t)(oi + ic);
    }
    int bc[3];
    block_coords<DIM>(blk, b.nb, bc);
    for (uint32_t j = 0; j < ic; ++j) {
      const uint32_t left = c - j * (uint32_t)kItem;
      b.items[oi + j] = make_int4(blk, (int)(oa + j * (uint32_t)kItem), (int)(left < (uint32_t)kItem ? left : (uint32_t)kItem),
                                   pack_coords<DIM>(bc));
    }
  }
  bool in = false;
  if (blk < b.m) {
    b.bm[blk] = 0u;
    b.bm[b.m + blk] = 0u;
    int bc[3];
    block_coords<DIM>(blk, b.nb, bc);
    uint32_t any = 0u;
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx)
#pragma unroll
      for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
        for (int dz = (DIM == 3 ? -1 : 0); dz <= (DIM == 3 ? 1 : 0); ++dz) {
          const int x = bc[0] + dx, y = bc[1] + dy, z = bc[2] + dz;
          const bool ok = x >= 0 && x < b.nb && y >= 0 && y < b.nb && (DIM == 2 || (z >= 0 && z < b.nb));
          const int32_t q = DIM == 3 ? (x * b.nb + y) * b.nb + z : x * b.nb + y;
          any |= ok ? b.counts[q] : 0u;
        }
    b.near[blk] = any != 0u ? 1u : 0u;
    in = any != 0u || b.act[blk] != 0u;
    b.listed[blk] = in ? 1u : 0u;
  }
  const unsigned long long mask = __ballot(in);
  if (mask != 0ull) {
    const int leader = __ffsll((long long)mask) - 1;
    uint32_t at = 0u;
    if (lane == leader) at = atomicAdd(&b.gcnt[0], (uint32_t)__popcll(mask));
    at = (uint32_t)__shfl((int)at, leader);
    if (in) b.glist[at + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = blk;
  }
}

// Particle p to its place: position in the block, layer by layer,
// sum_c min(count_c, r) + #{c < cell : count_c > r}.
template <class E> __device__ __forceinline__ void sort_scatter(const SortBuf &b, int64_t p) {
  if (p >= b.n) return;
  const uint32_t id = b.key[p], r = b.rank[p], cell = id & 63u, blk = id >> 6;
  uint32_t pos;
  if (r < (uint32_t)kLayers) {
    const unsigned long long below = b.lmask[(int64_t)blk * kLayers + r] & ((1ull << cell) - 1ull);
    pos = b.lpre[(int64_t)blk * kLayers + r] + (uint32_t)__popcll(below);
  } else {
    const uint32_t *cc = b.cells + (int64_t)blk * 64;
    pos = 0u;
    for (uint32_t i = 0; i < 64u; ++i) {
      const uint32_t c = cc[i];
      pos += (c < r ? c : r) + (i < cell && c > r ? 1u : 0u);
    }
  }
  const int64_t q = (int64_t)b.off[blk] + pos;
  const E *src = (const E *)b.state;
  E *dst = (E *)b.tmp;
  int i = 0;
  for (; i + 4 <= b.planes; i += 4) {  // four loads in flight
    E v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[(int64_t)(i + k) * b.cap + p];
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[(int64_t)(i + k) * b.cap + q] = v[k];
  }
  for (; i < b.planes; ++i) dst[(int64_t)i * b.cap + q] = src[(int64_t)i * b.cap + p];
  if (b.ids) b.tmp_ids[q] = b.ids[p];
}

// Workgroup g of the finish: ids (and, with COPY, the planes) of particles
// [256 g, 256 g + 256) back from the copy; the cell counters and marks of
// blocks [64 g, 64 g + 64) and their top entry cleared; the list's append
// cursor set.
template <class E, bool COPY> __device__ __forceinline__ void sort_finish(const SortBuf &b, int32_t g) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t p = (int64_t)g * 256 + threadIdx.x;
  if (p < b.n) {
    if (b.ids) b.ids[p] = b.tmp_ids[p];
    if constexpr (COPY)
      for (int i = 0; i < b.planes; ++i) ((E *)b.state)[(int64_t)i * b.cap + p] = ((const E *)b.tmp)[(int64_t)i * b.cap + p];
  }
  const int32_t base = g * 64 + wave * 16;
  if (base < b.m) {
    const bool has = lane < 16 && base + lane < b.m && b.marks[base + lane] != 0u;
    const unsigned long long set = __ballot(has);
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if ((set >> k) & 1ull) b.cells[(int64_t)(base + k) * 64 + lane] = 0u;
    if (has) b.marks[base + lane] = 0u;
    if (b.m > 64 * kTop && g % kTop == 0 && threadIdx.x < 2) b.top[2 * (g / kTop) + threadIdx.x] = 0u;
  }
  if (g == 0 && threadIdx.x == 0) b.gcnt[3] = b.gcnt[0];
}
