// LDS-tiled fused G2P/P2G kernel over work items (gfx950), shared by the
// library build and the run-time specialisation of the kernel to one record
// layout (aq_sim_specialize).
#pragma once

#include "aq_mpm_kernels.hpp"

namespace aq {

// ---- LDS-tiled kernels over work items ---------------------------------------
// A work item is up to kItem particles whose stencil base was in one grid block
// at the last aq_sort: int4 (block, first particle, count, block coordinates
// packed by pack_coords).  The item's
// tile covers the block, the 2-node stencil reach and a 1-cell drift margin
// on each side: TE = E + 4 nodes per axis from block_origin - 1 (LDS layout
// in Tile; in the tile buffer, TE^DIM nodes grouped by the grid block they
// belong to, Tile::store_pos).
//
// G2P reads grid velocities staged in LDS.  P2G accumulates in LDS in fixed
// point (integer LDS atomics, exact and so independent of the order): per
// item and component the contributions are scaled by 2^k, with
// 2^(BITS-k) above the item's summed contribution bound, so the integer sums
// cannot overflow and are exact sums of the terms rounded to 2^-BITS of that
// bound (BITS = 30 in int32 for f32 compute, 62 in int64 for f64).  The
// finished tile goes to the item's slot of the tile buffer with plain stores;
// the gather kernel sums the tiles covering each node in a fixed order.  A
// particle whose stencil leaves the tile (it drifted more than a cell since
// the sort), or an item with a non-finite bound, reads grid_v and scatters
// into grid_f.
// Particles per work item = threads of a tiled workgroup (4 wavefronts).
// 512 (8 wavefronts) halves the tiles and made the gather 7.5 µs faster on
// the 3D fluid benchmark, but the fused kernel 6-18 µs slower (fewer
// workgroups between barriers).
constexpr int kItem = 256;

template <int DIM> struct Tile {
  static constexpr int E = BlockShape<DIM>::E, LG = BlockShape<DIM>::LOG;
  static constexpr int TE = E + 4;                                // nodes per axis
  static constexpr int TN = DIM == 3 ? TE * TE * TE : TE * TE;    // nodes
  static constexpr int STRIDE = TN;                               // nodes per item in the tile buffer
  // LDS slot of tile node (x, y, z): x SX + y SY + z.  SX = 112 = 48 mod 64,
  // SY = 12 (3D) / SX = 72 = 8 mod 64 (2D): the nodes of any 4x4x4 (8x8)
  // window get 64 distinct banks, and stencil offsets are immediate offsets.
  static constexpr int SY = DIM == 3 ? 12 : 1;
  static constexpr int SX = DIM == 3 ? 112 : 72;
  static constexpr int TS = TE * SX;                              // LDS slots (< 1024)
  __host__ __device__ static constexpr int slot(int x, int y, int z) {
    return DIM == 3 ? x * SX + y * SY + z : x * SX + y;
  }
  // slot(rel) for 0 <= rel < TE: full-rate 24-bit products
  __device__ static int first_slot(const int (&rel)[3]) {
    return DIM == 3 ? (int)(__umul24(rel[0], SX) + __umul24(rel[1], SY)) + rel[2] : (int)__umul24(rel[0], SX) + rel[1];
  }
  // Position of tile node (x, y, z) in the tile buffer.  Per axis the tile
  // covers the last node of the previous block (t = 0), the E nodes of its
  // own block (1..E) and the first 3 of the next (E+1..E+3); the buffer
  // groups the nodes by the block they belong to (3^DIM groups, in group
  // order) and stores each group row-major, which is the gathering
  // wavefront's lane order: a wavefront reads each covering tile as one
  // contiguous run.
  __host__ __device__ static constexpr int store_pos(int x, int y, int z) {
    int g[3] = {0, 0, 0}, u[3] = {0, 0, 0}, sz[3] = {0, 0, 0};
    const int t[3] = {x, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      g[a] = t[a] == 0 ? 0 : (t[a] <= E ? 1 : 2);
      u[a] = t[a] == 0 ? 0 : (t[a] <= E ? t[a] - 1 : t[a] - E - 1);
      sz[a] = g[a] == 0 ? 1 : (g[a] == 1 ? E : 3);
    }
    // nodes of the groups before (g0, g1, g2): the slab below g0, the rows
    // of slab g0 below g1, the groups of row (g0, g1) below g2
    const int cum[3] = {0, 1, E + 1};  // nodes per axis before group g
    if constexpr (DIM == 3) {
      const int before = cum[g[0]] * TE * TE + sz[0] * cum[g[1]] * TE + sz[0] * sz[1] * cum[g[2]];
      return before + (u[0] * sz[1] + u[1]) * sz[2] + u[2];
    } else {
      const int before = cum[g[0]] * TE + sz[0] * cum[g[1]];
      return before + u[0] * sz[1] + u[1];
    }
  }
};

// LDS slot of the node at each position of the tile buffer (the inverse of
// Tile::store_pos), built at compile time: the write-out walks the buffer
// in order, so each wavefront stores a contiguous run.
// Bit 15 marks the drift margin: nodes with t = 0 or TE - 1 on some axis,
// which only particles that left their sort cell reach.
constexpr uint16_t kMarginBit = 0x8000u;
// coord: the node's tile coordinates, 4 bits each.
template <int DIM> struct TileOrder {
  uint16_t slot[Tile<DIM>::TN];
  uint16_t coord[Tile<DIM>::TN];
};
template <int DIM> constexpr TileOrder<DIM> make_tile_order() {
  using TL = Tile<DIM>;
  TileOrder<DIM> o{};
  for (int x = 0; x < TL::TE; ++x)
    for (int y = 0; y < TL::TE; ++y)
      for (int z = 0; z < (DIM == 3 ? TL::TE : 1); ++z) {
        const bool margin = x == 0 || x == TL::TE - 1 || y == 0 || y == TL::TE - 1 ||
                            (DIM == 3 && (z == 0 || z == TL::TE - 1));
        o.slot[TL::store_pos(x, y, z)] = (uint16_t)(TL::slot(x, y, z) | (margin ? kMarginBit : 0u));
        o.coord[TL::store_pos(x, y, z)] = (uint16_t)(x | (y << 4) | (z << 8));
      }
  return o;
}
__constant__ constexpr TileOrder<3> kTileOrder3 = make_tile_order<3>();
__constant__ constexpr TileOrder<2> kTileOrder2 = make_tile_order<2>();
template <int DIM> __device__ __forceinline__ int tile_slot_at(int pos) {
  if constexpr (DIM == 3)
    return kTileOrder3.slot[pos];
  else
    return kTileOrder2.slot[pos];
}
template <int DIM> __device__ __forceinline__ int tile_coord_at(int pos) {
  if constexpr (DIM == 3)
    return kTileOrder3.coord[pos];
  else
    return kTileOrder2.coord[pos];
}

template <int DIM>
__device__ __forceinline__ void block_coords(int32_t b, int nb, int (&bc)[3]) {
  if constexpr (DIM == 3) {
    bc[0] = b / (nb * nb);
    bc[1] = (b / nb) % nb;
    bc[2] = b % nb;
  } else {
    bc[0] = b / nb;
    bc[1] = b % nb;
    bc[2] = 0;
  }
}

// Block coordinates in one word (the sort writes them into the work items: a
// scalar division chain per item otherwise).  At most 256 blocks per axis in
// 3D, 4096 in 2D.
template <int DIM> __device__ __forceinline__ int32_t pack_coords(const int (&bc)[3]) {
  return DIM == 3 ? bc[0] | (bc[1] << 10) | (bc[2] << 20) : bc[0] | (bc[1] << 16);
}
template <int DIM> __device__ __forceinline__ void unpack_coords(int32_t w, int (&bc)[3]) {
  if constexpr (DIM == 3) {
    bc[0] = w & 1023;
    bc[1] = (w >> 10) & 1023;
    bc[2] = (w >> 20) & 1023;
  } else {
    bc[0] = w & 0xFFFF;
    bc[1] = w >> 16;
    bc[2] = 0;
  }
}

template <int DIM>
__device__ __forceinline__ int64_t node_index(int i, int j, int k, int nb) {
  constexpr int LG = BlockShape<DIM>::LOG, E = BlockShape<DIM>::E;
  if constexpr (DIM == 3) {
    const int64_t blk = ((int64_t)(i >> LG) * nb + (j >> LG)) * nb + (k >> LG);
    return blk * 64 + (((i & (E - 1)) << 4) | ((j & (E - 1)) << 2) | (k & (E - 1)));
  } else {
    const int64_t blk = (int64_t)(i >> LG) * nb + (j >> LG);
    return blk * 64 + (((i & (E - 1)) << 3) | (j & (E - 1)));
  }
}

template <class T> __device__ __forceinline__ T tldexp(T x, int k);
template <> __device__ __forceinline__ float tldexp<float>(float x, int k) { return ldexpf(x, k); }
template <> __device__ __forceinline__ double tldexp<double>(double x, int k) { return ldexp(x, k); }
template <class T> __device__ __forceinline__ int texp(T x);  // x = m 2^e, 0.5 <= |m| < 1
template <> __device__ __forceinline__ int texp<float>(float x) { int e; frexpf(x, &e); return e; }
template <> __device__ __forceinline__ int texp<double>(double x) { int e; frexp(x, &e); return e; }

// Fixed-point accumulator of the P2G tile.
template <class T> struct AccOf;
template <> struct AccOf<float> {
  using U = uint32_t;
  static constexpr int BITS = 30;
  // LDS planes: two int32 sums per 64-bit word, (m v_x, m) and (m v_y, m v_z)
  static constexpr int PLANES = 2;
  // floor(x + 1/2) as int32 (two's complement), |x| < 2^31
  __device__ static U fix(float x) {
    int32_t r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return (U)r;
  }
  __device__ static float unfix(U q, int k) { return ldexpf((float)(int32_t)q, -k); }
  // hi 2^32 + lo as a 64-bit integer (lo sign-extended).  A 64-bit sum of
  // such words is (sum hi) 2^32 + (sum lo) exactly, so as long as both sums
  // fit in int32 (the per-item scales keep them below 2^31) unpack recovers
  // them: one 64-bit LDS atomic does the work of two 32-bit ones.
  __device__ static unsigned long long pack(float hi, float lo) {
    // in 32 bits: a 64-bit sum of the shifted words takes an operation more
    const U l = fix(lo), h = fix(hi) + (U)((int32_t)l >> 31);
    return ((unsigned long long)h << 32) | (unsigned long long)l;
  }
  // the same word when lo >= 0 (a mass: non-negative weight times a positive
  // particle mass), without the sign carry: two VALU instructions fewer per node
  __device__ static unsigned long long pack_nonneg_lo(float hi, float lo) {
    return ((unsigned long long)fix(hi) << 32) | (unsigned long long)fix(lo);
  }
  __device__ static void unpack(unsigned long long w, int32_t &hi, int32_t &lo) {
    lo = (int32_t)(uint32_t)w;
    hi = (int32_t)(uint32_t)((w - (unsigned long long)(long long)lo) >> 32);
  }
};
template <> struct AccOf<double> {
  using U = unsigned long long;
  static constexpr int BITS = 62;
  static constexpr int PLANES = 4;  // one int64 sum per component
  // rint(x) as int64, |x| < 2^62: hi = rint(x 2^-32) and then rint of the
  // exact rest x - hi 2^32 appear in the low bits of sums with 1.5 2^52 (a
  // tie of the rest goes to even as x's does, hi 2^32 being even).  Four f64
  // operations and two integer ones; half of those that conversions and a
  // separate sign take.
  __device__ static U fix(double x) {
    constexpr double M = 6755399441055744.0;  // bits 0x4338000000000000
    const double t = fma(x, 2.3283064365386962890625e-10, M);
    const double r = fma(t - M, -4294967296.0, x) + M;
    U hi, lo;
    __builtin_memcpy(&hi, &t, 8);
    __builtin_memcpy(&lo, &r, 8);
    const uint32_t h = (uint32_t)hi + ((uint32_t)(lo >> 32) - 0x43380000u);
    return (U)h << 32 | (U)(uint32_t)lo;
  }
  __device__ static double unfix(U q, int k) {
    const double d = (double)(int32_t)((long long)q >> 32) * 4294967296.0 + (double)(uint32_t)q;
    return ldexp(d, -k);
  }
};

// Wavefronts per SIMD that the tiled kernels' registers are kept for: 4
// (<= 128 VGPRs: the fused kernels of f32 storage need 68 to 114, of records
// with a run-time layout of up to 16 words 83 to 135) except for 3D elastic
// records with a run-time layout (161 to 168; held to 128, the kernel spills
// thousands of times) and f64 storage (102 to 202).  VGPRs spilled: 4 (3D
// elastic, 16 words) and, grouped, 11 and 4 (3D fluid, 4 and 8 words) and 9
// (3D elastic, 16 words).
template <int ST, int DIM, int MAT> struct TiledWaves {
  static constexpr int W = ST == AQ_STORE_F64 ? 2 : (ST == AQ_STORE_QUANT && DIM == 3 && MAT == AQ_ELASTIC ? 3 : 4);
};

// Tile origin (in cells) of an item.
template <int DIM>
__device__ __forceinline__ void tile_origin(const int4 &item, int (&o)[3]) {
  int bc[3];
  unpack_coords<DIM>(item.w, bc);
#pragma unroll
  for (int a = 0; a < 3; ++a) o[a] = a < DIM ? bc[a] * Tile<DIM>::E - 1 : 0;
}

// A thread's share of every tile, the same nodes for every item: their LDS
// slots and their offsets in a node buffer from the first node of the item's
// block, found once per workgroup (and grid size), so that staging a node is
// a test, a load and an LDS store.  Blocks outside the grid hold zeros: the
// item's block lies at some faces of the grid, a node in a neighbour block
// across some of its own, and the two masks meet if that block is outside.
// The fused kernels are bound by VALU issue (a wavefront's f32 sum, product
// or move takes a SIMD 2.7 cycles, an fma 3.3, a shift, conversion, comparison
// or integer product 4.4 to 4.8: measured), so address arithmetic counts:
// with the bounds by LaneFold, 32 substeps of 1,048,576 particles of a 3D
// fluid (32-byte records) took 3.27 ms before and 3.13 ms with this.
template <int DIM> struct TileShare {
  using TL = Tile<DIM>;
  static constexpr int R = (TL::TN + kItem - 1) / kItem;  // nodes per thread
  int32_t nb;
  int32_t off[R];
  uint32_t node[R];  // at buffer position tid + r kItem: LDS slot | kMarginBit | faces crossed << 16
  __device__ __forceinline__ void init(int tid, int blocks_per_axis) {
    constexpr int E = TL::E;
    nb = blocks_per_axis;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int nd = tid + r * kItem < TL::TN ? tid + r * kItem : 0, at = tile_coord_at<DIM>(nd);
      int32_t blk = 0, loc = 0;
      uint32_t faces = 0u;
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        const int t = (at >> (4 * a)) & 15;
        blk = blk * nb + (t == 0 ? -1 : (t <= E ? 0 : 1));
        loc = loc * E + ((t + E - 1) & (E - 1));
        faces |= t == 0 ? 1u << (2 * a) : (t <= E ? 0u : 2u << (2 * a));
      }
      off[r] = blk * 64 + loc;
      node[r] = (uint32_t)tile_slot_at<DIM>(nd) | (faces << 16);
    }
  }
  // whether the thread's r-th node is in the drift margin, and its LDS slot
  __device__ __forceinline__ bool margin(int r) const { return (node[r] & kMarginBit) != 0u; }
  __device__ __forceinline__ int slot(int r) const { return (int)(node[r] & (kMarginBit - 1u)); }
  // stages the tile of `item` from the node buffer into lds
  template <class T>
  __device__ __forceinline__ void copy(const int4 &item, int tid, const vec4_t<T> *__restrict__ nodes,
                                       vec4_t<T> *lds) const {
    int bc[3];
    unpack_coords<DIM>(item.w, bc);
    uint32_t faces = 0u;  // scalar: bit 2a, bc[a] = 0; bit 2a + 1, bc[a] = nb - 1
#pragma unroll
    for (int a = 0; a < DIM; ++a)
      faces |= (uint32_t)(bc[a] - 1) >> 31 << (16 + 2 * a) | (uint32_t)(nb - 2 - bc[a]) >> 31 << (17 + 2 * a);
    const vec4_t<T> *from = nodes + (int64_t)item.x * 64;
    vec4_t<T> val[R];  // all loads before the first wait
#pragma unroll
    for (int r = 0; r < R; ++r) {
      val[r].x = val[r].y = val[r].z = val[r].w = (T)0;
      if (!(node[r] & faces) && (TL::TN % kItem == 0 || tid + r * kItem < TL::TN)) val[r] = from[off[r]];
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (TL::TN % kItem == 0 || tid + r * kItem < TL::TN) lds[slot(r)] = val[r];
  }
};

// Everything the tiled kernels need of one simulation.
template <class T> struct TiledArgs {
  StateK s;
  CodecK cod;
  ParamsT<T> P;
  int64_t n;
  const int4 *items;
  const vec4_t<T> *grid_v;
  vec4_t<T> *tiles;
  vec4_t<T> *grid_f;
  uint32_t *fflags;
  int32_t *flist;  // blocks newly flagged by untiled scatters (null: flags only)
  uint32_t *fcnt;
  // per grid block, bit i: the block's item i (bit 31: items 31 and later,
  // which always write it) wrote its tile's drift margin; null: every item
  // writes its whole tile (G2P without P2G: masks to clear, or null)
  uint32_t *bmargin;
  const int32_t *item_off;  // first item of each block (with bmargin)
  int32_t nblocks;
};

// Work of one simulation: its `count` items.
template <class T> struct OneSim {
  static constexpr bool kMany = false;
  TiledArgs<T> a;
  int count;
  __device__ __forceinline__ int total() const { return count; }
  __device__ __forceinline__ const TiledArgs<T> &args(int it, int &li) const {
    li = it;
    return a;
  }
  __device__ __forceinline__ uint32_t key_base(uint32_t kb) const { return kb; }
  __device__ __forceinline__ int blocks_per_axis() const { return a.P.nb; }
  __device__ __forceinline__ uint32_t *margin(const TiledArgs<T> &A) const { return A.bmargin; }
  __device__ __forceinline__ uint32_t *fcount(const TiledArgs<T> &A) const { return A.fcnt; }
};

// Work of a group of simulations: the items of all of them, numbered
// simulation after simulation (prefix[s] = items before simulation s,
// prefix[nsims] = all).  An item's simulation is found by binary search
// over the prefix; item numbers are uniform over a workgroup, so the search
// and the descriptor loads are scalar.  The descriptors' codec key is the
// seed's key; the dithering key of substep `step` is hash32(step ^ it), as
// for a single simulation.
template <class T> struct GroupSims {
  static constexpr bool kMany = true;
  const TiledArgs<T> *__restrict__ descs;
  const int32_t *__restrict__ prefix;
  int32_t nsims;
  uint32_t step;
  // the parity of the next list gather (TiledArgs holds parity 0's masks and
  // counter); masked: margins are tracked (G2P only: masks are cleared)
  int32_t parity;
  bool masked;
  __device__ __forceinline__ uint32_t *margin(const TiledArgs<T> &A) const {
    return masked ? A.bmargin + (int64_t)parity * A.nblocks : nullptr;
  }
  __device__ __forceinline__ uint32_t *fcount(const TiledArgs<T> &A) const { return A.fcnt + parity; }
  __device__ __forceinline__ uint32_t key_base(uint32_t seed_key) const { return hash32(step ^ seed_key); }
  __device__ __forceinline__ int total() const { return prefix[nsims]; }
  __device__ __forceinline__ const TiledArgs<T> &args(int it, int &li) const {
    int lo = 0, hi = nsims;  // prefix[lo] <= it < prefix[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (prefix[mid] <= it)
        lo = mid;
      else
        hi = mid;
    }
    li = it - prefix[lo];
    return descs[lo];
  }
};

// Values exchanged between lanes without LDS where the hardware can: in
// half_swap, x becomes (x of the lanes with bit O clear, y of those lanes)
// and y the same of the lanes with bit O set, in the order (bit clear, bit
// set); lane_xor reads lane ^ O.  All lanes take part.
template <int O> __device__ __forceinline__ void half_swap_word(uint32_t &x, uint32_t &y) {
  static_assert(O == 32 || O == 16, "");
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0];
    y = r[1];
  }
}
template <int O> __device__ __forceinline__ uint32_t lane_xor_word(uint32_t x) {
  static_assert(O == 8 || O == 4 || O == 2 || O == 1, "");
  if constexpr (O == 4) {
    return (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (O << 10) | 31);  // xor mask, 32 lanes
  } else {
    // DPP: rotation of a row of 16 by 8; quad permutations [2,3,0,1] and [1,0,3,2]
    constexpr int ctrl = O == 8 ? 0x128 : (O == 2 ? 0x4E : 0xB1);
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, 0xF, 0xF, true);
  }
}
template <int O, class E> __device__ __forceinline__ void half_swap(E &x, E &y) {
  constexpr int W = sizeof(E) / 4;
  uint32_t a[W], b[W];
  __builtin_memcpy(a, &x, sizeof(E));
  __builtin_memcpy(b, &y, sizeof(E));
#pragma unroll
  for (int i = 0; i < W; ++i) half_swap_word<O>(a[i], b[i]);
  __builtin_memcpy(&x, a, sizeof(E));
  __builtin_memcpy(&y, b, sizeof(E));
}
template <int O, class E> __device__ __forceinline__ E lane_xor(E x) {
  constexpr int W = sizeof(E) / 4;
  uint32_t a[W];
  __builtin_memcpy(a, &x, sizeof(E));
#pragma unroll
  for (int i = 0; i < W; ++i) a[i] = lane_xor_word<O>(a[i]);
  __builtin_memcpy(&x, a, sizeof(E));
  return x;
}

// Reduction over a wavefront of N values a lane (N a power of two up to 64),
// f commutative: halves of the values are exchanged across lane bit 32, 16,
// ..., so that a lane ends with one value's result (N + a few exchanges
// instead of 6 N).  Recursive, so that every register index is a constant.
template <int N> struct LaneFold {
  // the value whose result lane `lane` ends with
  template <int H = N / 2, int O = 32> __device__ static int value(int lane) {
    if constexpr (H >= 1)
      return ((lane & O) ? H : 0) + value<H / 2, O / 2>(lane);
    else
      return 0;
  }
  template <int H, int O, class E, class F> __device__ static void step(E (&v)[N], int lane, F &&f) {
    if constexpr (H >= 1) {
#pragma unroll
      for (int i = 0; i < H; ++i) {
        if constexpr (O >= 16) {
          half_swap<O>(v[i], v[i + H]);
          v[i] = f(v[i], v[i + H]);
        } else {
          const bool up = (lane & O) != 0;
          const E send = up ? v[i] : v[i + H], keep = up ? v[i + H] : v[i];
          v[i] = f(keep, lane_xor<O>(send));
        }
      }
      step<H / 2, O / 2>(v, lane, f);
    } else if constexpr (O >= 1) {  // lanes left with the same value
      if constexpr (O >= 16) {
        E other = v[0];
        half_swap<O>(v[0], other);
        v[0] = f(v[0], other);
      } else {
        v[0] = f(v[0], lane_xor<O>(v[0]));
      }
      step<0, O / 2>(v, lane, f);
    }
  }
  template <class E, class F> __device__ static E fold(E (&v)[N], int lane, F &&f) {
    step<N / 2, 32>(v, lane, f);
    return v[0];
  }
};

// Partial maxima of a range run, [kLimSlots][kLimRow]: per workgroup slot the
// largest value and the largest negated value of each component, in lines of
// its own.
constexpr int kLimSlots = 4096, kLimRow = 64;

// A workgroup walks its items (of one simulation, or of a group of them,
// `Src`); per item three barriers: the tile staged, the bounds of the
// fixed-point scales, the scatter complete.  (Loading the next item during
// the current item's scatter saves a barrier but holds ~20 more VGPRs: 2 %
// faster for the specialised quantized kernel with the particles of a block
// in random order, 1 % slower with the layered order; the fp32-storage
// kernel lost a wave per SIMD.)
// LIM (2D, plain storage): the new states' per-component limits are folded
// into the workgroup's slot of `lim` while the values are in registers (a
// kernel of its own: one launch and read more a substep; a range run of
// 65,536 particles took 42 us a substep with it and the reduction after it,
// 30 so).  In 3D the fold costs the kernel a wavefront per SIMD or spills
// (77 -> 105 us for 400,000 particles where the separate kernel takes 10).
template <int DIM, int MAT, int ST, int NW32, class T, bool DO_G2P, bool DO_P2G, bool LIM = false, class Src>
__device__ __forceinline__ void tiled_run(const Src &src, float *__restrict__ lim = nullptr) {
  using TL = Tile<DIM>;
  using ACC = AccOf<T>;
  using U = typename ACC::U;
  constexpr int TS = TL::TS, TN = TL::TN, TE = TL::TE, NC = Comps<DIM, MAT>::NC;
  __shared__ vec4_t<T> tv[DO_G2P ? TS : 1];
  constexpr int NP = ACC::PLANES;
  __shared__ unsigned long long ts[DO_P2G ? NP : 1][DO_P2G ? TS : 1];
  constexpr int NWAVES = kItem / 64;
  __shared__ T bpart[NWAVES][4];
  __shared__ uint32_t bdrift[NWAVES];
  __shared__ uint32_t rows[kItem * RowsOf<ST, NW32>::RS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  constexpr bool G2P_ONLY_LOAD = DO_G2P;  // G2P needs only the words of x and J/F
  uint32_t *row = rows + tid * RowsOf<ST, NW32>::RS;
  const int ni = src.total();
  // each XCD (blocks dealt round-robin to 8 XCDs) walks a contiguous item range
  const int xcd = (int)(blockIdx.x & 7u);
  const int per = (int)(gridDim.x >> 3);
  const int lo = (int)((int64_t)ni * xcd / 8), hi = (int)((int64_t)ni * (xcd + 1) / 8);
  int it = lo + (int)(blockIdx.x >> 3);
  if (it >= hi) return;  // uniform over the workgroup
  TileShare<DIM> share;
  if constexpr (!Src::kMany) share.init(tid, src.blocks_per_axis());
  else share.nb = 0;
  if constexpr (DO_P2G) {
    for (int q = tid; q < TS; q += kItem)
#pragma unroll
      for (int a = 0; a < NP; ++a) ts[a][q] = 0ull;  // cleared before the first barrier
  }
  constexpr int NLV = NC <= 16 ? 16 : 32;
  float lmax = -__builtin_inff(), lneg = -__builtin_inff();  // of the lane's component, over the items
  for (; it < hi; it += per) {
    int li;  // the item's number in its simulation
    const TiledArgs<T> &A = src.args(it, li);
    const StateK &s = A.s;
    CodecK cod = A.cod;
    cod.key_base = src.key_base(cod.key_base);
    const ParamsT<T> &P = A.P;
    const int64_t n = A.n;
    const vec4_t<T> *__restrict__ grid_v = A.grid_v;
    vec4_t<T> *__restrict__ grid_f = A.grid_f;
    uint32_t *__restrict__ fflags = A.fflags;
#ifdef AQ_JIT_LAYOUT
    constexpr uint32_t g2p_mask = jit::kG2PMask;
#else
    const uint32_t g2p_mask = s.g2p_mask;
#endif
    const uint32_t load_mask = DO_G2P ? g2p_mask : 0xFFFFFFFFu;
    const int4 item = A.items[li];
    if constexpr (!DO_P2G) {
      // the last kernel of a run: the masks that its P2G set are cleared for
      // the parity the next run starts with
      if (src.margin(A) && tid == 0) src.margin(A)[item.x] = 0u;
    }
    int o[3];
    tile_origin<DIM>(item, o);
    // the particle's loads go out before the tile's, so their latencies overlap
    Fetched<ST, NW32> fw;
    T v[NC];
    if (tid < item.z && (int64_t)item.y + tid < n)
      fetch_state<DIM, ST, NW32, NC, T, G2P_ONLY_LOAD>(s, (int64_t)item.y + tid, load_mask, fw, v);
    if constexpr (Src::kMany)
      if (share.nb != P.nb) share.init(tid, P.nb);
    if constexpr (DO_G2P) share.template copy<T>(item, tid, grid_v, tv);
    __syncthreads();  // tile staged; the previous item's tile written out
    const bool has = tid < item.z && (int64_t)item.y + tid < n;
    const int64_t p = (int64_t)item.y + tid;
    T out[NC];
    if (has) {
      if constexpr (DO_G2P) {
        finish_state<DIM, ST, NW32, NC, T, true>(s, cod, g2p_mask, fw, row, v);
        const Stencil<DIM, T> S = stencil_of<DIM, MAT, T>(v, P);
        int rel[3] = {0, 0, 0};
        bool inside = true;
#pragma unroll
        for (int a = 0; a < DIM; ++a) {
          rel[a] = S.base[a] - o[a];
          inside = inside && rel[a] >= 0 && rel[a] + 2 < TE;
        }
        if (inside) {
          g2p_apply<DIM, MAT, T>(
              v, P, S, [&, q = TL::first_slot(rel)](int i, int j, int k) { return tv[q + TL::slot(i, j, k)]; }, out);
        } else {
          g2p_particle<DIM, MAT, T>(v, P, grid_v, out);
        }
        store_state<ST, NW32, NC, T>(s, cod, p, out, row);  // out: what storage now holds
      } else {
        finish_state<DIM, ST, NW32, NC, T>(s, cod, 0xFFFFFFFFu, fw, row, v);
#pragma unroll
        for (int c = 0; c < NC; ++c) out[c] = v[c];
      }
    }
    if (LIM && __ballot(has) != 0ull) {
      const auto larger = [](float a, float b) { return fmaxf(a, b); };
      float lv[NLV];
#pragma unroll
      for (int c = 0; c < NLV; ++c)  // NaN counts for nothing, as in fmaxf
        lv[c] = c < NC && has ? fmaxf(-__builtin_inff(), (float)out[c < NC ? c : 0]) : -__builtin_inff();
      lmax = fmaxf(lmax, LaneFold<NLV>::fold(lv, lane, larger));
#pragma unroll
      for (int c = 0; c < NLV; ++c)
        lv[c] = c < NC && has ? fmaxf(-__builtin_inff(), -(float)out[c < NC ? c : 0]) : -__builtin_inff();
      lneg = fmaxf(lneg, LaneFold<NLV>::fold(lv, lane, larger));
    }
    Stencil<DIM, T> S;
    P2GTerms<DIM, T> R;
    int rel[3] = {0, 0, 0};
    bool inside = false;
    if constexpr (DO_P2G) {
      T B[4] = {(T)0, (T)0, (T)0, (T)0};
      bool drift = false;  // the stencil reaches the tile's drift margin
      if (has) {
        S = stencil_of<DIM, MAT, T>(out, P);
        R = p2g_terms<DIM, MAT, T>(out, P, S);
        inside = true;
#pragma unroll
        for (int a = 0; a < DIM; ++a) {
          rel[a] = S.base[a] - o[a];
          // fx outside [0.5, 1.5] (a base clamped at the domain edge) can make
          // a weight negative, and the packed mass sums need them >= 0: such a
          // particle scatters through the float-atomic path
          inside = inside && rel[a] >= 0 && rel[a] + 2 < TE && S.fx[a] >= (T)0.5 && S.fx[a] <= (T)1.5;
          drift = drift || rel[a] == 0 || rel[a] == TE - 3;
        }
        if (inside) p2g_bounds<DIM, T>(R, S, B);
        drift = drift && inside;
      }
      const T bsum = LaneFold<4>::fold(B, lane, [](T a, T b) { return a + b; });
      const bool wdrift = __ballot(drift) != 0ull;
      if ((lane & 15) == 0) bpart[wave][LaneFold<4>::value(lane)] = bsum;
      if (lane == 0) bdrift[wave] = wdrift ? 1u : 0u;
    }
    __syncthreads();  // item bounds complete; G2P done with the tile
    int k[4] = {0, 0, 0, 0};
    bool margin = true;  // the write-out covers the drift margin
    if constexpr (DO_P2G) {
      if (uint32_t *bm = src.margin(A)) {
        uint32_t d = 0u;
#pragma unroll
        for (int w = 0; w < NWAVES; ++w) d |= bdrift[w];
        const int ib = li - A.item_off[item.x];  // the item's number in its block
        margin = d != 0u || ib >= 31;
        if (margin && tid == 0) atomicOr(bm + item.x, 1u << (ib < 31 ? ib : 31));
      }
      bool finite = true;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        T sum = bpart[0][c];
#pragma unroll
        for (int w = 1; w < NWAVES; ++w) sum += bpart[w][c];
        finite = finite && sum <= (T)1.0e37;
        k[c] = ACC::BITS - texp<T>(sum * ((T)1 + (T)1 / (T)1024));
      }
      if (has) {
        if (inside && finite) {
#pragma unroll
          for (int a = 0; a < DIM; ++a) {
            R.c[a] = tldexp<T>(R.c[a], k[a]);
#pragma unroll
            for (int b = 0; b < DIM; ++b) R.A[a][b] = tldexp<T>(R.A[a][b], k[a]);
          }
          R.pm = tldexp<T>(R.pm, k[3]);
          const int q0 = TL::first_slot(rel);
          p2g_emit<DIM, T>(R, S, [&](int i, int j, int kk, const T (&mom)[3], T m) {
            const int q = q0 + TL::slot(i, j, kk);
            if constexpr (NP == 2) {
              atomicAdd(&ts[0][q], ACC::pack_nonneg_lo(mom[0], m));
              atomicAdd(&ts[1][q], ACC::pack(mom[1], DIM == 3 ? mom[2] : (T)0));
            } else {
#pragma unroll
              for (int a = 0; a < DIM; ++a) atomicAdd(&ts[a][q], (unsigned long long)ACC::fix(mom[a]));
              atomicAdd(&ts[3][q], (unsigned long long)ACC::fix(m));
            }
          });
        } else {
          // from the terms, so that the state is not held over the barrier
          p2g_scatter<DIM, T>(R, S, P, grid_f, FlagSink{fflags, A.flist, src.fcount(A)});
        }
      }
    }
    if constexpr (DO_P2G) {
      __syncthreads();  // tile sums complete
      vec4_t<T> *dst = A.tiles + (int64_t)li * TN;
#pragma unroll
      for (int r = 0; r < TileShare<DIM>::R; ++r) {
        const int nd = tid + r * kItem;  // position in the buffer
        if (nd >= TN) continue;
        // without drift the margin's LDS sums are zero (never added to, so
        // they need no clearing either) and the gather does not read them
        if (!margin && share.margin(r)) continue;
        const int q = share.slot(r);
        vec4_t<T> val;
        if constexpr (NP == 2) {
          int32_t mx, m, my, mz;
          ACC::unpack(ts[0][q], mx, m);
          ACC::unpack(ts[1][q], my, mz);
          val.x = ACC::unfix((U)mx, k[0]);
          val.y = ACC::unfix((U)my, k[1]);
          val.z = DIM == 3 ? ACC::unfix((U)mz, k[2]) : (T)0;
          val.w = ACC::unfix((U)m, k[3]);
        } else {
          val.x = ACC::unfix(ts[0][q], k[0]);
          val.y = ACC::unfix(ts[1][q], k[1]);
          val.z = DIM == 3 ? ACC::unfix(ts[2][q], k[2]) : (T)0;
          val.w = ACC::unfix(ts[3][q], k[3]);
        }
        dst[nd] = val;
#pragma unroll
        for (int a = 0; a < NP; ++a) ts[a][q] = 0ull;
      }
    }
  }
  if constexpr (LIM) {
    __shared__ float lred[NWAVES][2 * NLV];
    const int lc = LaneFold<NLV>::value(lane);  // the lanes of a component store the same maximum
    lred[wave][lc] = lmax;
    lred[wave][NLV + lc] = lneg;
    __syncthreads();
    if (tid < 2 * NC) {
      float a = lim[(int64_t)blockIdx.x * kLimRow + tid];
#pragma unroll
      for (int w = 0; w < NWAVES; ++w) a = fmaxf(a, lred[w][tid < NC ? tid : NLV + tid - NC]);
      lim[(int64_t)blockIdx.x * kLimRow + tid] = a;
    }
  }
}

// One simulation's items (the count is the last sort's, read on the device).
template <int DIM, int MAT, int ST, int NW32, class T, bool DO_G2P, bool DO_P2G, bool LIM = false>
__device__ __forceinline__ void tiled_body(StateK s, CodecK cod, ParamsT<T> P, int64_t n,
                                           const int4 *__restrict__ items, const int32_t *__restrict__ nitems,
                                           const vec4_t<T> *__restrict__ grid_v, vec4_t<T> *__restrict__ tiles,
                                           vec4_t<T> *__restrict__ grid_f, uint32_t *__restrict__ fflags,
                                           int32_t *flist, uint32_t *gcnt, uint32_t ctl, uint32_t *bmargin,
                                           float *lim = nullptr) {
  // commit of the last list gather's appends (no thread of this kernel
  // reads gcnt[0] or the cleared counter; appends go to the other one)
  const uint32_t commit = (ctl >> 2) & 3u;
  if (commit && blockIdx.x == 0 && threadIdx.x == 0) {
    gcnt[0] = gcnt[3];
    gcnt[commit] = 0u;
  }
  uint32_t *fcnt = flist ? gcnt + (ctl & 3u) : nullptr;
  const int32_t nblocks = DIM == 3 ? P.nb * P.nb * P.nb : P.nb * P.nb;
  const OneSim<T> src{{s, cod, P, n, items, grid_v, tiles, grid_f, fflags, flist, fcnt, bmargin, nitems - nblocks, nblocks},
                      *nitems};
  tiled_run<DIM, MAT, ST, NW32, T, DO_G2P, DO_P2G, LIM>(src, lim);
}

template <int DIM, int MAT, int ST, int NW32, class T, bool DO_G2P, bool DO_P2G>
__global__ void __launch_bounds__(kItem) __attribute__((amdgpu_waves_per_eu(TiledWaves<ST, DIM, MAT>::W)))
k_tiled(StateK s, CodecK cod, ParamsT<T> P, int64_t n, const int4 *__restrict__ items,
        const int32_t *__restrict__ nitems, const vec4_t<T> *__restrict__ grid_v, vec4_t<T> *__restrict__ tiles,
        vec4_t<T> *__restrict__ grid_f, uint32_t *__restrict__ fflags, int32_t *flist, uint32_t *gcnt,
        uint32_t ctl, uint32_t *bmargin) {
  tiled_body<DIM, MAT, ST, NW32, T, DO_G2P, DO_P2G>(s, cod, P, n, items, nitems, grid_v, tiles, grid_f, fflags,
                                                    flist, gcnt, ctl, bmargin);
}

// The tiled G2P (-> P2G) of a 2D range run on plain storage: limits folded in.
template <int MAT, int ST, class T, bool DO_P2G>
__global__ void __launch_bounds__(kItem)
k_tiled_limits(StateK s, CodecK cod, ParamsT<T> P, int64_t n, const int4 *__restrict__ items,
               const int32_t *__restrict__ nitems, const vec4_t<T> *__restrict__ grid_v, vec4_t<T> *__restrict__ tiles,
               vec4_t<T> *__restrict__ grid_f, uint32_t *__restrict__ fflags, int32_t *flist, uint32_t *gcnt,
               uint32_t ctl, uint32_t *bmargin, float *__restrict__ lim) {
  tiled_body<2, MAT, ST, 4, T, true, DO_P2G, true>(s, cod, P, n, items, nitems, grid_v, tiles, grid_f, fflags, flist,
                                                     gcnt, ctl, bmargin, lim);
}

// P2G, fused G2P -> P2G or G2P of a group of quantized simulations (one
// dimension and material, any record layouts) in one launch.  commit: the
// counter slot that the last list gather consumed (0: none), cleared for
// every simulation while its appends join its list (tiled_body).
template <int DIM, int MAT, int NW32, bool DO_G2P, bool DO_P2G>
__global__ void __launch_bounds__(kItem) __attribute__((amdgpu_waves_per_eu(TiledWaves<AQ_STORE_QUANT, DIM, MAT>::W)))
k_tiled_group(const TiledArgs<float> *__restrict__ descs, const int32_t *__restrict__ prefix, int32_t nsims,
              uint32_t step, int32_t parity, int32_t masked, uint32_t commit) {
  if (commit && blockIdx.x == 0)
    for (int i = threadIdx.x; i < nsims; i += kItem) {
      uint32_t *gcnt = descs[i].fcnt - 1;
      gcnt[0] = gcnt[3];
      gcnt[commit] = 0u;
    }
  const GroupSims<float> src{descs, prefix, nsims, step, parity, masked != 0};
  tiled_run<DIM, MAT, AQ_STORE_QUANT, NW32, float, DO_G2P, DO_P2G>(src);
}

}  // namespace aq
