// libaqmpm: groups of quantized simulations advanced together (aq_group_*).
#include <memory>

#include "aq_sim.hpp"
#include "aq_gather.hpp"
#include "aq_sort.hpp"

// The kernels of a group number their work simulation after simulation: a
// prefix over the simulations' workgroups (host-known), and a workgroup finds
// its simulation by binary search (uniform, scalar loads).
__device__ __forceinline__ int32_t sim_of(const int32_t *__restrict__ prefix, int32_t nsims, int32_t g) {
  int32_t lo = 0, hi = nsims;  // prefix[lo] <= g < prefix[hi]
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (prefix[mid] <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// One simulation's list gather.
struct GroupGatherArgs {
  GatherArgs<float> g;
  int32_t *glist;
  const int32_t *flist;
  uint32_t *gcnt, *listed, *bmargin;
};

// The gather + grid update of a group of simulations in one launch, over
// their block lists (parity: of this gather, as in take_list).  Over every
// block of every domain instead, twelve simulations of a batched search
// (60,000 blocks, a tenth near particles) took 44 + 10 us.
template <int DIM>
__global__ void __launch_bounds__(256) k_gather_group(const GroupGatherArgs *__restrict__ descs,
                                                      const int32_t *__restrict__ prefix, int32_t nsims,
                                                      int32_t parity) {
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  const GroupGatherArgs &A = descs[s];
  const ColliderK none{};  // group members have no collider
  const ListArgs L{A.glist, A.flist, A.gcnt, A.listed, 1 + parity, A.bmargin + (int64_t)parity * A.g.nblocks,
                   A.bmargin + (int64_t)(1 - parity) * A.g.nblocks};
  gather_list<DIM, float>((uint32_t)((int32_t)blockIdx.x - prefix[s]), (uint32_t)(prefix[s + 1] - prefix[s]), A.g.P,
                          EmitGrid<DIM, float, true>{A.g.P, none, A.g.grid_v}, L, A.g.item_off, A.g.near, A.g.tiles,
                          A.g.grid_f, A.g.fflags, A.g.grid_v, A.g.act);
}

// ---- sorts of a group -------------------------------------------------------
// The sort's kernels over all simulations (aq_sort.hpp): for twelve
// simulations 9 launches instead of 60.
struct GroupSortArgs {
  StateK s;
  CodecK cod;
  ParamsT<float> P;
  SortBuf b;
};

template <int DIM, int NW32>
__global__ void __launch_bounds__(256) k_group_keys(const GroupSortArgs *__restrict__ descs,
                                                    const int32_t *__restrict__ prefix, int32_t nsims) {
  __shared__ uint32_t rows[256 * RowsOf<AQ_STORE_QUANT, NW32>::RS];
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  const GroupSortArgs &A = descs[s];
  sort_key<DIM, AQ_STORE_QUANT, NW32, float>(A.s, A.cod, A.P, A.b,
                                             (int64_t)((int32_t)blockIdx.x - prefix[s]) * 256 + threadIdx.x,
                                             rows + threadIdx.x * RowsOf<AQ_STORE_QUANT, NW32>::RS);
}

__global__ void __launch_bounds__(kCountThreads) k_group_counts(const GroupSortArgs *__restrict__ descs,
                                                                const int32_t *__restrict__ prefix, int32_t nsims) {
  __shared__ uint32_t tot[kCountThreads / 64][2];
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  sort_counts(descs[s].b, (int32_t)blockIdx.x - prefix[s], tot);
}

template <int DIM>
__global__ void __launch_bounds__(256) k_group_scan(const GroupSortArgs *__restrict__ descs,
                                                    const int32_t *__restrict__ prefix, int32_t nsims) {
  __shared__ uint32_t sh[4][2];
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  sort_scan<DIM>(descs[s].b, (int32_t)blockIdx.x - prefix[s], sh);
}

__global__ void __launch_bounds__(256) k_group_scatter(const GroupSortArgs *__restrict__ descs,
                                                       const int32_t *__restrict__ prefix, int32_t nsims) {
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  sort_scatter<uint64_t>(descs[s].b, (int64_t)((int32_t)blockIdx.x - prefix[s]) * 256 + threadIdx.x);
}

__global__ void __launch_bounds__(256) k_group_finish(const GroupSortArgs *__restrict__ descs,
                                                      const int32_t *__restrict__ prefix, int32_t nsims) {
  const int32_t s = sim_of(prefix, nsims, (int32_t)blockIdx.x);
  sort_finish<uint64_t, false>(descs[s].b, (int32_t)blockIdx.x - prefix[s]);
}

// prefix[s] = items of a class's simulations before s (item_off[nblocks] of
// each, written by its last sort), prefix[nsims] = all of them.  One
// workgroup of 256 per class.
constexpr int kMaxClasses = 2 * 2 * 4;  // dimension, material, record bucket
struct ItemPrefixArgs {
  const TiledArgs<float> *descs[kMaxClasses];
  int32_t *prefix[kMaxClasses];
  int32_t nsims[kMaxClasses];
};
__global__ void __launch_bounds__(256) k_group_prefix(ItemPrefixArgs C) {
  const TiledArgs<float> *__restrict__ descs = C.descs[blockIdx.x];
  int32_t *__restrict__ prefix = C.prefix[blockIdx.x];
  const int32_t nsims = C.nsims[blockIdx.x];
  __shared__ int32_t wsum[4];
  __shared__ int32_t carry;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nsims; base += 256) {
    const int i = base + tid;
    const int32_t v = i < nsims ? descs[i].item_off[descs[i].nblocks] : 0;
    int32_t x = v;  // inclusive scan over the wavefront
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int32_t off = carry;
    for (int w = 0; w < wave; ++w) off += wsum[w];
    if (i < nsims) prefix[i] = off + x - v;
    __syncthreads();  // every thread has read carry and wsum
    if (tid == 255) carry = off + x;
    __syncthreads();
  }
  if (tid == 0) prefix[nsims] = carry;
}

// Simulations of one tiled launch (same dimension, material and word bucket).
struct GroupClass {
  int dim, mat, bucket;
  int32_t nsims, sort0;        // members; their first entry in aq_group::sorts
  int64_t items_bound;         // sum over members of (n + kItem - 1) / kItem + nblocks
  TiledArgs<float> *descs;     // workspace: [nsims]
  TiledArgs<float> *descs_src; // workspace: [nsims], reading the copy a sort left in the workspace
  int32_t *prefix;             // workspace: [nsims + 1] items before each member
  int32_t *keys_prefix;        // workspace: [nsims + 1] workgroups of the sort's keys before each member
  int32_t keys_blocks;
};

// Simulations of one gather launch (same dimension).
struct GroupGather {
  int dim;
  int32_t nsims;
  GroupGatherArgs *descs;   // workspace: [nsims]
  int32_t *prefix;          // workspace: [nsims + 1] workgroups of the gather before each member
  int32_t blocks;
  GroupSortArgs *sorts;     // workspace: [nsims], the members' sort
  int32_t *scan_prefix;     // workspace: [nsims + 1] workgroups of the sort's scan
  int32_t scan_blocks;
};

struct aq_group {
  std::vector<aq_sim *> sims;
  std::vector<void *> states;
  std::vector<int64_t> ns;
  std::vector<int32_t *> ids;
  std::vector<GroupClass> classes;
  std::vector<GroupGather> gathers;
  // all members, class after class
  std::vector<int> order;
  GroupSortArgs *sorts;
  int32_t *counts_prefix, *scatter_prefix, *finish_prefix;
  int32_t counts_blocks, scatter_blocks, finish_blocks;
};

static int64_t group_ws_total(int nsims) {
  // per simulation: two TiledArgs, one GroupGatherArgs, two GroupSortArgs
  // (its class's and its gather's order) and seven prefix entries; per array
  // (at most 4 x 16 of the classes, 4 x 2 of the gathers, 4 of the group)
  // the closing entry and the 256-byte alignment
  const int64_t per = 2 * (int64_t)sizeof(TiledArgs<float>) + (int64_t)sizeof(GroupGatherArgs) +
                      2 * (int64_t)sizeof(GroupSortArgs) + 7 * 4;
  return align256((int64_t)nsims * per) + 80 * 512;
}

extern "C" int64_t aq_group_workspace_bytes(int nsims) {
  if (nsims < 1) return fail(AQ_ERR_INVALID, "a group needs a simulation");
  return group_ws_total(nsims);
}

static GroupGatherArgs gather_args(const aq_sim *s) {
  GroupGatherArgs q;
  GatherArgs<float> &a = q.g;
  a.P = s->pf;
  a.nblocks = s->nblocks;
  a.item_off = s->item_off;
  a.near = s->near;
  a.tiles = (const vec4_t<float> *)s->tiles;
  a.grid_f = (vec4_t<float> *)s->grid_f;
  a.fflags = s->fflags;
  a.grid_v = (vec4_t<float> *)s->grid_v;
  a.act = s->act;
  q.glist = s->glist;
  q.flist = s->flist;
  q.gcnt = s->gcnt;
  q.listed = s->listed;
  q.bmargin = s->bmargin;
  return q;
}

// Workgroups of a simulation's list gather: a wavefront for each block near
// particles, about three for every 256 of them, and a loop over longer lists.
static int32_t gather_groups(const aq_sim *s, int64_t n) {
  int64_t g = 3 * n / 1024 + 4;
  const int64_t all = (s->nblocks + 3) / 4;
  if (g > all) g = all;
  return (int32_t)(g < 2048 ? g : 2048);
}

extern "C" int aq_group_create(aq_sim *const *sims, void *const *states, const int64_t *ns, int32_t *const *ids,
                               int nsims, void *workspace, int64_t workspace_bytes, aq_group **out) {
  if (!out) return fail(AQ_ERR_INVALID, "null output");
  *out = nullptr;
  if (!sims || !states || !ns) return fail(AQ_ERR_INVALID, "null argument");
  if (nsims < 1) return fail(AQ_ERR_INVALID, "a group needs a simulation");
  if (!workspace) return fail(AQ_ERR_INVALID, "null workspace");
  if (((uintptr_t)workspace & 255u) != 0u) return fail(AQ_ERR_INVALID, "workspace must be 256-byte aligned");
  if (workspace_bytes < group_ws_total(nsims)) return fail(AQ_ERR_CAPACITY, "group workspace too small");
  for (int i = 0; i < nsims; ++i) {
    const aq_sim *s = sims[i];
    if (!s) return fail(AQ_ERR_INVALID, "null simulation handle");
    if (s->d.storage != AQ_STORE_QUANT) return fail(AQ_ERR_INVALID, "group members need quantized storage");
    if (s->d.compute_f64) return fail(AQ_ERR_INVALID, "group members compute in f32");
    if (s->has_collider) return fail(AQ_ERR_INVALID, "group members cannot have an SDF collider");
    if (ns[i] < 1 || ns[i] > s->d.capacity) return fail(AQ_ERR_CAPACITY, "particle count outside [1, capacity]");
    if (!states[i]) return fail(AQ_ERR_INVALID, "null state");
    for (int j = 0; j < i; ++j)
      if (sims[j] == s) return fail(AQ_ERR_INVALID, "a simulation appears twice in the group");
  }
  auto g = std::make_unique<aq_group>();
  g->sims.assign(sims, sims + nsims);
  g->states.assign(states, states + nsims);
  g->ns.assign(ns, ns + nsims);
  g->ids.assign(nsims, nullptr);
  if (ids) g->ids.assign(ids, ids + nsims);
  // classes, members in the caller's order
  std::vector<std::vector<int>> cmem, gmem;
  for (int i = 0; i < nsims; ++i) {
    const aq_sim *s = sims[i];
    const int b = nw32_bucket(s->d.nwords);
    int fc = -1;
    for (size_t c = 0; c < g->classes.size(); ++c)
      if (g->classes[c].dim == s->d.dim && g->classes[c].mat == s->d.material && g->classes[c].bucket == b) fc = (int)c;
    if (fc < 0) {
      GroupClass f{};
      f.dim = s->d.dim;
      f.mat = s->d.material;
      f.bucket = b;
      g->classes.push_back(f);
      cmem.emplace_back();
      fc = (int)g->classes.size() - 1;
    }
    cmem[fc].push_back(i);
    int gc = -1;
    for (size_t c = 0; c < g->gathers.size(); ++c)
      if (g->gathers[c].dim == s->d.dim) gc = (int)c;
    if (gc < 0) {
      GroupGather q{};
      q.dim = s->d.dim;
      g->gathers.push_back(q);
      gmem.emplace_back();
      gc = (int)g->gathers.size() - 1;
    }
    gmem[gc].push_back(i);
  }
  // workspace: descriptor and prefix arrays, each 256-aligned, filled on the
  // host and uploaded once
  std::vector<char> host((size_t)workspace_bytes, 0);
  int64_t off = 0;
  bool fits = true;
  auto take = [&](int64_t bytes) {
    const int64_t o = off;
    off = align256(off + bytes);
    fits = fits && off <= workspace_bytes;
    return fits ? o : 0;
  };
  auto put = [&](int64_t at, const void *src, size_t bytes) {
    if (fits) std::memcpy(host.data() + at, src, bytes);
  };
  // exclusive prefix of `count(i)` over the members, with the total at the end
  bool small = true;
  auto prefix_of = [&](const std::vector<int> &mem, auto &&count, int32_t **dev) {
    const int64_t at = take((int64_t)(mem.size() + 1) * 4);
    int64_t sum = 0;
    for (size_t k = 0; k <= mem.size(); ++k) {
      const int32_t v = (int32_t)sum;
      put(at + (int64_t)k * 4, &v, 4);
      if (k < mem.size()) sum += count(mem[k]);
      small = small && sum <= (int64_t)INT32_MAX / 2;
    }
    *dev = (int32_t *)((char *)workspace + at);
    return (int32_t)sum;
  };
  auto sort_args = [&](int i) {
    aq_sim *s = g->sims[i];
    GroupSortArgs a;
    a.s = make_state(s, g->states[i], g->ids[i]);
    a.cod = make_codec(s, 0u);
    a.P = s->pf;
    a.b = sort_buf(s, g->states[i], g->ns[i], g->ids[i]);
    return a;
  };
  const auto particles = [&](int i) { return (g->ns[i] + 255) / 256; };
  std::vector<int> &all = g->order;
  for (size_t c = 0; c < g->classes.size(); ++c) {
    GroupClass &f = g->classes[c];
    f.nsims = (int32_t)cmem[c].size();
    f.sort0 = (int32_t)all.size();
    all.insert(all.end(), cmem[c].begin(), cmem[c].end());
    const int64_t od = take((int64_t)f.nsims * (int64_t)sizeof(TiledArgs<float>));
    const int64_t os = take((int64_t)f.nsims * (int64_t)sizeof(TiledArgs<float>));
    f.descs = (TiledArgs<float> *)((char *)workspace + od);
    f.descs_src = (TiledArgs<float> *)((char *)workspace + os);
    f.prefix = (int32_t *)((char *)workspace + take((int64_t)(f.nsims + 1) * 4));
    f.keys_blocks = prefix_of(cmem[c], particles, &f.keys_prefix);
    f.items_bound = 0;
    for (int k = 0; k < f.nsims; ++k) {
      const int i = cmem[c][k];
      aq_sim *s = g->sims[i];
      TiledArgs<float> a;
      a.s = make_state(s, g->states[i], g->ids[i]);
      a.cod = make_codec(s, 0u);
      // the seed's key; the kernel derives each substep's key from it
      a.cod.key_base = host_hash32((uint32_t)s->d.seed ^ host_hash32((uint32_t)(s->d.seed >> 32)));
      a.P = s->pf;
      a.n = g->ns[i];
      a.items = s->items;
      a.grid_v = (const vec4_t<float> *)s->grid_v;
      a.tiles = (vec4_t<float> *)s->tiles;
      a.grid_f = (vec4_t<float> *)s->grid_f;
      a.fflags = s->fflags;
      a.flist = s->flist;
      a.fcnt = s->gcnt + 1;  // parity 0's counter and masks
      a.bmargin = s->bmargin;
      a.item_off = s->item_off;
      a.nblocks = s->nblocks;
      put(od + (int64_t)k * (int64_t)sizeof(a), &a, sizeof(a));
      a.s.src = s->tmp_state;
      put(os + (int64_t)k * (int64_t)sizeof(a), &a, sizeof(a));
      f.items_bound += (g->ns[i] + kItem - 1) / kItem + s->nblocks;
    }
  }
  const int64_t oall = take((int64_t)nsims * (int64_t)sizeof(GroupSortArgs));
  g->sorts = (GroupSortArgs *)((char *)workspace + oall);
  for (int k = 0; k < nsims; ++k) {
    const GroupSortArgs a = sort_args(all[k]);
    put(oall + (int64_t)k * (int64_t)sizeof(a), &a, sizeof(a));
  }
  g->counts_blocks = prefix_of(all, [&](int i) { return (int64_t)(g->sims[i]->nblocks + 63) / 64; }, &g->counts_prefix);
  g->scatter_blocks = prefix_of(all, particles, &g->scatter_prefix);
  g->finish_blocks = prefix_of(
      all, [&](int i) { return (int64_t)sort_finish_blocks(sort_buf(g->sims[i], g->states[i], g->ns[i], nullptr)); },
      &g->finish_prefix);
  for (size_t c = 0; c < g->gathers.size(); ++c) {
    GroupGather &q = g->gathers[c];
    q.nsims = (int32_t)gmem[c].size();
    const int64_t od = take((int64_t)q.nsims * (int64_t)sizeof(GroupGatherArgs));
    const int64_t os = take((int64_t)q.nsims * (int64_t)sizeof(GroupSortArgs));
    q.descs = (GroupGatherArgs *)((char *)workspace + od);
    q.sorts = (GroupSortArgs *)((char *)workspace + os);
    for (int k = 0; k < q.nsims; ++k) {
      const GroupGatherArgs a = gather_args(g->sims[gmem[c][k]]);
      put(od + (int64_t)k * (int64_t)sizeof(a), &a, sizeof(a));
      const GroupSortArgs b = sort_args(gmem[c][k]);
      put(os + (int64_t)k * (int64_t)sizeof(b), &b, sizeof(b));
    }
    q.blocks = prefix_of(gmem[c], [&](int i) { return (int64_t)gather_groups(g->sims[i], g->ns[i]); }, &q.prefix);
    q.scan_blocks = prefix_of(gmem[c], [&](int i) { return (int64_t)(g->sims[i]->nblocks + 255) / 256; },
                              &q.scan_prefix);
  }
  if (!fits) return fail(AQ_ERR_CAPACITY, "group workspace too small");
  if (!small) return fail(AQ_ERR_CAPACITY, "too many grid blocks in one group");
  HIP_TRY(hipMemcpy(workspace, host.data(), (size_t)off, hipMemcpyHostToDevice));
  *out = g.release();
  return AQ_OK;
}

extern "C" int aq_group_destroy(aq_group *g) {
  delete g;
  return AQ_OK;
}

template <class F>
static void dispatch_class(int dim, int mat, int bucket, F &&f) {
  if (dim == 3 && mat == AQ_FLUID) dispatch_quant<3, AQ_FLUID, float>(bucket, f);
  else if (dim == 3) dispatch_quant<3, AQ_ELASTIC, float>(bucket, f);
  else if (mat == AQ_FLUID) dispatch_quant<2, AQ_FLUID, float>(bucket, f);
  else dispatch_quant<2, AQ_ELASTIC, float>(bucket, f);
}

// Sorts every member; the sorted planes stay in the workspaces (descs_src).
static int group_sort(aq_group *g, hipStream_t st) {
  const int32_t n = (int32_t)g->sims.size();
  for (aq_sim *s : g->sims) {
    const int rc = sort_begin(s, st);
    if (rc) return rc;
  }
  for (const GroupClass &f : g->classes) {
    dispatch_class(f.dim, f.mat, f.bucket, [&](auto tag_) {
      TAG_TYPES(tag_)
      (void)MAT;
      (void)ST;
      hipLaunchKernelGGL((k_group_keys<DIM, NW32>), dim3(f.keys_blocks), dim3(256), 0, st,
                         (const GroupSortArgs *)(g->sorts + f.sort0), (const int32_t *)f.keys_prefix, f.nsims);
    });
    LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_group_counts, dim3(g->counts_blocks), dim3(kCountThreads), 0, st,
                     (const GroupSortArgs *)g->sorts, (const int32_t *)g->counts_prefix, n);
  LAUNCH_CHECK();
  for (const GroupGather &q : g->gathers) {
    if (q.dim == 3)
      hipLaunchKernelGGL(k_group_scan<3>, dim3(q.scan_blocks), dim3(256), 0, st, (const GroupSortArgs *)q.sorts,
                         (const int32_t *)q.scan_prefix, q.nsims);
    else
      hipLaunchKernelGGL(k_group_scan<2>, dim3(q.scan_blocks), dim3(256), 0, st, (const GroupSortArgs *)q.sorts,
                         (const int32_t *)q.scan_prefix, q.nsims);
    LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_group_scatter, dim3(g->scatter_blocks), dim3(256), 0, st, (const GroupSortArgs *)g->sorts,
                     (const int32_t *)g->scatter_prefix, n);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_group_finish, dim3(g->finish_blocks), dim3(256), 0, st, (const GroupSortArgs *)g->sorts,
                     (const int32_t *)g->finish_prefix, n);
  LAUNCH_CHECK();
  for (int32_t i = 0; i < n; ++i) sort_end(g->sims[i], g->states[i], g->ns[i], g->sims[i]->tmp_state);
  ItemPrefixArgs C{};
  for (size_t c = 0; c < g->classes.size(); ++c) {
    C.descs[c] = g->classes[c].descs;
    C.prefix[c] = g->classes[c].prefix;
    C.nsims[c] = g->classes[c].nsims;
  }
  hipLaunchKernelGGL(k_group_prefix, dim3((unsigned)g->classes.size()), dim3(256), 0, st, C);
  LAUNCH_CHECK();
  return AQ_OK;
}

static int group_gather(aq_group *g, int32_t parity, hipStream_t st) {
  for (const GroupGather &q : g->gathers) {
    if (q.dim == 3)
      hipLaunchKernelGGL(k_gather_group<3>, dim3(q.blocks), dim3(256), 0, st, (const GroupGatherArgs *)q.descs,
                         (const int32_t *)q.prefix, q.nsims, parity);
    else
      hipLaunchKernelGGL(k_gather_group<2>, dim3(q.blocks), dim3(256), 0, st, (const GroupGatherArgs *)q.descs,
                         (const int32_t *)q.prefix, q.nsims, parity);
  }
  LAUNCH_CHECK();
  return AQ_OK;
}

// One tiled launch per class.  parity: of the next list gather; masked, commit:
// as k_tiled_group takes them; src: reading the copies of a sort.
template <bool DO_G2P, bool DO_P2G>
static int group_tiled(aq_group *g, uint32_t step, int workgroups, bool src, int32_t parity, bool masked,
                       uint32_t commit, hipStream_t st) {
  for (const GroupClass &f : g->classes) {
    int64_t want = workgroups;
    if (want == 0) {
      want = f.items_bound + 64;
      if (want > 4096) want = 4096;
      want = (want + 7) / 8 * 8;
    }
    dispatch_class(f.dim, f.mat, f.bucket, [&](auto tag_) {
      TAG_TYPES(tag_)
      (void)ST;
      hipLaunchKernelGGL((k_tiled_group<DIM, MAT, NW32, DO_G2P, DO_P2G>), dim3((unsigned)want), dim3(kItem), 0, st,
                         (const TiledArgs<float> *)(src ? f.descs_src : f.descs), (const int32_t *)f.prefix, f.nsims,
                         step, parity, masked ? 1 : 0, commit);
    });
    LAUNCH_CHECK();
    if (DO_G2P)  // every particle of the class is written to its caller's planes
      for (int32_t k = 0; k < f.nsims; ++k) g->sims[g->order[f.sort0 + k]]->src = nullptr;
  }
  return AQ_OK;
}

static int group_run(aq_group *g, int nsteps, uint32_t step0, int sort_every, int workgroups, hipStream_t st) {
  int rc;
  if ((rc = group_sort(g, st))) return rc;
  bool src = true;     // the states are in the workspaces' copies
  int32_t parity = 0;  // of the next list gather
  uint32_t commit = 0; // counter slot of the last one, not yet committed
  if ((rc = group_tiled<false, true>(g, 0u, workgroups, src, parity, true, 0u, st))) return rc;
  if ((rc = group_gather(g, parity, st))) return rc;
  commit = 1u + (uint32_t)parity;
  parity ^= 1;
  for (int t = 0; t + 1 < nsteps; ++t) {
    if (t > 0 && t % sort_every == 0) {  // resets the lists' counters and the masks
      if ((rc = group_sort(g, st))) return rc;
      src = true;
      parity = 0;
      commit = 0u;
    }
    if ((rc = group_tiled<true, true>(g, step0 + (uint32_t)t, workgroups, src, parity, true, commit, st))) return rc;
    src = false;
    if ((rc = group_gather(g, parity, st))) return rc;
    commit = 1u + (uint32_t)parity;
    parity ^= 1;
  }
  // the last G2P commits, and clears parity 0's masks where they are the ones set
  return group_tiled<true, false>(g, step0 + (uint32_t)(nsteps - 1), workgroups, src, 0, parity == 1, commit, st);
}

extern "C" int aq_group_advance(aq_group *g, int nsteps, uint32_t step0, int sort_every, int workgroups,
                                void *stream) {
  if (!g) return fail(AQ_ERR_INVALID, "null handle");
  if (nsteps < 0) return fail(AQ_ERR_INVALID, "negative step count");
  if (sort_every < 1) return fail(AQ_ERR_INVALID, "a group sorts: sort_every must be positive");
  if (workgroups < 0 || workgroups > 8192 || workgroups % 8 != 0)
    return fail(AQ_ERR_INVALID, "workgroups must be a multiple of 8 in [0, 8192]");
  if (nsteps == 0) return AQ_OK;
  LAUNCH_CHECK();  // an error that was there before is reported with nothing launched
  const int rc = group_run(g, nsteps, step0, sort_every, workgroups, (hipStream_t)stream);
  // the lists are left as every call leaves them (settle_list), the items of the last sort describe the states
  if (rc)
    for (aq_sim *s : g->sims) drop_run(s, (hipStream_t)stream);
  return rc;
}
