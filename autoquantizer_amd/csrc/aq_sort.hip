// libaqmpm: the sort by grid block (aq_sort) and its launches.
#include "aq_sort.hpp"

template <int DIM, int ST, int NW32, class T>
__global__ void __launch_bounds__(256) k_sort_keys(StateK s, CodecK cod, ParamsT<T> P, SortBuf b) {
  __shared__ uint32_t rows[256 * RowsOf<ST, NW32>::RS];
  sort_key<DIM, ST, NW32, T>(s, cod, P, b, (int64_t)blockIdx.x * 256 + threadIdx.x,
                             rows + threadIdx.x * RowsOf<ST, NW32>::RS);
}

__global__ void __launch_bounds__(kCountThreads) k_sort_counts(SortBuf b) {
  __shared__ uint32_t tot[kCountThreads / 64][2];
  sort_counts(b, (int32_t)blockIdx.x, tot);
}

template <int DIM> __global__ void __launch_bounds__(256) k_sort_scan(SortBuf b) {
  __shared__ uint32_t sh[4][2];
  sort_scan<DIM>(b, (int32_t)blockIdx.x, sh);
}

// One workgroup for all blocks, counting them first.
template <int DIM> __global__ void __launch_bounds__(kCountThreads) k_sort_count_scan(SortBuf b) {
  __shared__ uint32_t tot[kCountThreads / 64][2], sh[4][2];
  sort_counts(b, 0, tot);
  __syncthreads();  // counts visible
  sort_scan<DIM>(b, 0, sh);
}

template <class E> __global__ void __launch_bounds__(256) k_sort_scatter(SortBuf b) {
  sort_scatter<E>(b, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

template <class E, bool COPY> __global__ void __launch_bounds__(256) k_sort_finish(SortBuf b) {
  sort_finish<E, COPY>(b, (int32_t)blockIdx.x);
}

SortBuf sort_buf(const aq_sim *s, void *state, int64_t n, int32_t *ids) {
  SortBuf b;
  b.n = n;
  b.cap = s->d.capacity;
  b.m = s->nblocks;
  b.nb = s->pf.nb;
  b.planes = s->d.storage == AQ_STORE_QUANT ? s->d.nwords : s->d.ncomp;
  b.key = s->skey;
  b.rank = s->srank;
  b.cells = s->ccount;
  b.marks = s->marks;
  b.counts = s->scount;
  b.off = s->soff;
  b.part = s->spart;
  b.top = s->stop;
  b.lmask = s->lmask;
  b.lpre = s->lpre;
  b.item_off = s->item_off;
  b.items = s->items;
  b.near = s->near;
  b.bm = s->bmargin;
  b.gcnt = s->gcnt;
  b.listed = s->listed;
  b.act = s->act;
  b.glist = s->glist;
  b.state = state;
  b.tmp = s->tmp_state;
  b.ids = ids;
  b.tmp_ids = s->tmp_ids;
  return b;
}

unsigned sort_finish_blocks(const SortBuf &b) {
  const int64_t p = (b.n + 255) / 256, m = (b.m + 63) / 64;
  return (unsigned)(p > m ? p : m);
}

int sort_begin(aq_sim *s, hipStream_t st) {
  int rc;
  if (s->sort_open) {
    if ((rc = fill_u32(s->ccount, 0u, s->nodes, st))) return rc;
    if ((rc = fill_u32(s->marks, 0u, s->nblocks, st))) return rc;
    if ((rc = fill_u32(s->stop, 0u, 2 * (((int64_t)s->nblocks + 64 * kTop - 1) / (64 * kTop)), st))) return rc;
  }
  s->sort_open = true;
  s->have_items = false;
  return AQ_OK;
}

void sort_end(aq_sim *s, const void *state, int64_t n, const void *src) {
  s->sort_open = false;
  s->commit_pending = 0;
  s->list_parity = 0;
  s->have_items = true;
  s->items_state = state;
  s->items_n = n;
  s->src = src;
}

void drop_run(aq_sim *s, hipStream_t st) {
  if (s->src) {
    const size_t esz = s->d.storage == AQ_STORE_F32 ? 4 : 8;
    const size_t pitch = (size_t)s->d.capacity * esz;
    const size_t planes = (size_t)(s->d.storage == AQ_STORE_QUANT ? s->d.nwords : s->d.ncomp);
    (void)hipMemcpy2DAsync((void *)s->items_state, pitch, s->src, pitch, (size_t)s->items_n * esz, planes,
                           hipMemcpyDeviceToDevice, st);
    s->src = nullptr;
  }
  s->have_items = false;
  s->commit_pending = 0;  // of lists that the next sort makes anew
  s->list_parity = 0;
  (void)hipGetLastError();  // the run's error is reported by its caller, once
}

// Every launch is checked before the next: the scatter indexes with what the
// kernels before it wrote.
int launch_sort(aq_sim *s, void *state, int64_t n, int32_t *ids, bool defer, hipStream_t st) {
  if (n == 0) return AQ_OK;
  const int rc = sort_begin(s, st);
  if (rc) return rc;
  const StateK sk = make_state(s, state, nullptr);
  const CodecK cod = make_codec(s, 0u);
  const SortBuf b = sort_buf(s, state, n, ids);
  dispatch(s, [&](auto tag_) {
    TAG_TYPES(tag_)
    (void)MAT;
    hipLaunchKernelGGL((k_sort_keys<DIM, ST, NW32, T>), dim3(pblocks(n)), dim3(256), 0, st, sk, cod, params_of<T>(s),
                       b);
  });
  LAUNCH_CHECK();
  const bool d3 = s->d.dim == 3;
  if (b.m <= kScanInline) {
    if (d3)
      hipLaunchKernelGGL(k_sort_count_scan<3>, dim3(1), dim3(kCountThreads), 0, st, b);
    else
      hipLaunchKernelGGL(k_sort_count_scan<2>, dim3(1), dim3(kCountThreads), 0, st, b);
  } else {
    const unsigned g = (unsigned)((b.m + 255) / 256);
    hipLaunchKernelGGL(k_sort_counts, dim3((unsigned)((b.m + 63) / 64)), dim3(kCountThreads), 0, st, b);
    LAUNCH_CHECK();
    if (d3)
      hipLaunchKernelGGL(k_sort_scan<3>, dim3(g), dim3(256), 0, st, b);
    else
      hipLaunchKernelGGL(k_sort_scan<2>, dim3(g), dim3(256), 0, st, b);
  }
  LAUNCH_CHECK();
  const bool words = s->d.storage != AQ_STORE_F32;  // planes of 8 bytes
  if (words)
    hipLaunchKernelGGL(k_sort_scatter<uint64_t>, dim3(pblocks(n)), dim3(256), 0, st, b);
  else
    hipLaunchKernelGGL(k_sort_scatter<uint32_t>, dim3(pblocks(n)), dim3(256), 0, st, b);
  LAUNCH_CHECK();
  const unsigned f = sort_finish_blocks(b);
  if (defer)
    hipLaunchKernelGGL((k_sort_finish<uint32_t, false>), dim3(f), dim3(256), 0, st, b);
  else if (words)
    hipLaunchKernelGGL((k_sort_finish<uint64_t, true>), dim3(f), dim3(256), 0, st, b);
  else
    hipLaunchKernelGGL((k_sort_finish<uint32_t, true>), dim3(f), dim3(256), 0, st, b);
  LAUNCH_CHECK();
  sort_end(s, state, n, defer ? s->tmp_state : nullptr);
  return AQ_OK;
}

extern "C" int aq_sort(aq_sim *s, void *state, int64_t n, int32_t *ids, void *stream) {
  const int rc = check_n(s, state, n);
  if (rc) return rc;
  LAUNCH_CHECK();  // an error that was there before is reported with nothing launched
  return launch_sort(s, state, n, ids, false, (hipStream_t)stream);
}
