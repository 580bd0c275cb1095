// Per-graph schedule of the fused EGNN/MPNN layer (integer work, bit-exact).
//
// The reference launches one program per CSR row (forward_kernel.py:47,
// test_mem.py:22), so a degree-4096 row serialises one program while the
// rest of the grid idles.  Here the edge stream is cut into fixed 32-edge
// tiles instead, independent of row boundaries:
//   erow[e]       row (destination) of CSR edge e -- lets a tile find its rows
//                 without a search over rowptr
//   fix_rows[]    rows that are empty or whose edges cross a tile boundary;
//                 their partial sums are combined by a fixed-order fix-up
//   csc_ptr/eid   the edges sorted by source (stable), for the deterministic
//                 source-side gradient sum of the backward pass
//   tile_tab[]    per 32-edge tile: the row runs (ranks) inside it, with the
//                 span and destination of each, for the per-tile row sums
// Built once per graph and cached by the caller.
#include <hipcub/hipcub.hpp>
#include "egnn_device.h"
#include "egnn_internal.h"

namespace egnn {

size_t sched_layout(int64_t N, int64_t E, void* base, SchedView* v) {
  char* b = (char*)base;
  size_t off = 0;
  auto take = [&](size_t bytes) { void* p = b ? b + off : nullptr; off = align_up(off + bytes); return p; };
  v->erow = (int32_t*)take(sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1));
  v->fix_rows = (int32_t*)take(sizeof(int32_t) * (size_t)N);
  v->n_fix = (int32_t*)take(sizeof(int32_t));
  v->csc_ptr = (int32_t*)take(sizeof(int32_t) * (size_t)(N + 1));
  v->csc_eid = (int32_t*)take(sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1));
  v->tile_tab = (int32_t*)take(sizeof(int32_t) * kTabInts * (size_t)std::max<int64_t>(cdiv(E, kTileEdges), 1));
  return off;
}

// Rows per block of the two scan launches, and the longest source list that the counting path sorts (one wave per
// list, kSortMax / 64 values per lane).
constexpr int kScanRows = 2048, kSortMax = 512;
// The counting path counts the edges per source by atomics, scatters one 4-byte id per edge and sorts each node's
// list in registers: 334 k edges 36 us in four launches against 120 us in 24 with the library's sort.  The scatter's
// cost grows with the spread of the sources, so the two cross between 0.9M and 2M edges by kind of graph; the line lies
// below all of them.  One schedule, counting / sort: chains with kNN edges 983k 120 / 213 us, 1.97M 173 / 174, 3.9M
// 278 / 257; random sources 1.28M 251 / 165, 2.56M 422 / 179; power law 0.87M 193 / 253, 1.40M 273 / 210.
constexpr int64_t kCountMaxEdges = int64_t(3) << 18;

// Atomics on one address follow each other, so a few hubs that hold most edges as sources would make the count the slowest
// part.  The launch that clears the counts looks at kHubSample edges, a run of kHubRun (one cache line) at a scattered place
// in each of kClear equal pieces, so that no row length fits the distance, and leaves the graph to the sort when so many of
// them share a source (of a hash, so rarely two) that its list is likely longer than kSortMax.  One schedule of 600k edges,
// without / with the check: 5 hubs 3,033 / 212 us, 20 hubs 1,631 / 216, one hub with 1 % of the edges 282 / 221; flat lists
// of 123k, 614k and 640k edges 71 / 70, 101 / 99 and 153 / 153.  (Single edges instead of runs, 4,096 lines read by one
// block, added 5 us to each.)
constexpr int kClear = 1024;   // threads of the launch
constexpr int kHubRun = 4, kHubSample = kClear * kHubRun, kHubHits = 6, kHubHash = 16384;
constexpr int32_t kNotCounted = 0x7fffffff;   // in place of the longest list

struct SchedTmp {
  int32_t* cnt;       // [N] edges per source, then each list's fill position
  int32_t* state;     // [2] CSR error, longest source list
  int32_t* bsum;      // [scan blocks][2] per block: edges, fix rows
  int32_t* keys_out;
  int32_t* vals_in;
  void* cub;
  size_t cub_bytes;
};

static int key_bits(int64_t N) {
  int b = 1;
  while ((int64_t(1) << b) < N) ++b;
  return b;
}

static size_t cub_bytes(int64_t N, int64_t E) {
  size_t a = 0;
  hipcub::DeviceRadixSort::SortPairs(nullptr, a, (const int32_t*)nullptr, (int32_t*)nullptr, (const int32_t*)nullptr,
                                     (int32_t*)nullptr, (int)std::max<int64_t>(E, 1), 0, key_bits(N));
  return a;
}

static size_t tmp_layout(int64_t N, int64_t E, void* base, SchedTmp* t) {
  char* b = (char*)base;
  size_t off = 0;
  auto take = [&](size_t bytes) { void* p = b ? b + off : nullptr; off = align_up(off + bytes); return p; };
  t->cnt = (int32_t*)take(sizeof(int32_t) * (size_t)(N + 2));
  t->state = t->cnt ? t->cnt + N : nullptr;
  t->bsum = (int32_t*)take(sizeof(int32_t) * 2 * (size_t)cdiv(N, kScanRows));
  t->keys_out = (int32_t*)take(sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1));
  t->vals_in = (int32_t*)take(sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1));
  t->cub_bytes = cub_bytes(N, E);
  t->cub = take(t->cub_bytes);
  return off;
}

size_t schedule_tmp_bytes(int64_t N, int64_t E) {
  SchedTmp t;
  return tmp_layout(N, E, nullptr, &t);
}

// clears cnt and state; block 0 looks for hubs (hubs != 0): state[1] = kNotCounted
__global__ __launch_bounds__(kClear) void clear_kernel(const int32_t* __restrict__ col, int64_t N, int64_t E,
                                                    int32_t* __restrict__ cnt, int32_t* __restrict__ state, int hubs) {
  __shared__ int32_t hits[kHubHash];
  for (int64_t q = blockIdx.x * (int64_t)kClear + threadIdx.x; q < N; q += (int64_t)gridDim.x * kClear) cnt[q] = 0;
  if (blockIdx.x > 0) return;
  int found = 0;
  if (hubs) {
    const int64_t lo = threadIdx.x * E / kClear, len = (threadIdx.x + 1) * E / kClear - lo;
    const int64_t at = lo + ((int64_t)((threadIdx.x * 2654435761u) >> 8) * len >> 24);
    const int32_t* p = col + min(at, E - kHubRun);   // E > kSortMax
    int32_t j[kHubRun];
#pragma unroll
    for (int k = 0; k < kHubRun; ++k) j[k] = p[k];
    for (int q = threadIdx.x; q < kHubHash; q += kClear) hits[q] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kHubRun; ++k) {
      const int64_t n = atomicAdd(&hits[((uint32_t)j[k] * 2654435761u) >> 18], 1) + 1;
      if (n >= kHubHits && n * E > (int64_t)kHubSample * kSortMax) found = 1;
    }
  }
  found = __syncthreads_or(found);
  if (threadIdx.x == 0) {
    state[0] = 0;
    state[1] = found ? kNotCounted : 0;
  }
}

// CSR checks and (cnt != null) the number of edges per source
__global__ void csr_count_kernel(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col, int64_t N,
                                 int64_t E, int32_t* __restrict__ cnt, int32_t* state) {
  int32_t* const err = state;
  if (state[1] == kNotCounted) cnt = nullptr;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int bad = 0;
  for (int64_t r = t0; r < N; r += stride) {
    int32_t a = rowptr[r], b = rowptr[r + 1];
    if (a > b || a < 0 || b > E) bad = 1;
    if (r == 0 && a != 0) bad = 1;
    if (r == N - 1 && b != E) bad = 1;
  }
  for (int64_t e = t0; e < E; e += stride) {
    int32_t j = col[e];
    if (j < 0 || j >= N) bad = 1;
    else if (cnt) atomicAdd(&cnt[j], 1);
  }
  if (bad) err[0] = 1;
}

// rows that are empty or cross a 32-edge tile
__device__ __forceinline__ int fix_row(const int32_t* rowptr, int64_t r) {
  const int32_t a = rowptr[r], b = rowptr[r + 1];
  return (a == b) || (a / kTileEdges != (b - 1) / kTileEdges);
}
// block sums (x, y) over its threads' pairs; valid in every thread
__device__ __forceinline__ int2 block_sum(int2 v, int2* red) {
  for (int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_xor(v.x, o, 64);
    v.y += __shfl_xor(v.y, o, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  int2 s = make_int2(0, 0);
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    s.x += red[w].x;
    s.y += red[w].y;
  }
  __syncthreads();
  return s;
}
// per block of kScanRows nodes: its edges by source and its fix rows; the longest source list
__global__ __launch_bounds__(256) void scan_sums_kernel(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ cnt,
                                                        int64_t N, int32_t* __restrict__ bsum, int32_t* longest) {
  __shared__ int2 red[4];
  const int64_t r0 = (int64_t)blockIdx.x * kScanRows;
  int2 v = make_int2(0, 0);
  int most = 0;
  for (int q = threadIdx.x; q < kScanRows && r0 + q < N; q += 256) {
    const int n = cnt[r0 + q];
    v.x += n;
    v.y += fix_row(rowptr, r0 + q);
    most = n > most ? n : most;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const int m = __shfl_xor(most, o, 64);
    most = m > most ? m : most;
  }
  if ((threadIdx.x & 63) == 0 && most > 0) atomicMax(longest, most);
  const int2 s = block_sum(v, red);
  if (threadIdx.x == 0) {
    bsum[2 * (int64_t)blockIdx.x] = s.x;
    bsum[2 * (int64_t)blockIdx.x + 1] = s.y;
  }
}
// many blocks: their sums as exclusive prefixes, by one block
__global__ __launch_bounds__(256) void scan_mid_kernel(int32_t* __restrict__ bsum, int64_t nb) {
  __shared__ int2 red[4];
  int2 run = make_int2(0, 0);
  for (int64_t b0 = 0; b0 < nb; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    const int2 v = b < nb ? make_int2(bsum[2 * b], bsum[2 * b + 1]) : make_int2(0, 0);
    int2 p = v;   // inclusive over the wave
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(p.x, o, 64), y = __shfl_up(p.y, o, 64);
      if ((int)(threadIdx.x & 63) >= o) { p.x += x; p.y += y; }
    }
    if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = p;
    __syncthreads();
    int2 base = run, tot = run;
    for (int w = 0; w < 4; ++w) {
      if (w < (int)(threadIdx.x >> 6)) { base.x += red[w].x; base.y += red[w].y; }
      tot.x += red[w].x; tot.y += red[w].y;
    }
    if (b < nb) { bsum[2 * b] = base.x + p.x - v.x; bsum[2 * b + 1] = base.y + p.y - v.y; }
    run = tot;
    __syncthreads();
  }
}
// csc_ptr (also as the lists' fill positions, over cnt) and the fix rows in ascending order.  prefix: bsum holds
// exclusive prefixes; else each block adds up the sums before its own.
__global__ __launch_bounds__(256) void scan_write_kernel(const int32_t* __restrict__ rowptr, int32_t* __restrict__ cnt,
                                                         int64_t N, int64_t E, const int32_t* __restrict__ bsum, int prefix,
                                                         int32_t* __restrict__ csc_ptr, int32_t* __restrict__ fix_rows,
                                                         int32_t* __restrict__ n_fix) {
  __shared__ int2 red[4];
  const int64_t nb = gridDim.x, bid = blockIdx.x;
  int2 run = make_int2(0, 0);
  if (prefix) {
    run = make_int2(bsum[2 * bid], bsum[2 * bid + 1]);
  } else {
    for (int64_t b = threadIdx.x; b < bid; b += 256) { run.x += bsum[2 * b]; run.y += bsum[2 * b + 1]; }
    run = block_sum(run, red);
  }
  constexpr int PER = kScanRows / 256;   // consecutive rows of a thread
  const int64_t r0 = bid * kScanRows + (int64_t)threadIdx.x * PER;
  int n[PER], f[PER];
  int2 v = make_int2(0, 0);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool in = r0 + k < N;
    n[k] = in ? cnt[r0 + k] : 0;
    f[k] = in ? fix_row(rowptr, r0 + k) : 0;
    v.x += n[k];
    v.y += f[k];
  }
  int2 p = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(p.x, o, 64), y = __shfl_up(p.y, o, 64);
    if ((int)(threadIdx.x & 63) >= o) { p.x += x; p.y += y; }
  }
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = p;
  __syncthreads();
  int2 at = make_int2(run.x + p.x - v.x, run.y + p.y - v.y);
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) { at.x += red[w].x; at.y += red[w].y; }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (r0 + k >= N) break;
    csc_ptr[r0 + k] = at.x;
    cnt[r0 + k] = at.x;
    if (f[k]) fix_rows[at.y] = (int32_t)(r0 + k);
    at.x += n[k];
    at.y += f[k];
    if (r0 + k == N - 1) {
      csc_ptr[N] = (int32_t)E;
      n_fix[0] = at.y;
    }
  }
}

__global__ void csc_fill_kernel(const int32_t* __restrict__ col, int64_t E, int32_t* __restrict__ pos,
                                int32_t* __restrict__ csc_eid) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < E; e += (int64_t)gridDim.x * blockDim.x)
    csc_eid[atomicAdd(&pos[col[e]], 1)] = (int32_t)e;
}
// Each source's edge ids in ascending order, one wave per list of at most 64 V ids: every id's rank is the number of
// smaller ones (distinct values), so the result does not depend on the order in which they were filled in.
template <int V>
__device__ __forceinline__ void sort_list(int32_t* p, int len, int l) {
  int v[V], rank[V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    v[c] = l + 64 * c < len ? p[l + 64 * c] : 0x7fffffff;
    rank[c] = 0;
  }
#pragma unroll
  for (int c = 0; c < V; ++c) {
    const int m = len - 64 * c < 64 ? len - 64 * c : 64;
    for (int k = 0; k < m; ++k) {
      const int x = __builtin_amdgcn_readlane(v[c], k);
#pragma unroll
      for (int q = 0; q < V; ++q) rank[q] += x < v[q];
    }
  }
#pragma unroll
  for (int c = 0; c < V; ++c)
    if (l + 64 * c < len) p[rank[c]] = v[c];
}
__global__ __launch_bounds__(256) void csc_sort_kernel(const int32_t* __restrict__ csc_ptr, int64_t N,
                                                       int32_t* __restrict__ csc_eid) {
  const int l = threadIdx.x & 63;
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); n < N; n += nw) {
    const int b = __builtin_amdgcn_readfirstlane(csc_ptr[n]), len = __builtin_amdgcn_readfirstlane(csc_ptr[n + 1]) - b;
    if (len <= 1) continue;
    if (len <= 64) sort_list<1>(csc_eid + b, len, l);
    else if (len <= 128) sort_list<2>(csc_eid + b, len, l);
    else if (len <= 256) sort_list<4>(csc_eid + b, len, l);
    else sort_list<kSortMax / 64>(csc_eid + b, len, l);
  }
}

// one block of 256 threads per `rows` (at most 256) rows: rowptr slice in LDS, edges of the
// slice assigned by a binary search over it
__global__ __launch_bounds__(256) void erow_kernel(const int32_t* __restrict__ rowptr, int64_t N, int rows,
                                                  int32_t* __restrict__ erow) {
  __shared__ int32_t rp[257];
  const int64_t r0 = (int64_t)blockIdx.x * rows;
  const int nr = (int)std::min<int64_t>(rows, N - r0);
  for (int t = threadIdx.x; t <= nr; t += blockDim.x) rp[t] = rowptr[r0 + t];
  __syncthreads();
  const int32_t e0 = rp[0], e1 = rp[nr];
  for (int32_t e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
    int lo = 0, hi = nr;  // largest r with rp[r] <= e
    while (hi - lo > 1) {
      int mid = (lo + hi) >> 1;
      if (rp[mid] <= e) lo = mid; else hi = mid;
    }
    erow[e] = (int32_t)(r0 + lo);
  }
}

// One wave per 32-edge tile t: lanes 0..33 hold the rows of edges 32 t - 1 .. 32 t + 32 (clamped);
// edge k of the tile starts a rank when k = 0 or its row differs from that of edge k - 1.  The lane
// that starts rank q sends its span and row to lane q, which writes entry q of the table.
__global__ __launch_bounds__(256) void tile_tab_kernel(const int32_t* __restrict__ erow, int64_t E, int64_t ntiles,
                                                       int32_t* __restrict__ tab) {
  const int l = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= ntiles) return;   // whole waves
  const int64_t base = t * kTileEdges;
  const int64_t e = base - 1 + l;
  const int row = erow[e < 0 ? 0 : (e >= E ? E - 1 : e)];
  const int nvalid = (int)(E - base < kTileEdges ? E - base : kTileEdges);
  const int rk = __shfl(row, l + 1 < 64 ? l + 1 : 63, 64), rprev = row;   // edge l and edge l - 1
  const bool starts = l < nvalid && (l == 0 || rk != rprev);
  const uint32_t mask = (uint32_t)(__ballot(starts) & 0xffffffffull);
  const int nrank = __popc(mask);
  const bool start_in = base == 0 || __shfl(row, 0, 64) != __shfl(row, 1, 64);
  const bool end_in = base + kTileEdges >= E || __shfl(row, 33, 64) != __shfl(row, 32, 64);
  // the lane that starts rank q: its span (first edge | count << 8) and row, sent to lane q
  int q = 63, span = 0;
  if (starts) {
    const uint32_t rest = l >= 31 ? 0u : (mask & ~((2u << l) - 1u));
    const int end = rest ? __ffs(rest) - 1 : nvalid;
    q = __popc(mask & ((2u << l) - 1u)) - 1;
    span = l | ((end - l) << 8);
  }
  const int rspan = __builtin_amdgcn_ds_permute(q * 4, span);
  const int rrow = __builtin_amdgcn_ds_permute(q * 4, rk);
  int32_t* tt = tab + t * kTabInts;
  if (l < kTileEdges) {
    const bool has = l < nrank;
    const bool whole = (l > 0 || start_in) && (l < nrank - 1 || end_in);
    tt[kTabTgt + l] = !has ? -3 : whole ? rrow : (l == 0 ? -1 : -2);
    reinterpret_cast<uint16_t*>(tt + kTabSpan)[l] = (uint16_t)(has ? rspan : 0);
  } else if (l == kTileEdges) {
    tt[kTabNrank] = nrank;
  } else if (l > kTileEdges && l < kTileEdges + 16) {
    tt[kTabNrank + l - kTileEdges] = 0;   // padding
  }
}

__global__ void iota_kernel(int32_t* __restrict__ v, int64_t E) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < E; e += (int64_t)gridDim.x * blockDim.x)
    v[e] = (int32_t)e;
}

// csc_ptr[n] = first position of key n in the sorted source list
__global__ void csc_ptr_kernel(const int32_t* __restrict__ keys, int64_t N, int64_t E, int32_t* __restrict__ ptr) {
  for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n <= N; n += (int64_t)gridDim.x * blockDim.x) {
    int64_t lo = 0, hi = E;
    while (lo < hi) {
      int64_t mid = (lo + hi) >> 1;
      if (keys[mid] < n) lo = mid + 1; else hi = mid;
    }
    ptr[n] = (int32_t)lo;
  }
}

int launch_schedule(const int32_t* rowptr, const int32_t* col, int64_t N, int64_t E, const SchedView& v, void* tmp,
                    size_t tmp_bytes, hipStream_t st) {
  SchedTmp t;
  if (tmp_layout(N, E, tmp, &t) > tmp_bytes) return EGNN_ERR_WORKSPACE;
  int vb = (int)std::min<int64_t>(cdiv(std::max(N, E), 256), 4096);
  bool count = E <= kCountMaxEdges;   // else the fix rows alone come from the scan (of zero counts)
  hipLaunchKernelGGL(clear_kernel, dim3((unsigned)std::min<int64_t>(cdiv(N, 2 * kClear), 512)), dim3(kClear), 0, st, col, N, E, t.cnt,
                     t.state, count && E > kSortMax ? 1 : 0);
  hipLaunchKernelGGL(csr_count_kernel, dim3(vb), dim3(256), 0, st, rowptr, col, N, E, count ? t.cnt : nullptr, t.state);
  const int64_t sb = cdiv(N, kScanRows);
  hipLaunchKernelGGL(scan_sums_kernel, dim3((unsigned)sb), dim3(256), 0, st, rowptr, t.cnt, N, t.bsum, t.state + 1);
  int32_t host[2] = {0, 0};   // error, longest source list
  if (hipMemcpyAsync(host, t.state, sizeof(host), hipMemcpyDeviceToHost, st) != hipSuccess) return EGNN_ERR_HIP;
  if (hipStreamSynchronize(st) != hipSuccess) return EGNN_ERR_HIP;
  if (host[0]) return EGNN_ERR_CSR;
  count = count && host[1] != kNotCounted;

  const bool mid = sb > 1024;
  if (mid) hipLaunchKernelGGL(scan_mid_kernel, dim3(1), dim3(256), 0, st, t.bsum, sb);
  hipLaunchKernelGGL(scan_write_kernel, dim3((unsigned)sb), dim3(256), 0, st, rowptr, t.cnt, N, E, t.bsum, mid ? 1 : 0,
                     v.csc_ptr, v.fix_rows, v.n_fix);
  if (E > 0) {
    const int rows = N <= 65536 ? 32 : 256;   // enough blocks for small graphs, few edges a block for none
    hipLaunchKernelGGL(erow_kernel, dim3((unsigned)cdiv(N, rows)), dim3(256), 0, st, rowptr, N, rows, v.erow);
    const int64_t nt = cdiv(E, kTileEdges);
    hipLaunchKernelGGL(tile_tab_kernel, dim3((unsigned)cdiv(nt, 4)), dim3(256), 0, st, v.erow, E, nt, v.tile_tab);
    const int eb = (int)std::min<int64_t>(cdiv(E, 256), 8192);
    if (count && host[1] <= kSortMax) {
      hipLaunchKernelGGL(csc_fill_kernel, dim3(eb), dim3(256), 0, st, col, E, t.cnt, v.csc_eid);
      hipLaunchKernelGGL(csc_sort_kernel, dim3((unsigned)std::min<int64_t>(cdiv(N, 4), 65536)), dim3(256), 0, st,
                         v.csc_ptr, N, v.csc_eid);
    } else {
      hipLaunchKernelGGL(iota_kernel, dim3(eb), dim3(256), 0, st, t.vals_in, E);
      size_t cb = t.cub_bytes;
      if (hipcub::DeviceRadixSort::SortPairs(t.cub, cb, col, t.keys_out, t.vals_in, v.csc_eid, (int)E, 0, key_bits(N),
                                             st) != hipSuccess)
        return EGNN_ERR_HIP;
      if (!count) {
        const int pb = (int)std::min<int64_t>(cdiv(N + 1, 256), 4096);
        hipLaunchKernelGGL(csc_ptr_kernel, dim3(pb), dim3(256), 0, st, t.keys_out, N, E, v.csc_ptr);
      }
    }
  }
  if (hipGetLastError() != hipSuccess) return EGNN_ERR_HIP;
  return EGNN_OK;
}

}  // namespace egnn
