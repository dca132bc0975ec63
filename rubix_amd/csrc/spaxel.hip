// Spaxel assignment and the stable sort-by-spaxel index.
//
// rbx_spaxel_assign replaces square_spaxel_assignment
// (rubix/telescope/utils.py:77-152).  rbx_spaxel_sort is new: a stable,
// deterministic counting sort of the spaxel ids (the reference analogue is
// the lexsort + searchsorted of rubix/spectra/dust/dust_extinction.py:237-267).
//
// Sort design (integer work, HBM-bound, no floating point):
//   keys are bucketed into B = n_keys + 1 buckets (the last one collects ids
//   outside [0, n_keys)); the input is cut into tiles, each tile owned by one
//   workgroup whose wavefronts walk a stretch of it each in order, 64 stars per
//   round (sort_tile_kernel; sort_rank_kernel with one wavefront a tile past the
//   buckets whose counters fit LDS).
//   1. rank   : lanes with equal keys in a round are found with one ballot per
//               key bit; the lowest lane adds the group size to the stretch's
//               counter of the key and gets the count so far, so every
//               star's rank among the tile's stars of its key is known (and
//               stored) after one walk.  Only its own wavefront touches
//               a counter, so the result is deterministic.
//   2. scan   : exclusive scan over the bucket-major (bucket, tile) table
//               gives each tile its base position inside each bucket.
//   3. scatter: thread / star, position = base + rank: stars keep their input
//               order (stable).
//   The walk is a chain of rounds: about 1 us each with counters in memory,
//   where plan_tile() balances them against the table (about 4 ps an entry:
//   filled, read twice, written once), and a third of that with counters in LDS,
//   where plan_workgroup() fills the device with the largest tiles.  The table is kept to
//   2^24 entries.  Key counts past that with 4096-star tiles (a batch of many
//   galaxies: 310 000 keys over 31.8 M stars) sort in LSD radix passes over
//   D-bit digits of the bucket index, each pass the same stable rank + scan +
//   scatter over 2^D buckets, the scatter carrying each star's input index
//   and bucket along; stable passes give the same order as the one-pass sort.
//   Bucket offsets then come from a binary search of the sorted stars.
#include <math.h>
#include <stdarg.h>
#include <string.h>

#include <type_traits>

#include "rbx_common.h"

namespace rbx {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: %s", what, hipGetErrorString(e));
    return RBX_EHIP;
  }
  return RBX_OK;
}

// ------------------------------------------------------------ spaxel assign

template <bool kLds>
__global__ void spaxel_assign_kernel(const float* __restrict__ coords, int64_t n,
                                     int64_t stride, const float* __restrict__ edges,
                                     int n_edges, int32_t* __restrict__ out) {
  extern __shared__ float s_edges[];
  const float* e = edges;
  if (kLds) {
    for (int k = threadIdx.x; k < n_edges; k += blockDim.x) s_edges[k] = edges[k];
    __syncthreads();
    e = s_edges;
  }
  const int nb = n_edges - 1;
  for (int64_t i = gtid(); i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const float x = coords[i * stride];
    const float y = coords[i * stride + 1];
    int ix = upper_bound_f(e, n_edges, x) - 1;
    int iy = upper_bound_f(e, n_edges, y) - 1;
    ix = ix < 0 ? 0 : (ix > nb - 1 ? nb - 1 : ix);
    iy = iy < 0 ? 0 : (iy > nb - 1 ? nb - 1 : iy);
    out[i] = ix + nb * iy;
  }
}

// out[i, c] = v[i] in column `col`, 0 in the others (a velocity gradient of
// one component), one pass instead of a fill and a strided copy.
__global__ void __launch_bounds__(256) column_rows_kernel(const float* __restrict__ v, int64_t n,
                                                          int cols, int col,
                                                          float* __restrict__ out) {
  for (int64_t i = gtid(); i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const float x = v[i];
    for (int c = 0; c < cols; ++c) out[i * cols + c] = c == col ? x : 0.f;
  }
}

// ------------------------------------------------------------ integer scan

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanBlock = kScanThreads * kScanItems;

__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  for (int64_t i = gtid(); i < n; i += int64_t(gridDim.x) * blockDim.x) p[i] = v;
}

template <class T>
__device__ inline T block_exclusive_scan(T v, T* smem, T* total) {
  // smem: kScanThreads entries.  Hillis-Steele over the block (deterministic).
  const int t = threadIdx.x;
  smem[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    T add = (t >= off) ? smem[t - off] : T(0);
    __syncthreads();
    smem[t] += add;
    __syncthreads();
  }
  T incl = smem[t];
  *total = smem[kScanThreads - 1];
  __syncthreads();
  return incl - v;
}

__global__ void scan_reduce_kernel(const int32_t* __restrict__ in, int64_t n,
                                   int32_t* __restrict__ block_sums) {
  __shared__ int32_t smem[kScanThreads];
  const int64_t base = int64_t(blockIdx.x) * kScanBlock;
  int32_t s = 0;
  for (int k = 0; k < kScanItems; ++k) {
    int64_t i = base + int64_t(k) * kScanThreads + threadIdx.x;
    if (i < n) s += in[i];
  }
  int32_t tot;
  block_exclusive_scan<int32_t>(s, smem, &tot);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = tot;
}

// Single workgroup: exclusive scan of the block sums in place.
__global__ void scan_top_kernel(int32_t* __restrict__ sums, int64_t nblk) {
  __shared__ int32_t smem[kScanThreads];
  int32_t carry = 0;
  for (int64_t b0 = 0; b0 < nblk; b0 += kScanThreads) {
    int64_t i = b0 + threadIdx.x;
    int32_t v = i < nblk ? sums[i] : 0;
    int32_t tot;
    int32_t ex = block_exclusive_scan<int32_t>(v, smem, &tot);
    if (i < nblk) sums[i] = carry + ex;
    carry += tot;
  }
}

// Each block: exclusive scan of its kScanBlock elements (thread-contiguous
// runs of kScanItems) plus the block offset, in place.  kSums: block_off
// holds the blocks' own sums and the offset is the sum of the earlier ones
// (at most kScanSelf of them: a few loads a thread, one launch fewer);
// otherwise scan_top_kernel has scanned them.
constexpr int64_t kScanSelf = 4096;

template <bool kSums>
__global__ void __launch_bounds__(kScanThreads) scan_down_kernel(
    int32_t* __restrict__ data, int64_t n, const int32_t* __restrict__ block_off) {
  __shared__ int32_t smem[kScanThreads];
  int32_t off;
  if (kSums) {
    int32_t part = 0;
    for (int b = threadIdx.x; b < int(blockIdx.x); b += kScanThreads) part += block_off[b];
    block_exclusive_scan<int32_t>(part, smem, &off);
  } else {
    off = block_off[blockIdx.x];
  }
  const int64_t base = int64_t(blockIdx.x) * kScanBlock + int64_t(threadIdx.x) * kScanItems;
  // a full run of aligned data goes in 16-byte accesses
  const bool wide = base + kScanItems <= n && (reinterpret_cast<uintptr_t>(data) & 15) == 0;
  int32_t v[kScanItems];
  if (wide) {
#pragma unroll
    for (int k = 0; k < kScanItems; k += 4) {
      const int4 q = *reinterpret_cast<const int4*>(data + base + k);
      v[k] = q.x;
      v[k + 1] = q.y;
      v[k + 2] = q.z;
      v[k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? data[base + k] : 0;
  }
  int32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s += v[k];
  int32_t tot;
  int32_t ex = block_exclusive_scan<int32_t>(s, smem, &tot) + off;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int32_t c = v[k];
    v[k] = ex;
    ex += c;
  }
  if (wide) {
#pragma unroll
    for (int k = 0; k < kScanItems; k += 4)
      *reinterpret_cast<int4*>(data + base + k) = make_int4(v[k], v[k + 1], v[k + 2], v[k + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
      if (base + k < n) data[base + k] = v[k];
  }
}

// ------------------------------------------------------------ sort

struct SortPlan {
  int64_t n;
  int32_t n_keys;
  int32_t buckets;  // n_keys + 1 (overflow bucket last)
  int64_t tile;     // stars per tile, multiple of 64
  int64_t ntiles;
  int64_t table;    // (buckets or digit buckets) * ntiles
  int64_t room;     // table entries of the workspace: no fewer for more stars
  int nbits;        // bits needed to tell buckets apart
  int digit_bits;   // 0: one pass over all buckets; else radix digits of this width
  int passes;       // counting-sort passes
  int waves;        // wavefronts of a tile's workgroup (sort_tile_kernel), 0: sort_rank_kernel
  int rounds;       // and each one's rounds of 64 stars: 1, 2, 4, 8 or 16
};

constexpr int64_t kTableCap = int64_t(1) << 24;  // (bucket, tile) counters
constexpr int64_t kSortTile = 4096;              // most stars per tile

// Stars per tile for `buckets` counters a tile: tile / 64 rounds of ~1 us
// against buckets * n / tile table entries of ~4 ps, least at
// tile = sqrt(2.56e-4 buckets n), within [64, kSortTile].  Measured at 1 M
// stars and 2500 keys: rank + scatter + table 182 us at 4096 stars per tile.
static int64_t plan_tile(int64_t n, int64_t buckets) {
  const double t = sqrt(2.56e-4 * double(buckets) * double(n));
  int64_t tile = t >= double(kSortTile) ? kSortTile : (int64_t(t) + 63) / 64 * 64;
  if (tile < 64) tile = 64;
  while (tile < kSortTile && buckets * ((n + tile - 1) / tile) > kTableCap) tile += 64;
  return tile;
}

constexpr int64_t kTileLds = 64 * 1024;  // counters of a sort_tile_kernel workgroup

// sort_tile_kernel's workgroup for `buckets` counters a wavefront (2 bytes
// each): as many wavefronts as the LDS holds, up to 16 and over the SIMDs
// evenly, and as few rounds each as leave no more workgroups than the device
// takes at once (two on each of 256 CUs).  From 2 wavefronts (16384 buckets) up
// if the tiles keep the table within its cap.
static bool plan_workgroup(SortPlan* p, int64_t buckets) {
  int64_t w = kTileLds / (4 * ((buckets + 1) / 2));
  if (w < 2 || p->n < 1) return false;
  if (w > 16) w = 16;
  if (w > 4) w &= ~int64_t(3);
  int r = 1;
  while (r < 16 && (p->n + 64 * w * r - 1) / (64 * w * r) > 512) r *= 2;
  const int64_t tile = 64 * w * r, ntiles = (p->n + tile - 1) / tile;
  if (buckets * ntiles > kTableCap) return false;
  p->waves = int(w);
  p->rounds = r;
  p->tile = tile;
  p->ntiles = ntiles;
  return true;
}

// Table entries the workspace has for `buckets` keys in one pass.  The tiles
// grow with the star count, so the table of more stars can be the smaller one;
// this bound of both plans never shrinks, and a workspace sized for the most
// stars of a program takes every smaller call.
static int64_t table_room(int64_t n, int64_t buckets) {
  int64_t w = kTileLds / (4 * ((buckets + 1) / 2));
  int64_t tiles;
  if (w >= 2) {  // plan_workgroup: at most 512 tiles until its largest ones
    if (w > 16) w = 16;
    if (w > 4) w &= ~int64_t(3);
    const int64_t least = (n + 64 * w - 1) / (64 * w), most = (n + 1024 * w - 1) / (1024 * w);
    tiles = most > 512 ? most : (least < 512 ? least : 512);
  } else {  // plan_tile: n / tile before its rounding, which adds less than one
    const double t = sqrt(2.56e-4 * double(buckets) * double(n));
    tiles = int64_t(double(n) / (t > double(kSortTile) ? double(kSortTile) : (t < 64 ? 64. : t))) + 2;
  }
  if (tiles < 1) tiles = 1;
  return buckets * tiles < kTableCap ? buckets * tiles : kTableCap;
}

static SortPlan make_plan(int64_t n, int32_t n_keys) {
  SortPlan p;
  p.n = n;
  p.n_keys = n_keys;
  p.buckets = n_keys + 1;
  int b = 1;
  while ((int64_t(1) << b) < p.buckets) ++b;
  p.nbits = b;
  const int64_t most = n > 0 ? (n + kSortTile - 1) / kSortTile : 1;  // tiles at the largest tile
  int64_t buckets = p.buckets;
  if (int64_t(p.buckets) * most <= kTableCap) {
    p.digit_bits = 0;
    p.passes = 1;
  } else {
    // most <= 2^19 for n < 2^31, so digits of at least 5 bits fit; then the
    // fewest equal digits of that many passes
    int d = 16;
    while (d > 1 && (int64_t(1) << d) * most > kTableCap) --d;
    p.passes = (p.nbits + d - 1) / d;
    p.digit_bits = (p.nbits + p.passes - 1) / p.passes;
    buckets = int64_t(1) << p.digit_bits;
  }
  p.waves = p.rounds = 0;
  if (!plan_workgroup(&p, buckets)) {
    p.tile = plan_tile(n, buckets);
    p.ntiles = n > 0 ? (n + p.tile - 1) / p.tile : 1;
  }
  p.table = buckets * p.ntiles;
  p.room = p.digit_bits ? kTableCap : table_room(n, buckets);
  if (p.room < p.table) p.room = p.table;
  return p;
}

// Every star's rank in its tile, and for radix passes the input index and
// bucket of every position: three n-element buffers (one index, two buckets)
// beside the caller's perm.  The last radix pass writes no buckets, so with
// two passes the ranks take the second bucket buffer.
template <class S>
static void sort_layout(S& c, const SortPlan& p, int32_t** table, int32_t** blocks,
                        uint16_t** rank, int32_t** tperm, int32_t** b0, int32_t** b1) {
  auto* t = c.template take<int32_t>(p.room);
  auto* bl = c.template take<int32_t>((p.room + kScanBlock - 1) / kScanBlock + 1);
  const int64_t n1 = p.n > 0 ? p.n : 1;
  const int64_t rn = p.digit_bits ? n1 : 0;
  auto* tp = c.template take<int32_t>(rn);
  auto* x0 = c.template take<int32_t>(rn);
  auto* x1 = c.template take<int32_t>(rn);
  const bool shared = p.passes == 2;
  auto* rk = c.template take<uint16_t>(shared ? 0 : n1);
  if (table) *table = reinterpret_cast<int32_t*>(t);
  if (blocks) *blocks = reinterpret_cast<int32_t*>(bl);
  if (tperm) *tperm = reinterpret_cast<int32_t*>(tp);
  if (b0) *b0 = reinterpret_cast<int32_t*>(x0);
  if (b1) *b1 = reinterpret_cast<int32_t*>(x1);
  if (rank) *rank = shared ? reinterpret_cast<uint16_t*>(x1) : reinterpret_cast<uint16_t*>(rk);
}

struct SizerAdapter {
  Sizer s;
  template <class T>
  T* take(size_t count) {
    s.take<T>(count);
    return nullptr;
  }
};

__device__ inline int bucket_of(int32_t id, int32_t n_keys) {
  return (id >= 0 && id < n_keys) ? id : n_keys;
}

// Lanes of the wavefront holding the same key (restricted to `active`).
__device__ inline uint64_t peer_mask(int key, uint64_t active, int nbits) {
  uint64_t peers = active;
  for (int b = 0; b < nbits; ++b) {
    const int bit = (key >> b) & 1;
    const uint64_t bal = __ballot(bit);
    peers &= bit ? bal : ~bal;
  }
  return peers;
}

// The sort key of element i is its bucket bucket_of(in[i]), or with mask != 0
// the digit (bucket >> shift) & mask.
__device__ inline int sort_key(int full, int shift, int32_t mask) {
  return mask ? ((full >> shift) & mask) : full;
}

// One wavefront walks one tile in input order: rank[i] = number of earlier
// stars of the tile with the same key (< tile <= 4096), table[key][tile] = the
// tile's count of the key.  The next round's keys are loaded ahead of this
// round's counter round trip.  Bound by that chain: 64 rounds of 4096-star
// tiles took 54-76 us for any star count from 10 k up, and a second such
// walk scattered; 10 k stars now take one round.
__global__ void __launch_bounds__(64) sort_rank_kernel(
    const int32_t* __restrict__ in, int64_t n, int32_t n_keys, int64_t tile, int64_t ntiles,
    int nbits, int shift, int32_t mask, int32_t* __restrict__ table, uint16_t* __restrict__ rank) {
  const int lane = threadIdx.x;
  const int64_t t = blockIdx.x;
  const int64_t begin = t * tile;
  const int64_t end = begin + tile < n ? begin + tile : n;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int32_t next = begin + lane < end ? in[begin + lane] : 0;
  for (int64_t r = begin; r < end; r += 64) {
    const int64_t i = r + lane;
    const bool valid = i < end;
    const int key = sort_key(bucket_of(next, n_keys), shift, mask);
    next = i + 64 < end ? in[i + 64] : 0;
    const uint64_t active = __ballot(valid);
    const uint64_t peers = peer_mask(key, active, nbits);  // all lanes take part
    const int leader = __ffsll((unsigned long long)peers) - 1;
    int32_t base = 0;
    if (valid && lane == leader) base = atomicAdd(table + int64_t(key) * ntiles + t, __popcll(peers));
    base = __shfl(base, leader < 0 ? 0 : leader, 64);
    if (valid) rank[i] = uint16_t(base + __popcll(peers & lt_mask));
  }
}

// sort_rank_kernel for a tile of a workgroup: wavefront w walks stars
// [w, w + 1) * 64 R of the tile with counters of its own in LDS, so its rounds
// wait for LDS and not for memory, and the wavefronts' counts are summed in their
// order.  Two 16-bit counters a word: a wavefront counts to 1024, a tile to
// 16384.  The whole table is written, so nothing clears it.  Consecutive tiles
// go to one XCD, whose L2 joins their neighbouring counters.
// 1 M stars, 2500 keys: 13 us, 39 with a wavefront a tile (and its smaller
// tiles' table five times as large: scan 11 us, 31, and a fill of 6).
template <int R>
__global__ void __launch_bounds__(1024) sort_tile_kernel(
    const int32_t* __restrict__ in, int64_t n, int32_t n_keys, int buckets, int64_t ntiles,
    int nbits, int shift, int32_t mask, int32_t* __restrict__ table, uint16_t* __restrict__ rank) {
  extern __shared__ uint32_t counters[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), n_waves = blockDim.x >> 6;
  const int words = (buckets + 1) >> 1;
  const int64_t per = (ntiles + 7) / 8;
  const int64_t t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= ntiles) return;
  const int64_t begin = (t * n_waves + w) * (64 * R);
  int32_t id[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = begin + u * 64 + lane;
    id[u] = i < n ? in[i] : 0;
  }
  for (int k = tid; k < n_waves * words; k += blockDim.x) counters[k] = 0;
  __syncthreads();
  uint32_t* own = counters + w * words;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int key[R];
  uint32_t local[R];  // rank within the wavefront's stars
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const bool valid = begin + u * 64 + lane < n;
    key[u] = sort_key(bucket_of(id[u], n_keys), shift, mask);
    const uint64_t peers = peer_mask(key[u], __ballot(valid), nbits);  // all lanes take part
    const int leader = __ffsll((unsigned long long)peers) - 1;
    const int half = 16 * (key[u] & 1);
    uint32_t old = 0;
    if (valid && lane == leader) old = atomicAdd(own + (key[u] >> 1), uint32_t(__popcll(peers)) << half);
    old = __shfl(old, leader < 0 ? 0 : leader, 64);
    local[u] = ((old >> half) & 0xffffu) + uint32_t(__popcll(peers & lt_mask));
  }
  __syncthreads();
  for (int j = tid; j < words; j += blockDim.x) {
    uint32_t run = 0;
    for (int v = 0; v < n_waves; ++v) {
      const uint32_t c = counters[v * words + j];
      counters[v * words + j] = run;
      run += c;
    }
    table[int64_t(2 * j) * ntiles + t] = int32_t(run & 0xffffu);
    if (2 * j + 1 < buckets) table[int64_t(2 * j + 1) * ntiles + t] = int32_t(run >> 16);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t i = begin + u * 64 + lane;
    if (i < n)
      rank[i] = uint16_t(((own[key[u] >> 1] >> (16 * (key[u] & 1))) & 0xffffu) + local[u]);
  }
}

// pos = the star's base in the scanned table + its rank: perm[pos] = the
// element's input index (src_perm[i], or i on the first pass), bucket_out[pos]
// = its bucket, sorted[pos] = its original id (ids[perm[pos]]; in[i] itself on
// the first pass), offsets[k] (where wanted) = the first position of key k, k in
// [0, n_keys].
__global__ void __launch_bounds__(256) sort_scatter_kernel(
    const int32_t* __restrict__ in, int64_t n, int32_t n_keys, uint32_t tile, int64_t ntiles,
    int shift, int32_t mask, const int32_t* __restrict__ table, const uint16_t* __restrict__ rank,
    const int32_t* __restrict__ src_perm, const int32_t* __restrict__ ids,
    int32_t* __restrict__ perm, int32_t* __restrict__ bucket_out, int32_t* __restrict__ sorted,
    int32_t* __restrict__ offsets) {
  if (offsets)
    for (int64_t k = gtid(); k <= n_keys; k += int64_t(gridDim.x) * blockDim.x)
      offsets[k] = table[k * ntiles];
  for (int64_t i = gtid(); i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const int32_t id = in[i];
    const int full = bucket_of(id, n_keys);
    const int key = sort_key(full, shift, mask);
    const int32_t pos = table[int64_t(key) * ntiles + uint32_t(i) / tile] + int32_t(rank[i]);
    const int32_t src = src_perm ? src_perm[i] : int32_t(i);
    perm[pos] = src;
    if (bucket_out) bucket_out[pos] = full;
    if (sorted) sorted[pos] = src_perm ? ids[src] : id;
  }
}

// offsets[k] = number of sorted stars (perm) whose bucket lies below k, k in
// [0, n_keys].
__global__ void bucket_offsets_kernel(const int32_t* __restrict__ ids,
                                      const int32_t* __restrict__ perm, int64_t n, int32_t n_keys,
                                      int32_t* __restrict__ offsets) {
  for (int64_t k = gtid(); k <= n_keys; k += int64_t(gridDim.x) * blockDim.x) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (bucket_of(ids[perm[mid]], n_keys) < k) lo = mid + 1;
      else hi = mid;
    }
    offsets[k] = int32_t(lo);
  }
}

static int grid_for(int64_t n, int threads, int64_t cap = 65536) {
  int64_t g = (n + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return int(g);
}

int exclusive_scan_i32(int32_t* data, int64_t n, int32_t* blocks, hipStream_t s) {
  const int64_t nblk = (n + kScanBlock - 1) / kScanBlock;
  if (nblk == 0) return RBX_OK;
  if (nblk > 1)
    hipLaunchKernelGGL(scan_reduce_kernel, dim3(nblk), dim3(kScanThreads), 0, s, data, n, blocks);
  if (nblk > kScanSelf) {
    hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(kScanThreads), 0, s, blocks, nblk);
    hipLaunchKernelGGL(scan_down_kernel<false>, dim3(nblk), dim3(kScanThreads), 0, s, data, n,
                       blocks);
  } else {
    hipLaunchKernelGGL(scan_down_kernel<true>, dim3(nblk), dim3(kScanThreads), 0, s, data, n,
                       blocks);
  }
  return check_launch("exclusive_scan_i32");
}

void fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
}

size_t sort_workspace_size(int64_t n, int32_t n_keys) {
  SortPlan p = make_plan(n, n_keys);
  SizerAdapter a;
  sort_layout(a, p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
  return a.s.used;
}

// Workspace enough for any key count in [1, max_keys]: the table never
// passes 2^24 entries, and the radix buffers are there whenever max_keys
// would need them.
size_t sort_workspace_bound(int64_t n, int32_t max_keys) {
  SortPlan p = make_plan(n, max_keys);
  p.room = kTableCap;
  SizerAdapter a;
  sort_layout(a, p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
  return a.s.used;
}

// Rank, scan and scatter of one pass; returns the launch status.
static int sort_pass(const SortPlan& p, const int32_t* in, int shift, int32_t mask, int nbits,
                     int32_t* table, int32_t* blocks, uint16_t* rank, const int32_t* src_perm,
                     const int32_t* ids, int32_t* perm, int32_t* bucket_out, int32_t* sorted,
                     int32_t* offsets, hipStream_t s) {
  if (p.waves) {
    const int buckets = int(p.table / p.ntiles);
    const dim3 grid(unsigned((p.ntiles + 7) / 8 * 8)), block(64 * p.waves);
    const size_t lds = size_t(p.waves) * ((buckets + 1) / 2) * 4;
    auto launch = [&](auto r) {
      hipLaunchKernelGGL(sort_tile_kernel<decltype(r)::value>, grid, block, lds, s, in, p.n, p.n_keys,
                         buckets, p.ntiles, nbits, shift, mask, table, rank);
    };
    switch (p.rounds) {
      case 1: launch(std::integral_constant<int, 1>{}); break;
      case 2: launch(std::integral_constant<int, 2>{}); break;
      case 4: launch(std::integral_constant<int, 4>{}); break;
      case 8: launch(std::integral_constant<int, 8>{}); break;
      default: launch(std::integral_constant<int, 16>{}); break;
    }
  } else {
    fill_i32(table, p.table, 0, s);
    if (p.n > 0)
      hipLaunchKernelGGL(sort_rank_kernel, dim3(p.ntiles), dim3(64), 0, s, in, p.n, p.n_keys, p.tile,
                         p.ntiles, nbits, shift, mask, table, rank);
  }
  int rc = exclusive_scan_i32(table, p.table, blocks, s);
  if (rc) return rc;
  if (p.n > 0)
    hipLaunchKernelGGL(sort_scatter_kernel, dim3(grid_for(p.n, 256)), dim3(256), 0, s, in, p.n,
                       p.n_keys, uint32_t(p.tile), p.ntiles, shift, mask, table, rank, src_perm,
                       ids, perm, bucket_out, sorted, offsets);
  else if (offsets)
    fill_i32(offsets, int64_t(p.n_keys) + 1, 0, s);
  return check_launch("rbx_spaxel_sort");
}

// Sort used by the fused path too; the workspace is carved by the caller.
int spaxel_sort_impl(const int32_t* ids, int64_t n, int32_t n_keys, int32_t* perm,
                     int32_t* sorted, int32_t* offsets, void* ws, size_t ws_bytes,
                     hipStream_t s) {
  SortPlan p = make_plan(n, n_keys);
  Carver c(ws, ws_bytes);
  int32_t *table = nullptr, *blocks = nullptr, *tperm = nullptr, *b0 = nullptr, *b1 = nullptr;
  uint16_t* rank = nullptr;
  sort_layout(c, p, &table, &blocks, &rank, &tperm, &b0, &b1);
  if (!c.ok) return fail(RBX_EWORKSPACE, "rbx_spaxel_sort: workspace too small");
  if (!p.digit_bits)
    return sort_pass(p, ids, 0, 0, p.nbits, table, blocks, rank, nullptr, ids, perm, nullptr,
                     sorted, offsets, s);
  // LSD radix: pass q sorts by bits [q D, q D + D) of the bucket, stably;
  // the index buffers alternate so that the last pass writes perm
  const int32_t mask = (int32_t(1) << p.digit_bits) - 1;
  const int32_t* in = ids;
  const int32_t* src = nullptr;
  int32_t* bufs[2] = {b0, b1};
  for (int q = 0; q < p.passes; ++q) {
    const bool last = q == p.passes - 1;
    int32_t* pout = ((p.passes - 1 - q) & 1) ? tperm : perm;
    int32_t* bout = last ? nullptr : bufs[q & 1];
    const int width = last ? p.nbits - q * p.digit_bits : p.digit_bits;
    int rc = sort_pass(p, in, q * p.digit_bits, mask, width, table, blocks, rank, src, ids,
                       pout, bout, last ? sorted : nullptr, nullptr, s);
    if (rc) return rc;
    in = bout;
    src = pout;
  }
  hipLaunchKernelGGL(bucket_offsets_kernel, dim3(grid_for(int64_t(n_keys) + 1, 256)), dim3(256), 0,
                     s, ids, perm, n, n_keys, offsets);
  return check_launch("rbx_spaxel_sort");
}

}  // namespace rbx

extern "C" {

int rbx_version(void) { return 100; }

const char* rbx_last_error_string(void) { return rbx::g_err; }

int rbx_spaxel_assign(const float* coords, int64_t n, int64_t stride, const float* edges,
                      int32_t n_edges, int32_t* out_ids, void* stream) {
  using namespace rbx;
  if (n < 0 || stride < 2 || n_edges < 2 || (n > 0 && (!coords || !out_ids)) || !edges)
    return fail(RBX_EINVAL, "rbx_spaxel_assign: bad arguments (need n >= 0, stride >= 2, n_edges >= 2)");
  if (n == 0) return RBX_OK;
  hipStream_t s = as_stream(stream);
  const int threads = 256;
  const int grid = grid_for(n, threads);
  if (n_edges <= 8192) {
    hipLaunchKernelGGL(spaxel_assign_kernel<true>, dim3(grid), dim3(threads),
                       size_t(n_edges) * sizeof(float), s, coords, n, stride, edges, n_edges, out_ids);
  } else {
    hipLaunchKernelGGL(spaxel_assign_kernel<false>, dim3(grid), dim3(threads), 0, s, coords, n,
                       stride, edges, n_edges, out_ids);
  }
  return check_launch("rbx_spaxel_assign");
}

int rbx_column_rows(const float* v, int64_t n, int32_t cols, int32_t col, float* out, void* stream) {
  using namespace rbx;
  if (n < 0 || cols < 1 || col < 0 || col >= cols || (n > 0 && (!v || !out)))
    return fail(RBX_EINVAL, "rbx_column_rows: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL(column_rows_kernel, dim3(grid_for(n, 256)), dim3(256), 0,
                     as_stream(stream), v, n, cols, col, out);
  return check_launch("rbx_column_rows");
}

size_t rbx_spaxel_sort_workspace_size(int64_t n, int32_t n_keys) {
  if (n < 0 || n_keys < 1) return 0;
  return rbx::sort_workspace_size(n, n_keys);
}

int rbx_spaxel_sort(const int32_t* ids, int64_t n, int32_t n_keys, int32_t* perm,
                    int32_t* sorted, int32_t* offsets, void* workspace, size_t workspace_bytes,
                    void* stream) {
  using namespace rbx;
  if (n < 0 || n_keys < 1 || !offsets || (n > 0 && (!ids || !perm)))
    return fail(RBX_EINVAL, "rbx_spaxel_sort: bad arguments");
  if (n > INT32_MAX - 1) return fail(RBX_EINVAL, "rbx_spaxel_sort: n must fit int32");
  if (int64_t(n_keys) + 1 > (int64_t(1) << 30))
    return fail(RBX_EINVAL, "rbx_spaxel_sort: n_keys too large");
  return spaxel_sort_impl(ids, n, n_keys, perm, sorted, offsets, workspace, workspace_bytes,
                          as_stream(stream));
}

}  // extern "C"
