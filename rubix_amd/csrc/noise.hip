// apply_noise (rubix/core/noise.py:17-80, rubix/telescope/noise/noise.py:8-115)
// on a datacube of n_spaxel rows x n_target bins:
//   F[p]      = sum_l cube[p, l]                                   (noise.py:62)
//   M         = median of (F > 0 ? F : NaN) over all spaxels, NaN -> 0
//               (jnp.median propagates NaN: one spaxel without positive flux
//               makes M = 0 and the added noise zero everywhere; :65-69)
//   S[p]      = F[p] > 0 ? (sqrt(M) / sn[p]) / sqrt(F[p]) : 0        (:72-78)
//   out[p, l] = cube[p, l] + cube[p, l] * (z[p, l] * S[p])          (:108-113)
// z[i] (i = flat index p * n_target + l) follows jax.random's published
// construction for key = PRNGKey(seed) = (seed >> 32, seed & 0xffffffff):
//   bits = y0 ^ y1,  (y0, y1) = Threefry-2x32-20(key, counter (i >> 32, i & 0xffffffff))
//   u01  = float((bits >> 9) | 0x3f800000) - 1                       (uniform)
//   z    = sqrt(2) * erfinv(max(lo, 2 u01 + lo)),  lo = nextafter(-1, 0)  (normal)
// Threefry-2x32 with 20 rounds is Salmon et al., "Parallel random numbers: as
// easy as 1, 2, 3" (SC 2011).  The draws are recomputed in the adjoint, never
// stored.
#include <math.h>

#include <type_traits>

#include "rbx_common.h"

static_assert(sizeof(rbx_noise_stats) == 16, "rbx_noise_stats layout");

namespace rbx {

constexpr int kSelThreads = 1024;  // the one workgroup of the median kernel
constexpr int kSelLoads = 16;      // its loads in flight per thread
constexpr int kSelCopies = 32;     // copies of its digit counters (one LDS bank each)
constexpr int kSumLoads = 8;       // loads in flight per thread of noise_coef_kernel
constexpr int kRowThreads = 256;
constexpr int kItemBins = 2048;  // most bins per elementwise item (of one wavefront)
constexpr int kFewRows = 8192;   // below this a row of the adjoint gets a whole workgroup

__device__ inline uint32_t rotl32(uint32_t x, int r) { return (x << r) | (x >> (32 - r)); }

// Rotations 13 15 26 6 | 17 29 16 24, key parity constant 0x1BD11BDA, key
// injection (with the injection count added to word 1) after every 4 rounds.
__device__ inline void threefry2x32(uint32_t k0, uint32_t k1, uint32_t c0, uint32_t c1,
                                    uint32_t* o0, uint32_t* o1) {
  const int rot[8] = {13, 15, 26, 6, 17, 29, 16, 24};
  const uint32_t ks[3] = {k0, k1, k0 ^ k1 ^ 0x1BD11BDAu};
  uint32_t x0 = c0 + ks[0], x1 = c1 + ks[1];
#pragma unroll
  for (int r = 0; r < 20; ++r) {
    x0 += x1;
    x1 = rotl32(x1, rot[r & 7]);
    x1 ^= x0;
    if ((r & 3) == 3) {
      const int s = (r >> 2) + 1;
      x0 += ks[s % 3];
      x1 += ks[(s + 1) % 3] + uint32_t(s);
    }
  }
  *o0 = x0;
  *o1 = x1;
}

struct NoiseKey {
  uint32_t k0, k1;
};

inline NoiseKey key_of(uint64_t seed) { return {uint32_t(seed >> 32), uint32_t(seed)}; }

__device__ inline float mul_nc(float x, float y) {
#pragma clang fp contract(off)
  return x * y;
}

template <bool kUniform>
__device__ inline float draw(NoiseKey key, uint32_t hi, uint32_t lo_word) {
  uint32_t y0, y1;
  threefry2x32(key.k0, key.k1, hi, lo_word, &y0, &y1);
  const float f = __uint_as_float(((y0 ^ y1) >> 9) | 0x3f800000u) - 1.0f;
  if (kUniform) return f;
  const float lo = -0x1.fffffep-1f;          // nextafter(-1, 0)
  const float u = fmaxf(lo, f * 2.0f + lo);  // 2f is exact: one rounding, fused or not
  return mul_nc(0x1.6a09e6p+0f, erfinvf(u));  // float32(sqrt(2))
}

// z[i .. i + 3].  The counter's low word goes through a register that the
// compiler knows nothing about: it otherwise carries the sums of counter and
// key words along the caller's loop, one induction variable each.
template <bool kUniform>
__device__ inline void draw4(NoiseKey key, uint64_t i, float* z) {
  uint32_t lo = uint32_t(i);
  asm("" : "+v"(lo));
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t w = lo + uint32_t(e);
    z[e] = draw<kUniform>(key, uint32_t(i >> 32) + (w < uint32_t(e) ? 1u : 0u), w);
  }
}

template <bool kUniform>
__global__ void __launch_bounds__(256) noise_sample_kernel(int64_t n, NoiseKey key,
                                                           float* __restrict__ out) {
  for (int64_t i = gtid(); i < n; i += int64_t(gridDim.x) * blockDim.x)
    out[i] = draw<kUniform>(key, uint32_t(uint64_t(i) >> 32), uint32_t(i));
}

// Block-wide double sum in a fixed order (wave butterflies, then waves in order).
__device__ inline double block_sum(double v, double* sm) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) sm[wave] = v;
  __syncthreads();
  double tot = 0.0;
  for (int w = 0; w < int(blockDim.x / kWave); ++w) tot += sm[w];
  __syncthreads();
  return tot;
}

// Flux image: F[p] = sum_l cube[p, l], one workgroup per spaxel row,
// double accumulation in a fixed order, rounded once.
__global__ void __launch_bounds__(kRowThreads) flux_rows_kernel(const float* __restrict__ cube,
                                                                int n_spaxel, int nt,
                                                                float* __restrict__ flux) {
  __shared__ double sm[kRowThreads / kWave];
  for (int p = blockIdx.x; p < n_spaxel; p += gridDim.x) {
    const int64_t row = int64_t(p) * nt;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int l = threadIdx.x;
    for (; l + 3 * kRowThreads < nt; l += 4 * kRowThreads) {
      a0 += cube[row + l];
      a1 += cube[row + l + kRowThreads];
      a2 += cube[row + l + 2 * kRowThreads];
      a3 += cube[row + l + 3 * kRowThreads];
    }
    for (; l < nt; l += kRowThreads) a0 += cube[row + l];
    const double tot = block_sum((a0 + a1) + (a2 + a3), sm);
    if (threadIdx.x == 0) flux[p] = float(tot);
  }
}

// Four consecutive floats at any 4-byte alignment (one 16-byte access).
struct alignas(4) Float4u {
  float v[4];
};

// Calls f(l, n) for the caller's runs of n <= 4 consecutive bins of [l0, l1):
// thread `t` of `threads` side by side.
template <class F>
__device__ inline void quads(int l0, int l1, int t, int threads, F&& f) {
  for (int l = l0 + 4 * t; l < l1; l += 4 * threads) f(l, l1 - l < 4 ? l1 - l : 4);
}

__device__ inline void load4(float* v, const float* src, int n) {
  if (n == 4) {
    const Float4u q = *reinterpret_cast<const Float4u*>(src);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = q.v[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = e < n ? src[e] : 0.f;
  }
}

__device__ inline void store4(float* dst, const float* v, int n) {
  if (n == 4) {
    *reinterpret_cast<Float4u*>(dst) = {{v[0], v[1], v[2], v[3]}};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) dst[e] = v[e];
  }
}

// Adjoint, first pass over spaxel row p (each draw made once): the direct
// term dcube = dout + dout * (z * S[p]) and A[p] = sum_l dout * cube * z
// (double, fixed order).  Rows with S[p] == 0 copy dout and get A = 0.
// Two cubes read and one written against some 75 integer instructions a draw
// (0.29 ms and 0.22 ms at 300 x 300 x 1369): four bins a thread give the draws
// something to overlap with.  kRowWaves wavefronts take a row: one, with no
// barrier, where there are rows enough to fill the device, else four.
template <int kRowWaves, bool kUniform>
__global__ void __launch_bounds__(kRowThreads) noise_bwd_rows_kernel(
    const float* __restrict__ cube, const float* __restrict__ dout, int n_spaxel, int nt,
    const float* __restrict__ s2n, NoiseKey key, double* __restrict__ dots,
    float* __restrict__ dcube) {
  __shared__ double sm[kRowThreads / kWave];
  constexpr int kRows = kRowThreads / kWave / kRowWaves;  // rows of a workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int t = threadIdx.x % (kRowWaves * kWave);
  for (int p = blockIdx.x * kRows + wave / kRowWaves; p < n_spaxel; p += gridDim.x * kRows) {
    const int64_t row = int64_t(p) * nt;
    const float s = s2n[p];
    double acc = 0.0;
    quads(0, nt, t, kRowWaves * kWave, [&](int l, int n) {
      float g[4];
      load4(g, dout + row + l, n);
      if (s != 0.f) {
        float c[4], d[4], z[4];
        load4(c, cube + row + l, n);
        draw4<kUniform>(key, uint64_t(row + l), z);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (e < n) acc += double(g[e]) * double(c[e]) * double(z[e]);
          d[e] = g[e] + g[e] * (z[e] * s);
        }
        store4(dcube + row + l, d, n);
      } else {
        store4(dcube + row + l, g, n);
      }
    });
    const double tot = kRowWaves == 1 ? wave_sum(acc) : block_sum(acc, sm);
    if (t == 0) dots[p] = tot;
  }
}

// Index of the rank-th (0-based) element whose bits equal `bits`, in index
// order (the element a stable sort puts at that rank).
__device__ int nth_equal(const float* F, int n, uint32_t bits, int rank,
                         unsigned* wave_cnt, int* s_idx) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int n_waves = blockDim.x / kWave;
  if (threadIdx.x == 0) *s_idx = -1;
  int running = 0;
  for (int base = 0; base < n; base += blockDim.x) {
    const int i = base + threadIdx.x;
    const bool eq = i < n && __float_as_uint(F[i]) == bits;
    const uint64_t m = __ballot(eq);
    if (lane == 0) wave_cnt[wave] = unsigned(__popcll(m));
    __syncthreads();
    int before = running;
    int total = running;
    for (int w = 0; w < n_waves; ++w) {
      if (w < wave) before += int(wave_cnt[w]);
      total += int(wave_cnt[w]);
    }
    before += __popcll(m & ((uint64_t(1) << lane) - 1));
    if (eq && before == rank) *s_idx = i;
    __syncthreads();
    running = total;
    if (running > rank) break;
  }
  __syncthreads();
  return *s_idx;
}

// One workgroup: the median of the flux image (NaN-propagating, as
// jnp.median) and the spaxels that hold it (for the adjoint).  The bit patterns
// of positive floats order like the values: four passes of 8 bits give the
// lower of the two middle ranks, a last one how many spaxels hold that
// value and the smallest value above it, from which the upper rank follows.
// Bound by the latency of one workgroup's loads, so each thread has kSelLoads
// in flight, and the image stays in registers where they hold all of it
// (kHeld); a digit's counter has kSelCopies copies, because fluxes share their
// exponents and one counter would serialise a wavefront's 64 additions.
// 90 000 spaxels: 414 us with one load in flight and a pass per rank and bin, 67 us
// now; 2 500 (in LDS before, in registers now): 19.
template <bool kHeld>
__global__ void __launch_bounds__(kSelThreads) noise_median_kernel(
    const float* __restrict__ F, int n, rbx_noise_stats* __restrict__ stats) {
  __shared__ unsigned hist[256 * kSelCopies];
  __shared__ unsigned count[256];
  __shared__ unsigned wave_cnt[kSelThreads / kWave];
  __shared__ uint32_t s_pref;
  __shared__ int s_k, s_idx;
  __shared__ unsigned s_equal, s_first;
  __shared__ unsigned long long s_next;
  const int tid = threadIdx.x;
  float v[kSelLoads];
  auto load = [&](int64_t base) {
#pragma unroll
    for (int u = 0; u < kSelLoads; ++u) {
      const int64_t i = base + u * kSelThreads + tid;
      v[u] = i < n ? F[i] : 1.f;
    }
  };
  // f(i, bits of F[i]) over the thread's spaxels
  auto each = [&](auto&& f) {
    for (int64_t base = 0; base < n; base += kSelLoads * kSelThreads) {
      if (!kHeld) load(base);
#pragma unroll
      for (int u = 0; u < kSelLoads; ++u) {
        const int64_t i = base + u * kSelThreads + tid;
        if (i < n) f(unsigned(i), __float_as_uint(v[u]));
      }
    }
  };
  if (kHeld) load(0);
  // ranks floor((n-1)/2) and ceil((n-1)/2); the median is their midpoint
  const int k_lo = (n - 1) / 2, k_hi = n / 2;
  uint32_t prefix = 0, mask = 0;
  int k = k_lo;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int d = tid; d < 256 * kSelCopies; d += kSelThreads) hist[d] = 0;
    __syncthreads();
    int bad = 0;
    each([&](unsigned, uint32_t b) {
      if (!(__uint_as_float(b) > 0.f)) bad = 1;
      if ((b & mask) == prefix)
        atomicAdd(&hist[((b >> shift) & 255u) * kSelCopies + (tid & (kSelCopies - 1))], 1u);
    });
    if (__syncthreads_or(bad)) {  // some spaxel without positive flux
      if (tid == 0) *stats = {0.f, -1, -1, 1};
      return;
    }
    // four threads sum a digit's copies, each starting at another bank
    const int digit = tid >> 2;
    unsigned c = 0;
#pragma unroll
    for (int j = 0; j < kSelCopies / 4; ++j)
      c += hist[digit * kSelCopies + (tid & 3) * (kSelCopies / 4) +
                ((j + digit) & (kSelCopies / 4 - 1))];
    c += __shfl_xor(c, 1, kWave);
    c += __shfl_xor(c, 2, kWave);
    if ((tid & 3) == 0) count[digit] = c;
    __syncthreads();
    if (tid < kWave) {
      // wave 0: lane q owns digits 4q..4q+3; an inclusive shuffle scan finds
      // the one lane whose digits hold rank k (counts sum to more than k)
      unsigned h[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = count[4 * tid + j];
      const unsigned own = h[0] + h[1] + h[2] + h[3];
      unsigned incl = own;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const unsigned t = __shfl_up(incl, off, kWave);
        if (tid >= off) incl += t;
      }
      unsigned cum = incl - own;
      if (cum <= unsigned(k) && unsigned(k) < incl) {
        int d = 4 * tid;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          if (cum + h[j] > unsigned(k)) break;
          cum += h[j];
          ++d;
        }
        s_pref = prefix | (uint32_t(d) << shift);
        s_k = k - int(cum);
      }
    }
    __syncthreads();
    prefix = s_pref;
    k = s_k;
    mask |= 255u << shift;
    __syncthreads();
  }
  // prefix is the lower value, k its rank among the spaxels that hold it
  const uint32_t b_lo = prefix;
  if (tid == 0) {
    s_equal = 0;
    s_first = ~0u;
    s_next = ~0ull;
  }
  __syncthreads();
  unsigned equal = 0, first = ~0u;
  unsigned long long next = ~0ull;  // (bits, spaxel) of the smallest value above
  each([&](unsigned i, uint32_t b) {
    if (b == b_lo) {
      ++equal;
      if (i < first) first = i;
    } else if (b > b_lo) {
      const unsigned long long key = (static_cast<unsigned long long>(b) << 32) | i;
      if (key < next) next = key;
    }
  });
  if (equal) {
    atomicAdd(&s_equal, equal);
    atomicMin(&s_first, first);
  }
  if (next != ~0ull) atomicMin(&s_next, next);
  __syncthreads();
  const int lo_idx = k == 0 ? int(s_first) : nth_equal(F, n, b_lo, k, wave_cnt, &s_idx);
  uint32_t b_hi = b_lo;
  int hi_idx = lo_idx;
  if (k_hi != k_lo) {
    if (unsigned(k) + 1 < s_equal) {
      hi_idx = nth_equal(F, n, b_lo, k + 1, wave_cnt, &s_idx);
    } else {
      b_hi = uint32_t(s_next >> 32);
      hi_idx = int(uint32_t(s_next));
    }
  }
  if (tid == 0)
    *stats = {(__uint_as_float(b_lo) + __uint_as_float(b_hi)) * 0.5f, lo_idx, hi_idx, 0};
}

// Items of the elementwise passes, one per wavefront: spaxel p, bins [l0, l1).
struct RowItem {
  int p, l0, l1;
};
__device__ inline RowItem row_item(uint32_t item, uint32_t segs, int seg, int nt) {
  const uint32_t p = item / segs;
  const int l0 = int(item - p * segs) * seg;
  return {int(p), l0, nt - l0 > seg ? l0 + seg : nt};
}

// The first item and the stride between a wavefront's items.
__device__ inline uint64_t first_item() {
  return uint64_t(blockIdx.x) * (kRowThreads / kWave) +
         __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
}
__device__ inline uint64_t item_stride() { return uint64_t(gridDim.x) * (kRowThreads / kWave); }

// The S2N map and the noisy cube.  Bound by the draws (75 integer instructions
// each, 0.22 ms of 300 x 300 x 1369; HBM: 0.19): four consecutive bins a thread,
// 16-byte accesses, no thread without bins but in a row's last 256.  295 us, 410 with
// one bin a thread at a time and workgroups of 1024 bins.
template <bool kUniform>
__global__ void __launch_bounds__(kRowThreads) add_noise_kernel(
    const float* cube, int nt, uint32_t n_items, uint32_t segs, int seg,
    const float* __restrict__ flux, const float* __restrict__ sn,
    const rbx_noise_stats* __restrict__ stats, NoiseKey key,
    float* __restrict__ s2n, float* out) {
  const int lane = threadIdx.x & (kWave - 1);
  const float root_m = sqrtf(stats->median);
  for (uint64_t item = first_item(); item < n_items; item += item_stride()) {
    const RowItem it = row_item(uint32_t(item), segs, seg, nt);
    const float f = flux[it.p];
    const float s = f > 0.f ? (root_m / sn[it.p]) / sqrtf(f) : 0.f;
    if (it.l0 == 0 && lane == 0) s2n[it.p] = s;
    const int64_t row = int64_t(it.p) * nt;
    quads(it.l0, it.l1, lane, kWave, [&](int l, int n) {
      float c[4], z[4];
      load4(c, cube + row + l, n);
      draw4<kUniform>(key, uint64_t(row + l), z);
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] += mul_nc(c[e], z[e] * s);
      store4(out + row + l, c, n);
    });
  }
}

// dL/dF[p] of a spaxel that is not at the median, from A[p] = sum_l dout *
// cube * z.  With S[p] = sqrt(M)/sn[p] / sqrt(F[p]): dS/dF = -S / (2F).
__device__ inline double flux_gradient(double A, float s2n, float flux) {
  return -A * double(s2n) / (2.0 * double(flux));
}

// M > 0, so that the S map moves with the fluxes.
__device__ inline bool live(const rbx_noise_stats& st) {
  return st.any_nonpositive == 0 && st.median > 0.f;
}
__device__ inline bool has_median_spaxels(const rbx_noise_stats& st, int n) {
  return st.median_lo >= 0 && st.median_lo < n && st.median_hi >= 0 && st.median_hi < n;
}

// One workgroup: dL/dM = sum_p A[p] S[p] / (2M) (dS/dM = S / (2M)) goes to the
// flux of the spaxel(s) at the median, weight 1/2 for each of the two
// midpoint ranks: their dots[] become dL/dF, the others stay A for
// add_rows_kernel.  Bound by the latency of one workgroup's loads: kSumLoads in
// flight per thread.  90 000 spaxels: 49 us, 91 with one in flight and every
// spaxel's division here.
__global__ void __launch_bounds__(kSelThreads) noise_coef_kernel(
    int n, const float* __restrict__ F, const float* __restrict__ s2n,
    const rbx_noise_stats* __restrict__ stats, double* __restrict__ dots) {
  __shared__ double sm[kSelThreads / kWave];
  const rbx_noise_stats st = *stats;
  if (!live(st)) return;
  double acc[kSumLoads] = {};
  for (int64_t base = 0; base < n; base += kSumLoads * kSelThreads) {
    double a[kSumLoads];
    float s[kSumLoads];
#pragma unroll
    for (int u = 0; u < kSumLoads; ++u) {
      const int64_t p = base + u * kSelThreads + threadIdx.x;
      a[u] = p < n ? dots[p] : 0.0;
      s[u] = p < n ? s2n[p] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kSumLoads; ++u) acc[u] += a[u] * double(s[u]);
  }
  double sum = 0.0;
#pragma unroll
  for (int u = 0; u < kSumLoads; ++u) sum += acc[u];
  const double dM = block_sum(sum, sm) / (2.0 * double(st.median));
  if (threadIdx.x == 0 && has_median_spaxels(st, n)) {
    const int lo = st.median_lo, hi = st.median_hi;
    const double d_lo = flux_gradient(dots[lo], s2n[lo], F[lo]) + 0.5 * dM;
    const double d_hi = lo == hi ? d_lo + 0.5 * dM
                                 : flux_gradient(dots[hi], s2n[hi], F[hi]) + 0.5 * dM;
    dots[lo] = d_lo;
    dots[hi] = d_hi;
  }
}

// Adjoint, last pass: dcube[p, l] += dL/dF[p] (the flux path).  M = 0 (some
// spaxel without positive flux) leaves the S map identically 0: nothing to
// add.  Bound by HBM (300 x 300 x 1369: 191 us): 205 us, 326 with 4-byte accesses.
__global__ void __launch_bounds__(kRowThreads) add_rows_kernel(
    float* __restrict__ dcube, int n_spaxel, int nt, uint32_t n_items, uint32_t segs, int seg,
    const float* __restrict__ F, const float* __restrict__ s2n,
    const rbx_noise_stats* __restrict__ stats, const double* __restrict__ dots) {
  const rbx_noise_stats st = *stats;
  if (!live(st)) return;
  const bool medians = has_median_spaxels(st, n_spaxel);
  const int lane = threadIdx.x & (kWave - 1);
  for (uint64_t item = first_item(); item < n_items; item += item_stride()) {
    const RowItem it = row_item(uint32_t(item), segs, seg, nt);
    const bool at_median = medians && (it.p == st.median_lo || it.p == st.median_hi);
    const double d = dots[it.p];
    const float b = float(at_median ? d : flux_gradient(d, s2n[it.p], F[it.p]));
    float* row = dcube + int64_t(it.p) * nt;
    quads(it.l0, it.l1, lane, kWave, [&](int l, int n) {
      float v[4];
      load4(v, row + l, n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += b;
      store4(row + l, v, n);
    });
  }
}

// Segments of a row: the fewest of at most kItemBins bins, of equal length up
// to a multiple of 4.
struct RowSegs {
  uint32_t segs, items;
  int seg;
};
RowSegs row_segs(int32_t n_spaxel, int32_t n_target) {
  const uint32_t segs = (uint32_t(n_target) + kItemBins - 1) / kItemBins;
  const uint32_t seg = ((uint32_t(n_target) + segs - 1) / segs + 3) / 4 * 4;
  return {segs, uint32_t(n_spaxel) * segs, int(seg)};
}

// Calls f(true_type) for uniform draws, else f(false_type).
template <class F>
void with_distribution(int32_t distribution, F&& f) {
  if (distribution == RBX_NOISE_UNIFORM)
    f(std::true_type{});
  else
    f(std::false_type{});
}

int row_grid(int n_spaxel) { return n_spaxel < (1 << 16) ? n_spaxel : (1 << 16); }

// Workgroups of the elementwise passes: four items each.
int item_blocks(uint32_t n_items) {
  const uint32_t blocks = (n_items + 3u) / 4u;
  return blocks < (1u << 20) ? int(blocks) : (1 << 20);
}

int check_noise_args(const char* who, int32_t n_spaxel, int32_t n_target, int32_t distribution) {
  if (n_spaxel < 1 || n_target < 1)
    return failf(RBX_EINVAL, "%s: empty datacube (%d spaxels x %d bins)", who, n_spaxel, n_target);
  if (distribution != RBX_NOISE_NORMAL && distribution != RBX_NOISE_UNIFORM)
    return failf(RBX_EINVAL, "%s: unknown noise distribution %d (0 = normal, 1 = uniform)", who,
                 distribution);
  if (uint64_t(n_spaxel) * ((uint64_t(n_target) + 1023) / 1024) >= (uint64_t(1) << 32))
    return failf(RBX_EINVAL, "%s: datacube too large", who);
  return RBX_OK;
}

}  // namespace rbx

extern "C" {

int rbx_noise_sample(int64_t n, uint64_t seed, int32_t distribution, float* out, void* stream) {
  using namespace rbx;
  if (n < 0 || (n > 0 && !out)) return fail(RBX_EINVAL, "rbx_noise_sample: bad arguments");
  if (distribution != RBX_NOISE_NORMAL && distribution != RBX_NOISE_UNIFORM)
    return failf(RBX_EINVAL, "rbx_noise_sample: unknown noise distribution %d", distribution);
  if (n == 0) return RBX_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > (1 << 20)) blocks = 1 << 20;
  with_distribution(distribution, [&](auto u) {
    hipLaunchKernelGGL(noise_sample_kernel<decltype(u)::value>, dim3(unsigned(blocks)), dim3(256), 0,
                       as_stream(stream), n, key_of(seed), out);
  });
  return check_launch("rbx_noise_sample");
}

size_t rbx_noise_workspace_size(int32_t n_spaxel) {
  return n_spaxel > 0 ? size_t(n_spaxel) * sizeof(double) : 0;
}

int rbx_apply_noise(const float* cube, int32_t n_spaxel, int32_t n_target,
                    const float* signal_to_noise, uint64_t seed, int32_t distribution,
                    float* flux, float* s2n, rbx_noise_stats* stats, float* out, void* stream) {
  using namespace rbx;
  if (int rc = check_noise_args("rbx_apply_noise", n_spaxel, n_target, distribution)) return rc;
  if (!cube || !signal_to_noise || !flux || !s2n || !stats || !out)
    return fail(RBX_EINVAL, "rbx_apply_noise: null pointer");
  hipStream_t st = as_stream(stream);
  const NoiseKey key = key_of(seed);
  hipLaunchKernelGGL(flux_rows_kernel, dim3(row_grid(n_spaxel)), dim3(kRowThreads), 0, st, cube,
                     n_spaxel, n_target, flux);
  // up to kSelLoads spaxels a thread stay in its registers
  if (n_spaxel <= kSelLoads * kSelThreads)
    hipLaunchKernelGGL(noise_median_kernel<true>, dim3(1), dim3(kSelThreads), 0, st, flux, n_spaxel,
                       stats);
  else
    hipLaunchKernelGGL(noise_median_kernel<false>, dim3(1), dim3(kSelThreads), 0, st, flux, n_spaxel,
                       stats);
  const RowSegs r = row_segs(n_spaxel, n_target);
  with_distribution(distribution, [&](auto u) {
    hipLaunchKernelGGL(add_noise_kernel<decltype(u)::value>, dim3(item_blocks(r.items)),
                       dim3(kRowThreads), 0, st, cube, n_target, r.items, r.segs, r.seg, flux,
                       signal_to_noise, stats, key, s2n, out);
  });
  return check_launch("rbx_apply_noise");
}

int rbx_apply_noise_bwd(const float* cube, const float* dout, int32_t n_spaxel, int32_t n_target,
                        const float* flux, const float* s2n, const rbx_noise_stats* stats,
                        uint64_t seed, int32_t distribution, void* workspace,
                        size_t workspace_bytes, float* dcube, void* stream) {
  using namespace rbx;
  if (int rc = check_noise_args("rbx_apply_noise_bwd", n_spaxel, n_target, distribution))
    return rc;
  if (!cube || !dout || !flux || !s2n || !stats || !dcube || !workspace)
    return fail(RBX_EINVAL, "rbx_apply_noise_bwd: null pointer");
  if (workspace_bytes < rbx_noise_workspace_size(n_spaxel))
    return failf(RBX_EWORKSPACE, "rbx_apply_noise_bwd: workspace of %zu bytes, %zu needed",
                 workspace_bytes, rbx_noise_workspace_size(n_spaxel));
  hipStream_t st = as_stream(stream);
  const NoiseKey key = key_of(seed);
  double* dots = static_cast<double*>(workspace);
  // a workgroup per row while the rows alone leave the device short of
  // wavefronts (50 x 50 x 3721: 38 us, 53 with one each), else a wavefront per
  // row (300 x 300 x 1369: 342 us, 398 with four, 450 with one bin a thread at a time)
  with_distribution(distribution, [&](auto u) {
    constexpr bool kU = decltype(u)::value;
    if (n_spaxel < kFewRows)
      hipLaunchKernelGGL((noise_bwd_rows_kernel<4, kU>), dim3(row_grid(n_spaxel)), dim3(kRowThreads),
                         0, st, cube, dout, n_spaxel, n_target, s2n, key, dots, dcube);
    else
      hipLaunchKernelGGL((noise_bwd_rows_kernel<1, kU>), dim3(row_grid((n_spaxel + 3) / 4)),
                         dim3(kRowThreads), 0, st, cube, dout, n_spaxel, n_target, s2n, key, dots,
                         dcube);
  });
  hipLaunchKernelGGL(noise_coef_kernel, dim3(1), dim3(kSelThreads), 0, st, n_spaxel, flux, s2n,
                     stats, dots);
  const RowSegs r = row_segs(n_spaxel, n_target);
  hipLaunchKernelGGL(add_rows_kernel, dim3(item_blocks(r.items)), dim3(kRowThreads), 0, st, dcube,
                     n_spaxel, n_target, r.items, r.segs, r.seg, flux, s2n, stats, dots);
  return check_launch("rbx_apply_noise_bwd");
}

}  // extern "C"
