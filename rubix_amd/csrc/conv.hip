// PSF and LSF convolutions over the (ny, nx, n_lambda) datacube.
//
// convolve_psf (rubix/telescope/psf/psf.py:33-58) convolves every lambda plane
// with a 2D kernel, mode "same"; the Gaussian kernel of
// rubix/telescope/psf/kernels.py:5-31 is outer(g, g) with g the normalised 1D
// Gaussian, so it runs as two 1D passes (x then y).  convolve_lsf
// (rubix/telescope/lsf/lsf.py:29-105) is a 25-tap full convolution along
// lambda cropped at the extend factor.  Both are one kernel: a 1D
// convolution along the middle axis of an (n_outer, n_axis, n_inner) view.
// Work is split so that index arithmetic happens once per workgroup item,
// never per element (64-bit division per element would dominate):
// * conv_cols_kernel (n_inner > 1 and one of the instantiated tap counts, the
//   spatial PSF passes): a wavefront walks 64 contiguous inner elements along
//   a segment of the axis with the last M inputs in registers, so each input
//   is read once and a tap is one multiply-add, without LDS.
// * conv_tile_kernel (other tap counts, an axis of at most kTileAxis): item =
//   a block of 64 contiguous inner elements with the whole axis staged in LDS.
// * conv_lines_kernel (n_inner > 1, longer axes): item = one (outer, axis)
//   line and a chunk of up to kLineChunk contiguous inner elements; threads
//   run along the contiguous inner axis.
// * conv_rows_kernel (n_inner == 1, the LSF along lambda): item = a segment
//   of at most kSeg outputs of one row; the segment's inputs plus the kernel's
//   halo are staged in LDS once, a thread forms four consecutive outputs and
//   reads 16 bytes of LDS per four taps.
// The batched PSF (rbx_conv_batch) walks the lines of all galaxies as
// conv_cols_kernel does.  Every output sums taps in the same order
// t = 0 .. m-1 as the flat definition.
#include <mutex>
#include <type_traits>

#include "rbx_common.h"

namespace rbx {

__global__ void conv_axis_kernel(const float* __restrict__ in, float* __restrict__ out,
                                 int64_t n_outer, int n_axis, int64_t n_inner,
                                 const float* __restrict__ taps, int n_taps, int start) {
  const int64_t total = n_outer * n_axis * n_inner;
  for (int64_t idx = gtid(); idx < total; idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = idx % n_inner;
    const int64_t ox = idx / n_inner;
    const int x = int(ox % n_axis);
    const int64_t o = ox / n_axis;
    const float* src = in + o * n_axis * n_inner + i;
    float acc = 0.f;
    for (int t = 0; t < n_taps; ++t) {
      const int xs = x + start - t;
      if (xs >= 0 && xs < n_axis) acc += taps[t] * src[int64_t(xs) * n_inner];
    }
    out[idx] = acc;
  }
}

__global__ void conv2d_planes_kernel(const float* __restrict__ in, float* __restrict__ out,
                                     int ny, int nx, int nl, const float* __restrict__ K,
                                     int ky, int kx, int sy, int sx) {
  const int64_t total = int64_t(ny) * nx * nl;
  for (int64_t idx = gtid(); idx < total; idx += int64_t(gridDim.x) * blockDim.x) {
    const int l = int(idx % nl);
    const int64_t yx = idx / nl;
    const int x = int(yx % nx);
    const int y = int(yx / nx);
    float acc = 0.f;
    for (int a = 0; a < ky; ++a) {
      const int ys = y + sy - a;
      if (ys < 0 || ys >= ny) continue;
      for (int b = 0; b < kx; ++b) {
        const int xs = x + sx - b;
        if (xs < 0 || xs >= nx) continue;
        acc += K[a * kx + b] * in[(int64_t(ys) * nx + xs) * nl + l];
      }
    }
    out[idx] = acc;
  }
}

constexpr int kDotThreads = 256;
constexpr int kDotBlocksMax = 4096;
constexpr int kLineChunk = 1024;  // inner elements per line item
constexpr int kSeg = 1024;        // most outputs per row item of the LSF
constexpr int kHalo = 256;        // taps - 1 supported by the row kernel
constexpr int kTileAxis = 240;    // longest axis the tiled line kernels stage (60 KB of LDS)

// One 1D convolution item of a line: out[o, x, i0 + k] for k < len.
template <class Acc, class Tap>
__device__ inline Acc line_tap_sum(const float* __restrict__ src, int x, int n_axis,
                                   int64_t n_inner, const Tap* __restrict__ taps, int n_taps,
                                   int start) {
  Acc acc = 0;
  for (int t = 0; t < n_taps; ++t) {
    const int xs = x + start - t;
    if (xs >= 0 && xs < n_axis) acc += Acc(taps[t]) * Acc(src[int64_t(xs) * n_inner]);
  }
  return acc;
}

// Items: (o, x, chunk) with chunk fastest.  Grid-strided.
__global__ void __launch_bounds__(256) conv_lines_kernel(
    const float* __restrict__ in, float* __restrict__ out, int64_t n_outer, int n_axis,
    int64_t n_inner, const float* __restrict__ taps, int n_taps, int start, int64_t n_chunks,
    int64_t n_items) {
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t c = item % n_chunks;
    const int64_t ox = item / n_chunks;
    const int x = int(ox % n_axis);
    const int64_t o = ox / n_axis;
    const int64_t i0 = c * kLineChunk;
    const int64_t i1 = i0 + kLineChunk < n_inner ? i0 + kLineChunk : n_inner;
    const float* base = in + o * n_axis * n_inner;
    float* dst = out + (o * n_axis + x) * n_inner;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += blockDim.x)
      dst[i] = line_tap_sum<float>(base + i, x, n_axis, n_inner, taps, n_taps, start);
  }
}

// Rows u0, u0 + 4, u0 + 8, u0 + 12 of the convolution of a staged tile (rows
// 0 .. n-1 of 64 lanes): for each output the taps t = 0 .. m-1 in order,
// rows outside [0, n) skipped (zero padding).  Four independent sums per
// lane hide the LDS latency; each output's own order is unchanged.
template <class Acc, class Tap>
__device__ inline void tile_conv4(const float* tile, int lane, int n, const Tap* __restrict__ taps,
                                  int m, int start, int u0, Acc acc[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = Acc(0);
  for (int t = 0; t < m; ++t) {
    const Acc tv = Acc(taps[t]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int us = u0 + 4 * r + start - t;
      if (us >= 0 && us < n) acc[r] += tv * Acc(tile[us * 64 + lane]);
    }
  }
}

// Items: (o, block of 64 contiguous inner elements).  The workgroup stages
// the block's whole axis (n_axis x 64 floats, dynamic LDS) once with
// coalesced loads; wavefront w then forms the outputs x = w, w + 4, ...
// from LDS, the taps in the order t = 0 .. m-1 of line_tap_sum (same
// values).  Every input element is read from memory once instead of once
// per tap.  n_axis <= kTileAxis.
__global__ void __launch_bounds__(256) conv_tile_kernel(
    const float* __restrict__ in, float* __restrict__ out, int n_axis, int64_t n_inner,
    const float* __restrict__ taps, int n_taps, int start, int64_t n_blocks, int64_t n_items) {
  extern __shared__ float tile[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t o = item / n_blocks;
    const int64_t i = (item - o * n_blocks) * 64 + lane;
    const bool ok = i < n_inner;
    const int64_t base = o * n_axis * n_inner + (ok ? i : 0);
    __syncthreads();  // the previous item's reads are done
    for (int x = w; x < n_axis; x += 4) tile[x * 64 + lane] = ok ? in[base + int64_t(x) * n_inner] : 0.f;
    __syncthreads();
    for (int x0 = w; x0 < n_axis; x0 += 16) {
      float acc[4];
      tile_conv4<float>(tile, lane, n_axis, taps, n_taps, start, x0, acc);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = x0 + 4 * r;
        if (ok && x < n_axis) out[base + int64_t(x) * n_inner] = acc[r];
      }
    }
  }
}

// One wavefront's lane of a convolution along a strided axis: outputs
// x in [x0, x1) of the column at `src` (element xs at src + xs * stride, zero
// outside [0, n)).  The last M inputs stay in registers (a ring whose places
// are fixed by unrolling M steps), the next M are loaded ahead, and
// sink(x, sum_t taps[t] in[x + start - t]) gets every output, its taps in the
// order t = 0 .. M-1.  x0, x1 are wave-uniform; a lane without a column
// (ok false) reads nothing.
template <int M, class Acc, class Tap, class Sink>
__device__ inline void column_walk(const float* __restrict__ src, int64_t stride, int n, bool ok,
                                   int x0, int x1, int start, const Tap* __restrict__ taps,
                                   Sink&& sink) {
  Acc tap[M], ring[M];
  float next[M];
#pragma unroll
  for (int t = 0; t < M; ++t) tap[t] = Acc(taps[t]);
  auto load = [&](int xs) { return ok && xs >= 0 && xs < n ? src[int64_t(xs) * stride] : 0.f; };
  // ring[u] holds the newest input x + start of step u (mod M)
#pragma unroll
  for (int u = 1; u < M; ++u) ring[u] = Acc(load(x0 + start - M + u));
#pragma unroll
  for (int u = 0; u < M; ++u) next[u] = load(x0 + start + u);
  for (int xb = x0; xb < x1; xb += M) {
    float cur[M];
#pragma unroll
    for (int u = 0; u < M; ++u) cur[u] = next[u];
    if (xb + M < x1) {
#pragma unroll
      for (int u = 0; u < M; ++u) next[u] = load(xb + M + start + u);
    }
#pragma unroll
    for (int u = 0; u < M; ++u) {
      ring[u] = Acc(cur[u]);
      if (xb + u < x1) {
        Acc acc = Acc(0);
#pragma unroll
        for (int t = 0; t < M; ++t) acc += tap[t] * ring[(u - t + M) % M];
        sink(xb + u, acc);
      }
    }
  }
}

// The adjoint's walk for a centred kernel (start = (M - 1) / 2, M odd) along
// the column of a (the incoming gradient) and b (the forward's input) at once:
// emit(x, sum_t rev[t] a[x + start - t]) is the transposed convolution, and
// the sum of a[x] sum_t dtaps[t] b[x + start - t] (double) is returned; a[x] is in
// the ring.  a and b are read once for both.
template <int M, class Emit>
__device__ inline double column_walk_bwd(const float* __restrict__ a, const float* __restrict__ b,
                                         int64_t stride, int n, bool ok, int x0, int x1,
                                         const float* __restrict__ rev,
                                         const double* __restrict__ dtaps, Emit&& emit) {
  constexpr int start = (M - 1) / 2;
  float ring[M], next_a[M], next_b[M];
  double ringd[M];
  double dot = 0.0;
  auto inside = [&](int xs) { return ok && xs >= 0 && xs < n; };
  auto load = [&](const float* src, int xs) { return inside(xs) ? src[int64_t(xs) * stride] : 0.f; };
#pragma unroll
  for (int u = 1; u < M; ++u) {
    ring[u] = load(a, x0 + start - M + u);
    ringd[u] = double(load(b, x0 + start - M + u));
  }
#pragma unroll
  for (int u = 0; u < M; ++u) {
    next_a[u] = load(a, x0 + start + u);
    next_b[u] = load(b, x0 + start + u);
  }
  for (int xb = x0; xb < x1; xb += M) {
    float cur_a[M], cur_b[M];
#pragma unroll
    for (int u = 0; u < M; ++u) {
      cur_a[u] = next_a[u];
      cur_b[u] = next_b[u];
    }
    if (xb + M < x1) {
#pragma unroll
      for (int u = 0; u < M; ++u) {
        next_a[u] = load(a, xb + M + start + u);
        next_b[u] = load(b, xb + M + start + u);
      }
    }
#pragma unroll
    for (int u = 0; u < M; ++u) {
      ring[u] = cur_a[u];
      ringd[u] = double(cur_b[u]);
      if (xb + u < x1) {
        float acc = 0.f;
        double c = 0.0;
#pragma unroll
        for (int t = 0; t < M; ++t) {
          acc += rev[t] * ring[(u - t + M) % M];
          c += dtaps[t] * ringd[(u - t + M) % M];
        }
        emit(xb + u, acc);
        dot += double(ring[(u - start + M) % M]) * c;
      }
    }
  }
  return ok ? dot : 0.0;
}

// Items, one per wavefront: (o, block of 64 contiguous inner elements,
// segment of the axis), the segments of a block next to each other (they share
// the halo in cache).  Bound by HBM: a 15-tap pass over 50 x 50 x 3721 (74 MB)
// took 43 us from LDS and takes 19, an 11-tap pass over 300 x 300 x 1369
// (0.99 GB, the axis too long for LDS) 1.3 ms and 0.25 (3.9 TB/s).
template <int M>
__global__ void __launch_bounds__(256) conv_cols_kernel(
    const float* __restrict__ in, float* __restrict__ out, int n_axis, int64_t n_inner,
    const float* __restrict__ taps, int start, int64_t n_blocks, int n_segs, int seg,
    int64_t n_items) {
  const int lane = threadIdx.x & 63;
  const int64_t first = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t item = first; item < n_items; item += int64_t(gridDim.x) * 4) {
    const int64_t blk = item / n_segs;
    const int x0 = int(item - blk * n_segs) * seg;
    const int x1 = x0 + seg < n_axis ? x0 + seg : n_axis;
    const int64_t o = blk / n_blocks;
    const int64_t i = (blk - o * n_blocks) * 64 + lane;
    const bool ok = i < n_inner;
    const int64_t base = o * n_axis * n_inner + (ok ? i : 0);
    column_walk<M, float>(in + base, n_inner, n_axis, ok, x0, x1, start, taps,
                          [&](int x, float v) {
                            if (ok) out[base + int64_t(x) * n_inner] = v;
                          });
  }
}

// The taps of a row pass in LDS, reversed: tap[p] = taps[m - 1 - p].  (Read as
// uniform global loads, each tap waited a scalar-cache round trip.)
template <class Tap>
__device__ inline void stage_taps(Tap* tap, const Tap* __restrict__ taps, int m) {
  for (int p = threadIdx.x; p < m; p += blockDim.x) tap[p] = taps[m - 1 - p];
}

// Four consecutive outputs v .. v + 3 of a staged row: sum_t taps[t]
// lds[v + e + m - 1 - t], the taps in the order t = 0 .. m-1 (tap[] from its
// end), 16 bytes of LDS per four of them (v a multiple of 4; lds holds 4
// floats past v + m + 2).
template <class Acc, class Tap>
__device__ inline void row_conv4(const float* lds, int v, const Tap* tap, int m, Acc (&acc)[4]) {
  const float4* q4 = reinterpret_cast<const float4*>(lds + v);
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = Acc(0);
  int q = (m - 1) >> 2;
  float4 hi = q4[q + 1];
  float4 lo = q4[q];
  auto window = [&](Acc (&w)[8]) {
    w[0] = Acc(lo.x); w[1] = Acc(lo.y); w[2] = Acc(lo.z); w[3] = Acc(lo.w);
    w[4] = Acc(hi.x); w[5] = Acc(hi.y); w[6] = Acc(hi.z); w[7] = Acc(hi.w);
  };
  {  // the last one to four places
    Acc w[8];
    window(w);
#pragma unroll
    for (int b = 3; b >= 0; --b) {
      if (4 * q + b < m) {
        const Acc tv = Acc(tap[4 * q + b]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += tv * w[b + e];
      }
    }
  }
  while (--q >= 0) {
    hi = lo;
    lo = q4[q];
    Acc t4[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) t4[b] = Acc(tap[4 * q + b]);
    Acc w[8];
    window(w);
#pragma unroll
    for (int b = 3; b >= 0; --b) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += t4[b] * w[b + e];
    }
  }
}

// A staged row segment of the LDS buffers below: a thread's share of
// row[off + k], k < len, 0 outside [0, n), and 4 more zeros behind.
constexpr int kRowLoads = (kSeg + kHalo + 4 + 255) / 256;
__device__ inline void load_row(float* v, const float* __restrict__ row, int off, int len, int n) {
#pragma unroll
  for (int u = 0; u < kRowLoads; ++u) {
    const int k = threadIdx.x + 256 * u, xs = off + k;
    v[u] = (k < len && xs >= 0 && xs < n) ? row[xs] : 0.f;
  }
}
__device__ inline void store_row(float* lds, const float* v, int len) {
#pragma unroll
  for (int u = 0; u < kRowLoads; ++u) {
    const int k = threadIdx.x + 256 * u;
    if (k < len + 4) lds[k] = v[u];
  }
}

// lds[k] = row[off + k] for k < len, 0 outside [0, n); 4 more zeros behind.
__device__ inline void stage_row(float* lds, const float* __restrict__ row, int off, int len, int n) {
  float v[kRowLoads];  // every load in flight before the first is stored
  load_row(v, row, off, len, n);
  __syncthreads();
  store_row(lds, v, len);
  __syncthreads();
}

// Four consecutive floats at any 4-byte alignment (one 16-byte access).
struct alignas(4) Float4u {
  float v[4];
};

// Items: (row o, segment of `seg` outputs, a multiple of 4 up to kSeg) of a
// row-contiguous convolution (n_inner == 1).
// lds[k] = in[o, x0 + start - (m - 1) + k] (0 outside the row: a tap past the
// row's end adds taps[t] * 0), so out[o, x0 + v] = sum_t taps[t] lds[v + m - 1 - t].
// 25 taps over 50 x 50 x 3721: 26 us with one LDS read per tap and output, 17
// now (HBM: 14).
__global__ void __launch_bounds__(256) conv_rows_kernel(
    const float* __restrict__ in, float* __restrict__ out, int n_axis,
    const float* __restrict__ taps, int n_taps, int start, int64_t n_seg, int seg,
    int64_t n_items) {
  __shared__ __align__(16) float lds[kSeg + kHalo + 8];
  __shared__ __align__(16) float tap[kHalo + 1];
  stage_taps(tap, taps, n_taps);
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t o = item / n_seg;
    const int x0 = int(item - o * n_seg) * seg;
    const int len = n_axis - x0 < seg ? n_axis - x0 : seg;
    stage_row(lds, in + o * n_axis, x0 + start - (n_taps - 1), (len + 3) / 4 * 4 + n_taps - 1, n_axis);
    const int v = 4 * threadIdx.x;
    if (v >= len) continue;
    float acc[4];
    row_conv4<float>(lds, v, tap, n_taps, acc);
    float* dst = out + o * n_axis + x0 + v;
    if (v + 4 <= len) {
      *reinterpret_cast<Float4u*>(dst) = {{acc[0], acc[1], acc[2], acc[3]}};
    } else {
      for (int e = 0; v + e < len; ++e) dst[e] = e == 0 ? acc[0] : (e == 1 ? acc[1] : acc[2]);
    }
  }
}

// Fixed-order block reduction of one double per thread into partial[block].
__device__ inline void block_partial(double acc, double* sm, double* __restrict__ partial) {
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int off = kDotThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) sm[threadIdx.x] += sm[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sm[0];
}

// sum(a * conv(b)) per block, line items (n_inner > 1), double taps.
__global__ void __launch_bounds__(kDotThreads) conv_dot_lines_kernel(
    const float* __restrict__ a, const float* __restrict__ b, int64_t n_outer, int n_axis,
    int64_t n_inner, const double* __restrict__ taps, int n_taps, int start, int64_t n_chunks,
    int64_t n_items, double* __restrict__ partial) {
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t c = item % n_chunks;
    const int64_t ox = item / n_chunks;
    const int x = int(ox % n_axis);
    const int64_t o = ox / n_axis;
    const int64_t i0 = c * kLineChunk;
    const int64_t i1 = i0 + kLineChunk < n_inner ? i0 + kLineChunk : n_inner;
    const float* base = b + o * n_axis * n_inner;
    const float* av = a + (o * n_axis + x) * n_inner;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += blockDim.x)
      acc += double(av[i]) * line_tap_sum<double>(base + i, x, n_axis, n_inner, taps, n_taps, start);
  }
  block_partial(acc, sm, partial);
}

// sum(a * conv(b)) per block over conv_cols_kernel's items, double taps.
template <int M>
__global__ void __launch_bounds__(kDotThreads) conv_dot_cols_kernel(
    const float* __restrict__ a, const float* __restrict__ b, int n_axis, int64_t n_inner,
    const double* __restrict__ taps, int start, int64_t n_blocks, int n_segs, int seg,
    int64_t n_items, double* __restrict__ partial) {
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  const int lane = threadIdx.x & 63;
  const int64_t first = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t item = first; item < n_items; item += int64_t(gridDim.x) * 4) {
    const int64_t blk = item / n_segs;
    const int x0 = int(item - blk * n_segs) * seg;
    const int x1 = x0 + seg < n_axis ? x0 + seg : n_axis;
    const int64_t o = blk / n_blocks;
    const int64_t i = (blk - o * n_blocks) * 64 + lane;
    const bool ok = i < n_inner;
    const int64_t base = o * n_axis * n_inner + (ok ? i : 0);
    column_walk<M, double>(b + base, n_inner, n_axis, ok, x0, x1, start, taps,
                           [&](int x, double v) {
                             if (ok) acc += double(a[base + int64_t(x) * n_inner]) * v;
                           });
  }
  block_partial(acc, sm, partial);
}

// sum(a * conv(b)) per block, rows (n_inner == 1), double taps.
__global__ void __launch_bounds__(kDotThreads) conv_dot_rows_kernel(
    const float* __restrict__ a, const float* __restrict__ b, int n_axis,
    const double* __restrict__ taps, int n_taps, int start, int64_t n_seg, int seg,
    int64_t n_items, double* __restrict__ partial) {
  __shared__ __align__(16) float lds[kSeg + kHalo + 8];
  __shared__ __align__(16) double tap[kHalo + 1];
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  stage_taps(tap, taps, n_taps);
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t o = item / n_seg;
    const int x0 = int(item - o * n_seg) * seg;
    const int len = n_axis - x0 < seg ? n_axis - x0 : seg;
    stage_row(lds, b + o * n_axis, x0 + start - (n_taps - 1), (len + 3) / 4 * 4 + n_taps - 1, n_axis);
    const int v = 4 * threadIdx.x;
    if (v >= len) continue;
    double c[4];
    row_conv4<double>(lds, v, tap, n_taps, c);
    const float* av = a + o * n_axis + x0 + v;
    if (v + 4 <= len) {
      const Float4u a4 = *reinterpret_cast<const Float4u*>(av);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc += double(a4.v[e]) * c[e];
    } else {
      for (int e = 0; v + e < len; ++e)
        acc += double(av[e]) * (e == 0 ? c[0] : (e == 1 ? c[1] : c[2]));
    }
  }
  block_partial(acc, sm, partial);
}

// conv_cols_kernel and conv_dot_cols_kernel of the adjoint in one pass over a
// and b.  Bound by HBM: two cubes read and one written, where the two passes
// read three.  300 x 300 x 1369, 11 taps: 397 us, 490 for the two.  Up to 15 taps:
// the two rings take 8 registers per tap, and past 128 of them fewer waves are
// resident than the loads need.
template <int M>
__global__ void __launch_bounds__(kDotThreads) conv_bwd_cols_kernel(
    const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ out, int n_axis,
    int64_t n_inner, const float* __restrict__ rev, const double* __restrict__ dtaps,
    int64_t n_blocks, int n_segs, int seg, int64_t n_items, double* __restrict__ partial) {
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  const int lane = threadIdx.x & 63;
  const int64_t first = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t item = first; item < n_items; item += int64_t(gridDim.x) * 4) {
    const int64_t blk = item / n_segs;
    const int x0 = int(item - blk * n_segs) * seg;
    const int x1 = x0 + seg < n_axis ? x0 + seg : n_axis;
    const int64_t o = blk / n_blocks;
    const int64_t i = (blk - o * n_blocks) * 64 + lane;
    const bool ok = i < n_inner;
    const int64_t base = o * n_axis * n_inner + (ok ? i : 0);
    acc += column_walk_bwd<M>(a + base, b + base, n_inner, n_axis, ok, x0, x1, rev, dtaps,
                              [&](int x, float v) {
                                if (ok) out[base + int64_t(x) * n_inner] = v;
                              });
  }
  block_partial(acc, sm, partial);
}

// conv_rows_kernel and conv_dot_rows_kernel of the adjoint in one pass:
// out = conv(a, rev) from rstart = m - 1 - start, and sum(a * conv(b, dtaps)).
// The workgroup's LDS holds one item, so the next one's loads are issued before
// this one's arithmetic (25 float and 25 double multiply-adds an output).
// 300 x 300 x 1369, 25 taps: 555 us; 630 without the loads ahead, 620 in two passes.
__global__ void __launch_bounds__(kDotThreads) conv_bwd_rows_kernel(
    const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ out, int n_axis,
    const float* __restrict__ rev, const double* __restrict__ dtaps, int n_taps, int start,
    int64_t n_seg, int seg, int64_t n_items, double* __restrict__ partial) {
  __shared__ __align__(16) float la[kSeg + kHalo + 8];
  __shared__ __align__(16) float lb[kSeg + kHalo + 8];
  __shared__ __align__(16) float tap[kHalo + 1];
  __shared__ __align__(16) double dtap[kHalo + 1];
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  stage_taps(tap, rev, n_taps);
  stage_taps(dtap, dtaps, n_taps);
  const int rstart = n_taps - 1 - start;
  // the next item's segments are loaded while this one's are worked on
  float na[kRowLoads], nb[kRowLoads];
  auto geometry = [&](int64_t item, int64_t* o, int* x0, int* len) {
    *o = item / n_seg;
    *x0 = int(item - *o * n_seg) * seg;
    *len = n_axis - *x0 < seg ? n_axis - *x0 : seg;
    return (*len + 3) / 4 * 4 + n_taps - 1;
  };
  int64_t o;
  int x0, len;
  if (blockIdx.x < n_items) {
    const int span = geometry(blockIdx.x, &o, &x0, &len);
    load_row(na, a + o * n_axis, x0 + rstart - (n_taps - 1), span, n_axis);
    load_row(nb, b + o * n_axis, x0 + start - (n_taps - 1), span, n_axis);
  }
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int span = geometry(item, &o, &x0, &len);
    __syncthreads();
    store_row(la, na, span);
    store_row(lb, nb, span);
    __syncthreads();
    if (item + gridDim.x < n_items) {
      int64_t on;
      int xn, ln;
      const int sn = geometry(item + gridDim.x, &on, &xn, &ln);
      load_row(na, a + on * n_axis, xn + rstart - (n_taps - 1), sn, n_axis);
      load_row(nb, b + on * n_axis, xn + start - (n_taps - 1), sn, n_axis);
    }
    const int v = 4 * threadIdx.x;
    if (v >= len) continue;
    float r[4];
    row_conv4<float>(la, v, tap, n_taps, r);
    double c[4];
    row_conv4<double>(lb, v, dtap, n_taps, c);
    float* dst = out + o * n_axis + x0 + v;
    const float* av = la + v + start;  // a[x0 + v]: la starts at x0 - start
    if (v + 4 <= len) {
      *reinterpret_cast<Float4u*>(dst) = {{r[0], r[1], r[2], r[3]}};
#pragma unroll
      for (int e = 0; e < 4; ++e) acc += double(av[e]) * c[e];
    } else {
      for (int e = 0; v + e < len; ++e) {
        dst[e] = e == 0 ? r[0] : (e == 1 ? r[1] : r[2]);
        acc += double(av[e]) * (e == 0 ? c[0] : (e == 1 ? c[1] : c[2]));
      }
    }
  }
  block_partial(acc, sm, partial);
}

// sum(a * conv(b)) per block over tiled items (as conv_tile_kernel), double
// taps.  Each thread adds its outputs' a * conv(b) in item order.
__global__ void __launch_bounds__(kDotThreads) conv_dot_tile_kernel(
    const float* __restrict__ a, const float* __restrict__ b, int n_axis, int64_t n_inner,
    const double* __restrict__ taps, int n_taps, int start, int64_t n_blocks, int64_t n_items,
    double* __restrict__ partial) {
  extern __shared__ float tile[];
  __shared__ double sm[kDotThreads];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double acc = 0.0;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int64_t o = item / n_blocks;
    const int64_t i = (item - o * n_blocks) * 64 + lane;
    const bool ok = i < n_inner;
    const int64_t base = o * n_axis * n_inner + (ok ? i : 0);
    __syncthreads();
    for (int x = w; x < n_axis; x += 4) tile[x * 64 + lane] = ok ? b[base + int64_t(x) * n_inner] : 0.f;
    __syncthreads();
    if (ok) {
      for (int x0 = w; x0 < n_axis; x0 += 16) {
        double c[4];
        tile_conv4<double>(tile, lane, n_axis, taps, n_taps, start, x0, c);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int x = x0 + 4 * r;
          if (x < n_axis) acc += double(a[base + int64_t(x) * n_inner]) * c[r];
        }
      }
    }
  }
  block_partial(acc, sm, partial);
}

// Per-block partial of sum(a * conv_axis(b)) in double, fixed tree order.
// The sigma-derivative taps sum to zero, so conv(dtaps, b) cancels strongly:
// taps and the convolution are double.
__global__ void __launch_bounds__(kDotThreads) conv_dot_partial_kernel(
    const float* __restrict__ a, const float* __restrict__ b, int64_t n_outer, int n_axis,
    int64_t n_inner, const double* __restrict__ taps, int n_taps, int start,
    double* __restrict__ partial) {
  __shared__ double sm[kDotThreads];
  const int64_t total = n_outer * n_axis * n_inner;
  double acc = 0.0;
  for (int64_t idx = gtid(); idx < total; idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = idx % n_inner;
    const int64_t ox = idx / n_inner;
    const int x = int(ox % n_axis);
    const int64_t o = ox / n_axis;
    const float* src = b + o * n_axis * n_inner + i;
    double c = 0.0;
    for (int t = 0; t < n_taps; ++t) {
      const int xs = x + start - t;
      if (xs >= 0 && xs < n_axis) c += taps[t] * double(src[int64_t(xs) * n_inner]);
    }
    acc += double(a[idx]) * c;
  }
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int off = kDotThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) sm[threadIdx.x] += sm[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sm[0];
}

// result = the sum of the block partials in a fixed order, plus `add` (nullable);
// result32 (nullable) = the same in float.
__global__ void __launch_bounds__(kDotThreads) dot_final_kernel(const double* __restrict__ partial,
                                                                int nblk, const double* add,
                                                                double* result, float* result32) {
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  for (int k = threadIdx.x; k < nblk; k += kDotThreads) acc += partial[k];
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int off = kDotThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) sm[threadIdx.x] += sm[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double r = add ? *add + sm[0] : sm[0];
    *result = r;
    if (result32) *result32 = float(r);
  }
}

// ------------------------------------------------------------ Gaussian taps

// Normalised Gaussian g = exp(-x^2 / 2 sigma^2) / sum on the grid x, its
// reversed copy and dg/dsigma = g (x^2 / sigma^3 - sum_k g_k x_k^2 / sigma^3),
// all in double (taps rounded once to float).  One workgroup, sums in a fixed
// order.  As a dozen elementwise and reduction launches per PSF or LSF these
// were a third of a 10 k-star step.
template <class T>
__global__ void __launch_bounds__(kDotThreads) gauss_taps_kernel(const double* __restrict__ x, int n,
                                                                 const T* __restrict__ sigma,
                                                                 float* __restrict__ taps,
                                                                 float* __restrict__ reversed,
                                                                 double* __restrict__ dtaps) {
  __shared__ double sm[kDotThreads];
  const double s = double(*sigma);
  auto total = [&](double v) {
    __syncthreads();
    sm[threadIdx.x] = v;
    __syncthreads();
    for (int off = kDotThreads / 2; off > 0; off >>= 1) {
      if (threadIdx.x < off) sm[threadIdx.x] += sm[threadIdx.x + off];
      __syncthreads();
    }
    return sm[0];
  };
  auto bell = [&](int k) { return exp(-0.5 * x[k] * x[k] / (s * s)); };
  double e = 0.0, ex = 0.0;
  for (int k = threadIdx.x; k < n; k += kDotThreads) e += bell(k);
  const double sum = total(e);
  for (int k = threadIdx.x; k < n; k += kDotThreads) ex += bell(k) / sum * (x[k] * x[k] / (s * s * s));
  const double mean = total(ex);
  for (int k = threadIdx.x; k < n; k += kDotThreads) {
    const double g = bell(k) / sum;
    taps[k] = float(g);
    reversed[n - 1 - k] = float(g);
    dtaps[k] = g * (x[k] * x[k] / (s * s * s) - mean);
  }
}

// ------------------------------------------------------------ batches
//
// A batch cube stacks the (nb, nb, n_lambda) cubes of several galaxies row
// after row (rbx_galaxy: first row and nb of each).  One launch convolves
// every galaxy: each output element finds its galaxy by binary search over
// the (ascending) first rows, then runs the same 1D convolution inside that
// galaxy's grid with zero padding at its edges.

struct BatchPos {
  bool ok;      // the row belongs to a galaxy whose grid fits the batch
  int64_t base; // element of coordinate u = 0 along the convolved axis
  int64_t stride;
  int u, nb;
};

__device__ inline BatchPos batch_pos(const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows,
                                     int nt, int axis, int64_t idx) {
  BatchPos b;
  const int p = int(idx / nt);
  const int l = int(idx - int64_t(p) * nt);
  int lo = 0, hi = n_gal;  // last galaxy with spaxel_begin <= p
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (gal[mid].spaxel_begin <= p) lo = mid; else hi = mid;
  }
  const int64_t begin = gal[lo].spaxel_begin;
  const int nb = gal[lo].nb;
  const int64_t q = p - begin;
  b.nb = nb;
  b.ok = nb > 0 && q >= 0 && q < int64_t(nb) * nb && begin + int64_t(nb) * nb <= n_rows;
  if (!b.ok) {
    b.base = 0; b.stride = 0; b.u = 0;
    return b;
  }
  const int y = int(q / nb), x = int(q - int64_t(y) * nb);
  if (axis == 1) {
    b.u = x;
    b.stride = nt;
    b.base = (begin + int64_t(y) * nb) * nt + l;
  } else {
    b.u = y;
    b.stride = int64_t(nb) * nt;
    b.base = (begin + x) * nt + l;
  }
  return b;
}

// Row items: (spaxel row p of the batch cube, chunk of kLineChunk lambda);
// the galaxy and the row's (y, x) are found once per item.
__global__ void __launch_bounds__(256) conv_batch_kernel(
    const float* __restrict__ in, float* __restrict__ out, const rbx_galaxy* __restrict__ gal,
    int n_gal, int n_rows, int nt, int axis, const float* __restrict__ taps, int n_taps,
    int start, int n_chunks, int64_t n_items) {
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int p = int(item / n_chunks);
    const int l0 = int(item - int64_t(p) * n_chunks) * kLineChunk;
    const int l1 = l0 + kLineChunk < nt ? l0 + kLineChunk : nt;
    const BatchPos b = batch_pos(gal, n_gal, n_rows, nt, axis, int64_t(p) * nt);
    for (int l = l0 + threadIdx.x; l < l1; l += blockDim.x) {
      float acc = 0.f;
      if (b.ok) {
        for (int t = 0; t < n_taps; ++t) {
          const int us = b.u + start - t;
          if (us >= 0 && us < b.nb) acc += taps[t] * in[b.base + l + us * b.stride];
        }
      }
      out[int64_t(p) * nt + l] = acc;
    }
  }
}

// LDS-tiled batch passes.  A packed table (galaxy g's rows begin where
// galaxy g - 1's end, from row 0 to n_rows, every nb >= 1: what a batch
// layout builds) is convolved line by line: item = (line L, block of 64
// lambda), L counting the lines of galaxy 0, then galaxy 1, ...; the
// workgroup stages the line's nb x 64 inputs in LDS once (lines of at most
// kBatchTileAxis spaxels; longer ones read the inputs directly) and adds
// the taps in the order of conv_batch_kernel, so the values are the same.
// Each workgroup first builds the line prefix of the table in LDS and
// checks that it is packed; any other table runs the row items of
// conv_batch_kernel (rows of no galaxy get zeros).
constexpr int kBatchTileAxis = 100;
constexpr int kBatchGalMax = 512;  // galaxies the line prefix holds (host falls back above)

// lines[g] = number of lines of galaxies 0 .. g-1 (lines[n_gal] = total) and
// whether the table is packed; all threads of the workgroup return the same.
__device__ inline bool batch_line_prefix(const rbx_galaxy* __restrict__ gal, int n_gal,
                                         int n_rows, int* lines, int* part) {
  const int tid = threadIdx.x;
  const int per = (n_gal + 255) / 256;
  const int g0 = tid * per;
  int sum = 0, bad = 0;
  for (int k = 0; k < per; ++k) {
    const int g = g0 + k;
    if (g >= n_gal) break;
    const int64_t nb = gal[g].nb, begin = gal[g].spaxel_begin;
    const int64_t end = g + 1 < n_gal ? int64_t(gal[g + 1].spaxel_begin) : int64_t(n_rows);
    if (nb < 1 || begin + nb * nb != end || (g == 0 && begin != 0)) bad = 1;
    sum += nb > 0 ? int(nb) : 0;
  }
  part[tid] = sum;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {  // inclusive scan of the 256 partial sums
    const int v = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  int run = part[tid] - sum;
  for (int k = 0; k < per; ++k) {
    const int g = g0 + k;
    if (g >= n_gal) break;
    lines[g] = run;
    run += gal[g].nb > 0 ? gal[g].nb : 0;
  }
  if (tid == 255) lines[n_gal] = part[255];
  const bool packed = __syncthreads_or(bad) == 0;
  return packed;
}

// Galaxy g of line L of a packed table and the line's first element / stride.
struct BatchLine {
  int nb;
  int64_t base, stride;
};

__device__ inline BatchLine batch_line(const rbx_galaxy* __restrict__ gal, const int* lines,
                                       int n_gal, int nt, int axis, int L) {
  int lo = 0, hi = n_gal;  // last galaxy with lines[g] <= L
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (lines[mid] <= L) lo = mid; else hi = mid;
  }
  const int j = L - lines[lo];
  BatchLine b;
  b.nb = gal[lo].nb;
  const int64_t begin = gal[lo].spaxel_begin;
  if (axis == 1) {  // along x: line y = j
    b.base = (begin + int64_t(j) * b.nb) * nt;
    b.stride = nt;
  } else {          // along y: line x = j
    b.base = (begin + j) * int64_t(nt);
    b.stride = int64_t(b.nb) * nt;
  }
  return b;
}

// A line that is the same for the whole wavefront, in scalar registers.
__device__ inline BatchLine uniform_line(const BatchLine& b) {
  auto scalar = [](int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(uint64_t(v) >> 32));
    return int64_t(uint64_t(hi) << 32 | lo);
  };
  BatchLine u;
  u.nb = __builtin_amdgcn_readfirstlane(b.nb);
  u.base = scalar(b.base);
  u.stride = scalar(b.stride);
  return u;
}

// conv_batch_kernel's row item (row p, lambda chunk c) for tables that are
// not packed.
__device__ inline void batch_row_item(const float* __restrict__ in, float* __restrict__ out,
                                      const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows,
                                      int nt, int axis, const float* __restrict__ taps,
                                      int n_taps, int start, int n_chunks, int64_t item) {
  const int p = int(item / n_chunks);
  const int l0 = int(item - int64_t(p) * n_chunks) * kLineChunk;
  const int l1 = l0 + kLineChunk < nt ? l0 + kLineChunk : nt;
  const BatchPos b = batch_pos(gal, n_gal, n_rows, nt, axis, int64_t(p) * nt);
  for (int l = l0 + threadIdx.x; l < l1; l += blockDim.x) {
    float acc = 0.f;
    if (b.ok) {
      for (int t = 0; t < n_taps; ++t) {
        const int us = b.u + start - t;
        if (us >= 0 && us < b.nb) acc += taps[t] * in[b.base + l + us * b.stride];
      }
    }
    out[int64_t(p) * nt + l] = acc;
  }
}

// This thread's share of sum(a * conv(b)) over the row items of a table that is
// not packed (rows of no galaxy add nothing).
__device__ inline double batch_row_dots(const float* __restrict__ a, const float* __restrict__ bsrc,
                                        const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows,
                                        int nt, int axis, const double* __restrict__ taps,
                                        int n_taps, int start) {
  double acc = 0.0;
  const int n_chunks = (nt + kLineChunk - 1) / kLineChunk;
  const int64_t n_items = int64_t(n_rows) * n_chunks;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int p = int(item / n_chunks);
    const int l0 = int(item - int64_t(p) * n_chunks) * kLineChunk;
    const int l1 = l0 + kLineChunk < nt ? l0 + kLineChunk : nt;
    const BatchPos b = batch_pos(gal, n_gal, n_rows, nt, axis, int64_t(p) * nt);
    if (!b.ok) continue;
    for (int l = l0 + threadIdx.x; l < l1; l += blockDim.x) {
      double c = 0.0;
      for (int t = 0; t < n_taps; ++t) {
        const int us = b.u + start - t;
        if (us >= 0 && us < b.nb) c += taps[t] * double(bsrc[b.base + l + us * b.stride]);
      }
      acc += double(a[int64_t(p) * nt + l]) * c;
    }
  }
  return acc;
}

__global__ void __launch_bounds__(256) conv_batch_tile_kernel(
    const float* __restrict__ in, float* __restrict__ out, const rbx_galaxy* __restrict__ gal,
    int n_gal, int n_rows, int nt, int axis, const float* __restrict__ taps, int n_taps,
    int start) {
  extern __shared__ float tile[];
  __shared__ int lines[kBatchGalMax + 1];
  __shared__ int part[256];
  const bool packed = batch_line_prefix(gal, n_gal, n_rows, lines, part);
  if (!packed) {
    const int n_chunks = (nt + kLineChunk - 1) / kLineChunk;
    const int64_t n_items = int64_t(n_rows) * n_chunks;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x)
      batch_row_item(in, out, gal, n_gal, n_rows, nt, axis, taps, n_taps, start, n_chunks, item);
    return;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n_lblk = (nt + 63) / 64;
  const int64_t n_items = int64_t(lines[n_gal]) * n_lblk;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int L = int(item / n_lblk);
    const int l = int(item - int64_t(L) * n_lblk) * 64 + lane;
    const bool lok = l < nt;
    const BatchLine b = batch_line(gal, lines, n_gal, nt, axis, L);
    const int nb = b.nb;
    const int64_t e0 = b.base + (lok ? l : 0);
    if (nb <= kBatchTileAxis) {
      __syncthreads();  // the previous line's reads are done
      for (int u = w; u < nb; u += 4) tile[u * 64 + lane] = lok ? in[e0 + u * b.stride] : 0.f;
      __syncthreads();
      if (lok) {
        for (int u0 = w; u0 < nb; u0 += 16) {
          float acc[4];
          tile_conv4<float>(tile, lane, nb, taps, n_taps, start, u0, acc);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int u = u0 + 4 * r;
            if (u < nb) out[e0 + u * b.stride] = acc[r];
          }
        }
      }
    } else if (lok) {
      for (int u = w; u < nb; u += 4) {
        float acc = 0.f;
        for (int t = 0; t < n_taps; ++t) {
          const int us = u + start - t;
          if (us >= 0 && us < nb) acc += taps[t] * in[e0 + us * b.stride];
        }
        out[e0 + u * b.stride] = acc;
      }
    }
  }
}

// conv_batch_tile_kernel for the instantiated tap counts: a wavefront walks
// (line L, block of 64 lambda) as conv_cols_kernel does, lines of any length.
template <int M>
__global__ void __launch_bounds__(256) conv_batch_cols_kernel(
    const float* __restrict__ in, float* __restrict__ out, const rbx_galaxy* __restrict__ gal,
    int n_gal, int n_rows, int nt, int axis, const float* __restrict__ taps, int start) {
  __shared__ int lines[kBatchGalMax + 1];
  __shared__ int part[256];
  const bool packed = batch_line_prefix(gal, n_gal, n_rows, lines, part);
  if (!packed) {
    const int n_chunks = (nt + kLineChunk - 1) / kLineChunk;
    const int64_t n_items = int64_t(n_rows) * n_chunks;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x)
      batch_row_item(in, out, gal, n_gal, n_rows, nt, axis, taps, M, start, n_chunks, item);
    return;
  }
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_lblk = (nt + 63) / 64;
  const int64_t n_items = int64_t(lines[n_gal]) * n_lblk;
  for (int64_t item = int64_t(blockIdx.x) * 4 + w; item < n_items; item += int64_t(gridDim.x) * 4) {
    const int L = int(item / n_lblk);
    const int l = int(item - int64_t(L) * n_lblk) * 64 + lane;
    const bool ok = l < nt;
    const BatchLine b = uniform_line(batch_line(gal, lines, n_gal, nt, axis, L));
    const int64_t e0 = b.base + (ok ? l : 0);
    column_walk<M, float>(in + e0, b.stride, b.nb, ok, 0, b.nb, start, taps,
                          [&](int u, float v) {
                            if (ok) out[e0 + u * b.stride] = v;
                          });
  }
}

// sum(a * conv(b)) per block over conv_batch_cols_kernel's items (packed
// tables; the row items of conv_batch_dot_partial_kernel otherwise).
template <int M>
__global__ void __launch_bounds__(kDotThreads) conv_batch_dot_cols_kernel(
    const float* __restrict__ a, const float* __restrict__ bsrc,
    const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows, int nt, int axis,
    const double* __restrict__ taps, int start, double* __restrict__ partial) {
  __shared__ int lines[kBatchGalMax + 1];
  __shared__ int part[256];
  __shared__ double sm[kDotThreads];
  const bool packed = batch_line_prefix(gal, n_gal, n_rows, lines, part);
  double acc = 0.0;
  if (!packed) {
    acc = batch_row_dots(a, bsrc, gal, n_gal, n_rows, nt, axis, taps, M, start);
  } else {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_lblk = (nt + 63) / 64;
    const int64_t n_items = int64_t(lines[n_gal]) * n_lblk;
    for (int64_t item = int64_t(blockIdx.x) * 4 + w; item < n_items; item += int64_t(gridDim.x) * 4) {
      const int L = int(item / n_lblk);
      const int l = int(item - int64_t(L) * n_lblk) * 64 + lane;
      const bool ok = l < nt;
      const BatchLine b = uniform_line(batch_line(gal, lines, n_gal, nt, axis, L));
      const int64_t e0 = b.base + (ok ? l : 0);
      column_walk<M, double>(bsrc + e0, b.stride, b.nb, ok, 0, b.nb, start, taps,
                             [&](int u, double v) {
                               if (ok) acc += double(a[e0 + u * b.stride]) * v;
                             });
    }
  }
  block_partial(acc, sm, partial);
}

// conv_batch_cols_kernel and conv_batch_dot_cols_kernel of the adjoint in one
// pass over a and b.
template <int M>
__global__ void __launch_bounds__(kDotThreads) conv_batch_bwd_cols_kernel(
    const float* __restrict__ a, const float* __restrict__ bsrc, float* __restrict__ out,
    const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows, int nt, int axis,
    const float* __restrict__ rev, const double* __restrict__ dtaps, double* __restrict__ partial) {
  __shared__ int lines[kBatchGalMax + 1];
  __shared__ int part[256];
  __shared__ double sm[kDotThreads];
  const bool packed = batch_line_prefix(gal, n_gal, n_rows, lines, part);
  double acc = 0.0;
  constexpr int start = (M - 1) / 2;
  if (!packed) {
    const int n_chunks = (nt + kLineChunk - 1) / kLineChunk;
    const int64_t n_items = int64_t(n_rows) * n_chunks;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x)
      batch_row_item(a, out, gal, n_gal, n_rows, nt, axis, rev, M, start, n_chunks, item);
    acc = batch_row_dots(a, bsrc, gal, n_gal, n_rows, nt, axis, dtaps, M, start);
  } else {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_lblk = (nt + 63) / 64;
    const int64_t n_items = int64_t(lines[n_gal]) * n_lblk;
    for (int64_t item = int64_t(blockIdx.x) * 4 + w; item < n_items; item += int64_t(gridDim.x) * 4) {
      const int L = int(item / n_lblk);
      const int l = int(item - int64_t(L) * n_lblk) * 64 + lane;
      const bool ok = l < nt;
      const BatchLine b = uniform_line(batch_line(gal, lines, n_gal, nt, axis, L));
      const int64_t e0 = b.base + (ok ? l : 0);
      acc += column_walk_bwd<M>(a + e0, bsrc + e0, b.stride, b.nb, ok, 0, b.nb, rev, dtaps,
                                [&](int u, float v) {
                                  if (ok) out[e0 + u * b.stride] = v;
                                });
    }
  }
  block_partial(acc, sm, partial);
}

// sum(a * conv(b)) per block: line items of a packed table as
// conv_batch_tile_kernel, else the row items of conv_batch_dot_partial_kernel.
__global__ void __launch_bounds__(kDotThreads) conv_batch_dot_tile_kernel(
    const float* __restrict__ a, const float* __restrict__ bsrc,
    const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows, int nt, int axis,
    const double* __restrict__ taps, int n_taps, int start, double* __restrict__ partial) {
  extern __shared__ float tile[];
  __shared__ int lines[kBatchGalMax + 1];
  __shared__ int part[256];
  __shared__ double sm[kDotThreads];
  const bool packed = batch_line_prefix(gal, n_gal, n_rows, lines, part);
  double acc = 0.0;
  if (!packed) {
    acc = batch_row_dots(a, bsrc, gal, n_gal, n_rows, nt, axis, taps, n_taps, start);
  } else {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int n_lblk = (nt + 63) / 64;
    const int64_t n_items = int64_t(lines[n_gal]) * n_lblk;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
      const int L = int(item / n_lblk);
      const int l = int(item - int64_t(L) * n_lblk) * 64 + lane;
      const bool lok = l < nt;
      const BatchLine b = batch_line(gal, lines, n_gal, nt, axis, L);
      const int nb = b.nb;
      const int64_t e0 = b.base + (lok ? l : 0);
      if (nb <= kBatchTileAxis) {
        __syncthreads();
        for (int u = w; u < nb; u += 4) tile[u * 64 + lane] = lok ? bsrc[e0 + u * b.stride] : 0.f;
        __syncthreads();
        if (lok) {
          for (int u0 = w; u0 < nb; u0 += 16) {
            double c[4];
            tile_conv4<double>(tile, lane, nb, taps, n_taps, start, u0, c);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int u = u0 + 4 * r;
              if (u < nb) acc += double(a[e0 + u * b.stride]) * c[r];
            }
          }
        }
      } else if (lok) {
        for (int u = w; u < nb; u += 4) {
          double c = 0.0;
          for (int t = 0; t < n_taps; ++t) {
            const int us = u + start - t;
            if (us >= 0 && us < nb) c += taps[t] * double(bsrc[e0 + us * b.stride]);
          }
          acc += double(a[e0 + u * b.stride]) * c;
        }
      }
    }
  }
  block_partial(acc, sm, partial);
}

__global__ void __launch_bounds__(kDotThreads) conv_batch_dot_partial_kernel(
    const float* __restrict__ a, const float* __restrict__ bsrc,
    const rbx_galaxy* __restrict__ gal, int n_gal, int n_rows, int nt, int axis,
    const double* __restrict__ taps, int n_taps, int start, int n_chunks, int64_t n_items,
    double* __restrict__ partial) {
  __shared__ double sm[kDotThreads];
  double acc = 0.0;
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int p = int(item / n_chunks);
    const int l0 = int(item - int64_t(p) * n_chunks) * kLineChunk;
    const int l1 = l0 + kLineChunk < nt ? l0 + kLineChunk : nt;
    const BatchPos b = batch_pos(gal, n_gal, n_rows, nt, axis, int64_t(p) * nt);
    if (!b.ok) continue;
    for (int l = l0 + threadIdx.x; l < l1; l += blockDim.x) {
      double c = 0.0;
      for (int t = 0; t < n_taps; ++t) {
        const int us = b.u + start - t;
        if (us >= 0 && us < b.nb) c += taps[t] * double(bsrc[b.base + l + us * b.stride]);
      }
      acc += double(a[int64_t(p) * nt + l]) * c;
    }
  }
  block_partial(acc, sm, partial);
}

static int grid_for(int64_t n, int threads, int64_t cap) {
  int64_t g = (n + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return int(g);
}

static int dot_blocks(int64_t total) { return grid_for(total, kDotThreads * 8, kDotBlocksMax); }

static int64_t item_blocks(int64_t items, int64_t cap) { return items < cap ? (items > 0 ? items : 1) : cap; }

// Calls f with the tap count as a constant where conv_cols_kernel has it: the
// odd sizes of a PSF kernel up to 25 pixels (M^2 multiply-adds of code and
// about 3 M registers each).
template <class F>
static bool with_taps(int m, F&& f) {
  switch (m) {
    case 3: f(std::integral_constant<int, 3>{}); return true;
    case 5: f(std::integral_constant<int, 5>{}); return true;
    case 7: f(std::integral_constant<int, 7>{}); return true;
    case 9: f(std::integral_constant<int, 9>{}); return true;
    case 11: f(std::integral_constant<int, 11>{}); return true;
    case 13: f(std::integral_constant<int, 13>{}); return true;
    case 15: f(std::integral_constant<int, 15>{}); return true;
    case 17: f(std::integral_constant<int, 17>{}); return true;
    case 21: f(std::integral_constant<int, 21>{}); return true;
    case 25: f(std::integral_constant<int, 25>{}); return true;
    default: return false;
  }
}

// conv_cols_kernel's items: segments of the axis so that about 16 000
// wavefronts are there (two for each that fits the chip), but none shorter
// than 16 outputs (its M - 1 halo inputs are read again, from cache).
struct ColItems {
  int64_t n_blocks, n_items;
  int n_segs, seg;
};

static ColItems col_items(int64_t n_outer, int n_axis, int64_t n_inner) {
  ColItems c;
  c.n_blocks = (n_inner + 63) / 64;
  const int64_t cols = n_outer * c.n_blocks;
  int64_t want = cols > 0 ? (16384 + cols - 1) / cols : 1;
  const int64_t most = (n_axis + 15) / 16;
  if (want > most) want = most;
  c.seg = int((n_axis + want - 1) / want);
  c.n_segs = (n_axis + c.seg - 1) / c.seg;
  c.n_items = cols * c.n_segs;
  return c;
}

// Outputs per row segment: the fewest segments of at most kSeg, of equal length.
static int row_seg(int n_axis) {
  const int n = (n_axis + kSeg - 1) / kSeg;
  return ((n_axis + n - 1) / n + 3) / 4 * 4;
}

int conv_axis(const float* in, float* out, int64_t n_outer, int n_axis, int64_t n_inner,
              const float* taps, int n_taps, int start, hipStream_t s) {
  const int64_t total = n_outer * n_axis * n_inner;
  if (total == 0) return RBX_OK;
  if (n_inner == 1 && n_taps - 1 <= kHalo) {
    const int seg = row_seg(n_axis);
    const int64_t n_seg = (n_axis + seg - 1) / seg;
    const int64_t items = n_outer * n_seg;
    hipLaunchKernelGGL(conv_rows_kernel, dim3(item_blocks(items, 1 << 20)), dim3(256), 0, s, in,
                       out, n_axis, taps, n_taps, start, n_seg, seg, items);
  } else if (n_inner > 1 && with_taps(n_taps, [&](auto m) {
               const ColItems c = col_items(n_outer, n_axis, n_inner);
               hipLaunchKernelGGL(conv_cols_kernel<decltype(m)::value>,
                                  dim3(item_blocks((c.n_items + 3) / 4, 1 << 20)), dim3(256), 0, s,
                                  in, out, n_axis, n_inner, taps, start, c.n_blocks, c.n_segs,
                                  c.seg, c.n_items);
             })) {
  } else if (n_inner > 1 && n_axis <= kTileAxis) {
    const int64_t n_blocks = (n_inner + 63) / 64;
    const int64_t items = n_outer * n_blocks;
    hipLaunchKernelGGL(conv_tile_kernel, dim3(item_blocks(items, 1 << 20)), dim3(256),
                       size_t(n_axis) * 64 * sizeof(float), s, in, out, n_axis, n_inner, taps,
                       n_taps, start, n_blocks, items);
  } else if (n_inner > 1) {
    const int64_t n_chunks = (n_inner + kLineChunk - 1) / kLineChunk;
    const int64_t items = n_outer * n_axis * n_chunks;
    hipLaunchKernelGGL(conv_lines_kernel, dim3(item_blocks(items, 1 << 20)), dim3(256), 0, s, in,
                       out, n_outer, n_axis, n_inner, taps, n_taps, start, n_chunks, items);
  } else {
    hipLaunchKernelGGL(conv_axis_kernel, dim3(grid_for(total, 256, 1 << 20)), dim3(256), 0, s, in,
                       out, n_outer, n_axis, n_inner, taps, n_taps, start);
  }
  return check_launch("rbx_conv_axis");
}

// dot = sum(a * conv_axis(b)) into result, the block partials in `partial`
// (nblk doubles, every one written by its block before the final sum).
static int conv_axis_dot(const float* a, const float* b, int64_t n_outer, int n_axis,
                         int64_t n_inner, const double* taps, int n_taps, int start,
                         double* partial, int nblk, double* result, hipStream_t s,
                         const char* who, const double* add = nullptr,
                         float* result32 = nullptr) {
  if (n_inner == 1 && n_taps - 1 <= kHalo) {
    const int seg = row_seg(n_axis);
    const int64_t n_seg = (n_axis + seg - 1) / seg;
    hipLaunchKernelGGL(conv_dot_rows_kernel, dim3(nblk), dim3(kDotThreads), 0, s, a, b, n_axis,
                       taps, n_taps, start, n_seg, seg, n_outer * n_seg, partial);
  } else if (n_inner > 1 && with_taps(n_taps, [&](auto m) {
               const ColItems c = col_items(n_outer, n_axis, n_inner);
               hipLaunchKernelGGL(conv_dot_cols_kernel<decltype(m)::value>, dim3(nblk),
                                  dim3(kDotThreads), 0, s, a, b, n_axis, n_inner, taps, start,
                                  c.n_blocks, c.n_segs, c.seg, c.n_items, partial);
             })) {
  } else if (n_inner > 1 && n_axis <= kTileAxis) {
    const int64_t n_blocks = (n_inner + 63) / 64;
    hipLaunchKernelGGL(conv_dot_tile_kernel, dim3(nblk), dim3(kDotThreads),
                       size_t(n_axis) * 64 * sizeof(float), s, a, b, n_axis, n_inner, taps, n_taps,
                       start, n_blocks, n_outer * n_blocks, partial);
  } else if (n_inner > 1) {
    const int64_t n_chunks = (n_inner + kLineChunk - 1) / kLineChunk;
    hipLaunchKernelGGL(conv_dot_lines_kernel, dim3(nblk), dim3(kDotThreads), 0, s, a, b, n_outer,
                       n_axis, n_inner, taps, n_taps, start, n_chunks, n_outer * n_axis * n_chunks,
                       partial);
  } else {
    hipLaunchKernelGGL(conv_dot_partial_kernel, dim3(nblk), dim3(kDotThreads), 0, s, a, b, n_outer,
                       n_axis, n_inner, taps, n_taps, start, partial);
  }
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kDotThreads), 0, s, partial, nblk, add, result,
                     result32);
  return check_launch(who);
}

// Adjoint of conv_axis (taps whose reversal is `rev`, from `start`) and its
// sigma dot: out = conv(a, rev) from m - 1 - start, result = add + sum(a *
// conv(b, dtaps)).  One pass over a and b for the LSF and for centred kernels
// of the instantiated sizes, else the two passes.
static int conv_axis_bwd(const float* a, const float* b, float* out, int64_t n_outer, int n_axis,
                         int64_t n_inner, const float* rev, const double* dtaps, int m, int start,
                         double* partial, int nblk, const double* add, double* result,
                         float* result32, hipStream_t s, const char* who) {
  if (n_inner == 1 && m - 1 <= kHalo && start >= 0 && start < m) {
    const int seg = row_seg(n_axis);
    const int64_t n_seg = (n_axis + seg - 1) / seg;
    hipLaunchKernelGGL(conv_bwd_rows_kernel, dim3(nblk), dim3(kDotThreads), 0, s, a, b, out, n_axis,
                       rev, dtaps, m, start, n_seg, seg, n_outer * n_seg, partial);
  } else if (n_inner > 1 && 2 * start == m - 1 && m <= 15 && with_taps(m, [&](auto mc) {
               constexpr int M = decltype(mc)::value;
               if constexpr (M <= 15) {
                 const ColItems c = col_items(n_outer, n_axis, n_inner);
                 hipLaunchKernelGGL(conv_bwd_cols_kernel<M>, dim3(nblk), dim3(kDotThreads), 0, s, a,
                                    b, out, n_axis, n_inner, rev, dtaps, c.n_blocks, c.n_segs, c.seg,
                                    c.n_items, partial);
               }
             })) {
  } else {
    int rc = conv_axis(a, out, n_outer, n_axis, n_inner, rev, m, m - 1 - start, s);
    if (!rc) rc = conv_axis_dot(a, b, n_outer, n_axis, n_inner, dtaps, m, start, partial, nblk, result,
                                s, who, add, result32);
    return rc;
  }
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kDotThreads), 0, s, partial, nblk, add, result,
                     result32);
  return check_launch(who);
}

// Block partials of rbx_conv_axis_dot_noalloc: a file-scope device array
// instead of a caller's workspace, kDotBlocksMax doubles (32 KiB), which
// every device the library runs on holds until the process ends.  Host code
// uses its per-device address (scratch_ptr), never the array's name.
static __device__ __align__(256) double scratch[kDotBlocksMax];

// Device address of `scratch` on the current device, looked up with
// hipGetSymbolAddress on the device's first call and kept per device.
static int scratch_ptr(double** out, const char* who) {
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return failf(RBX_EHIP, "%s: no current device", who);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return failf(RBX_EHIP, "%s: hipGetSymbolAddress(scratch) failed: %s", who,
                   hipGetErrorString(e));
    ptrs[dev] = p;
  }
  *out = static_cast<double*>(ptrs[dev]);
  return RBX_OK;
}

// Block partials of sum(a * conv_batch(b)).
static int batch_dot_partials(const float* a, const float* b, const rbx_galaxy* galaxies, int32_t n_gal,
                              int32_t n_rows, int32_t n_target, int32_t axis, const double* taps,
                              int32_t n_taps, int32_t start, double* partial, int nblk,
                              hipStream_t s) {
  if (n_gal <= kBatchGalMax && with_taps(n_taps, [&](auto m) {
        hipLaunchKernelGGL(conv_batch_dot_cols_kernel<decltype(m)::value>, dim3(nblk),
                           dim3(kDotThreads), 0, s, a, b, galaxies, n_gal, n_rows, n_target, axis,
                           taps, start, partial);
      })) {
  } else if (n_gal <= kBatchGalMax) {
    hipLaunchKernelGGL(conv_batch_dot_tile_kernel, dim3(nblk), dim3(kDotThreads),
                       size_t(kBatchTileAxis) * 64 * sizeof(float), s, a, b, galaxies, n_gal,
                       n_rows, n_target, axis, taps, n_taps, start, partial);
  } else {
    const int n_chunks = (n_target + kLineChunk - 1) / kLineChunk;
    hipLaunchKernelGGL(conv_batch_dot_partial_kernel, dim3(nblk), dim3(kDotThreads), 0, s, a, b,
                       galaxies, n_gal, n_rows, n_target, axis, taps, n_taps, start, n_chunks,
                       int64_t(n_rows) * n_chunks, partial);
  }
  return check_launch("rbx_conv_batch_dot");
}

}  // namespace rbx

extern "C" {

int rbx_gauss_taps(const double* x, int32_t n, const void* sigma, int32_t sigma_f64, float* taps,
                   float* reversed, double* dtaps, void* stream) {
  using namespace rbx;
  if (!x || !sigma || !taps || !reversed || !dtaps || n < 1)
    return fail(RBX_EINVAL, "rbx_gauss_taps: bad arguments");
  hipStream_t s = as_stream(stream);
  if (sigma_f64)
    hipLaunchKernelGGL(gauss_taps_kernel<double>, dim3(1), dim3(kDotThreads), 0, s, x, n,
                       static_cast<const double*>(sigma), taps, reversed, dtaps);
  else
    hipLaunchKernelGGL(gauss_taps_kernel<float>, dim3(1), dim3(kDotThreads), 0, s, x, n,
                       static_cast<const float*>(sigma), taps, reversed, dtaps);
  return check_launch("rbx_gauss_taps");
}

int rbx_conv_axis(const float* in, float* out, int64_t n_outer, int32_t n_axis, int64_t n_inner,
                  const float* taps, int32_t n_taps, int32_t start, void* stream) {
  using namespace rbx;
  if (!in || !out || !taps || n_outer < 0 || n_axis < 1 || n_inner < 1 || n_taps < 1)
    return fail(RBX_EINVAL, "rbx_conv_axis: bad arguments");
  if (in == out) return fail(RBX_EINVAL, "rbx_conv_axis: in-place convolution not supported");
  return conv_axis(in, out, n_outer, n_axis, n_inner, taps, n_taps, start, as_stream(stream));
}

int rbx_psf_sep(const float* in, float* out, float* tmp, int32_t ny, int32_t nx, int32_t nl,
                const float* gy, int32_t my, int32_t start_y, const float* gx, int32_t mx,
                int32_t start_x, void* stream) {
  using namespace rbx;
  if (!in || !out || !tmp || !gy || !gx || ny < 1 || nx < 1 || nl < 1 || my < 1 || mx < 1)
    return fail(RBX_EINVAL, "rbx_psf_sep: bad arguments");
  if (in == out || in == tmp || out == tmp)
    return fail(RBX_EINVAL, "rbx_psf_sep: in, out and tmp must be distinct");
  hipStream_t s = as_stream(stream);
  int rc = conv_axis(in, tmp, ny, nx, nl, gx, mx, start_x, s);
  if (rc) return rc;
  return conv_axis(tmp, out, 1, ny, int64_t(nx) * nl, gy, my, start_y, s);
}

int rbx_conv2d_planes(const float* in, float* out, int32_t ny, int32_t nx, int32_t nl,
                      const float* kernel, int32_t ky, int32_t kx, int32_t sy, int32_t sx,
                      void* stream) {
  using namespace rbx;
  if (!in || !out || !kernel || ny < 1 || nx < 1 || nl < 1 || ky < 1 || kx < 1 || in == out)
    return fail(RBX_EINVAL, "rbx_conv2d_planes: bad arguments");
  const int64_t total = int64_t(ny) * nx * nl;
  hipLaunchKernelGGL(conv2d_planes_kernel, dim3(grid_for(total, 256, 1 << 20)), dim3(256), 0,
                     as_stream(stream), in, out, ny, nx, nl, kernel, ky, kx, sy, sx);
  return check_launch("rbx_conv2d_planes");
}

size_t rbx_dot_workspace_size(int64_t total) {
  if (total < 0) return 0;
  return size_t(rbx::dot_blocks(total)) * sizeof(double);
}

int rbx_conv_axis_dot(const float* a, const float* b, int64_t n_outer, int32_t n_axis,
                      int64_t n_inner, const double* taps, int32_t n_taps, int32_t start,
                      double* result, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace rbx;
  if (!a || !b || !taps || !result || n_outer < 0 || n_axis < 1 || n_inner < 1 || n_taps < 1)
    return fail(RBX_EINVAL, "rbx_conv_axis_dot: bad arguments");
  const int64_t total = n_outer * n_axis * n_inner;
  const int nblk = dot_blocks(total);
  if (!workspace || workspace_bytes < size_t(nblk) * sizeof(double))
    return fail(RBX_EWORKSPACE, "rbx_conv_axis_dot: workspace too small");
  return conv_axis_dot(a, b, n_outer, n_axis, n_inner, taps, n_taps, start,
                       static_cast<double*>(workspace), nblk, result, as_stream(stream),
                       "rbx_conv_axis_dot");
}

int rbx_conv_axis_dot_noalloc(const float* a, const float* b, int64_t n_outer, int32_t n_axis,
                              int64_t n_inner, const double* taps, int32_t n_taps,
                              int32_t start, double* result, void* stream) {
  using namespace rbx;
  const char* who = "rbx_conv_axis_dot_noalloc";
  if (!a || !b || !taps || !result || n_outer < 0 || n_axis < 1 || n_inner < 1 || n_taps < 1)
    return failf(RBX_EINVAL, "%s: bad arguments", who);
  const int64_t total = n_outer * n_axis * n_inner;
  const int nblk = dot_blocks(total);
  if (nblk > kDotBlocksMax)
    return failf(RBX_EINVAL, "%s: %d block partials exceed the %d-double scratch", who, nblk,
                 kDotBlocksMax);
  double* partial = nullptr;
  const int rc = scratch_ptr(&partial, who);
  if (rc) return rc;
  return conv_axis_dot(a, b, n_outer, n_axis, n_inner, taps, n_taps, start, partial, nblk, result,
                       as_stream(stream), who);
}

int rbx_conv_axis_bwd(const float* dout, const float* in, float* din, int64_t n_outer,
                      int32_t n_axis, int64_t n_inner, const float* reversed, const double* dtaps,
                      int32_t n_taps, int32_t start, const double* add, double* result,
                      float* result32, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace rbx;
  if (!dout || !in || !din || !reversed || !dtaps || !result || n_outer < 0 || n_axis < 1 ||
      n_inner < 1 || n_taps < 1)
    return fail(RBX_EINVAL, "rbx_conv_axis_bwd: bad arguments");
  if (din == dout || din == in)
    return fail(RBX_EINVAL, "rbx_conv_axis_bwd: in-place convolution not supported");
  const int nblk = dot_blocks(n_outer * n_axis * n_inner);
  if (!workspace || workspace_bytes < size_t(nblk) * sizeof(double))
    return fail(RBX_EWORKSPACE, "rbx_conv_axis_bwd: workspace too small");
  return conv_axis_bwd(dout, in, din, n_outer, n_axis, n_inner, reversed, dtaps, n_taps, start,
                       static_cast<double*>(workspace), nblk, add, result, result32,
                       as_stream(stream), "rbx_conv_axis_bwd");
}

int rbx_conv_batch(const float* in, float* out, const rbx_galaxy* galaxies, int32_t n_gal,
                   int32_t n_rows, int32_t n_target, int32_t axis, const float* taps,
                   int32_t n_taps, int32_t start, void* stream) {
  using namespace rbx;
  if (!in || !out || !galaxies || !taps || n_gal < 1 || n_rows < 0 || n_target < 1 ||
      n_taps < 1 || (axis != 0 && axis != 1))
    return fail(RBX_EINVAL, "rbx_conv_batch: bad arguments");
  if (in == out) return fail(RBX_EINVAL, "rbx_conv_batch: in-place convolution not supported");
  const int64_t total = int64_t(n_rows) * n_target;
  if (total == 0) return RBX_OK;
  if (n_gal <= kBatchGalMax) {
    // persistent grid: every workgroup builds the table's line prefix once
    if (with_taps(n_taps, [&](auto m) {
          hipLaunchKernelGGL(conv_batch_cols_kernel<decltype(m)::value>, dim3(2048), dim3(256), 0,
                             as_stream(stream), in, out, galaxies, n_gal, n_rows, n_target, axis,
                             taps, start);
        }))
      return check_launch("rbx_conv_batch");
    hipLaunchKernelGGL(conv_batch_tile_kernel, dim3(2048), dim3(256),
                       size_t(kBatchTileAxis) * 64 * sizeof(float), as_stream(stream), in, out,
                       galaxies, n_gal, n_rows, n_target, axis, taps, n_taps, start);
    return check_launch("rbx_conv_batch");
  }
  const int n_chunks = (n_target + kLineChunk - 1) / kLineChunk;
  const int64_t items = int64_t(n_rows) * n_chunks;
  hipLaunchKernelGGL(conv_batch_kernel, dim3(item_blocks(items, 1 << 20)), dim3(256), 0,
                     as_stream(stream), in, out, galaxies, n_gal, n_rows, n_target, axis, taps,
                     n_taps, start, n_chunks, items);
  return check_launch("rbx_conv_batch");
}

int rbx_conv_batch_dot(const float* a, const float* b, const rbx_galaxy* galaxies, int32_t n_gal,
                       int32_t n_rows, int32_t n_target, int32_t axis, const double* taps,
                       int32_t n_taps, int32_t start, double* out, void* workspace,
                       size_t workspace_bytes, void* stream) {
  using namespace rbx;
  if (!a || !b || !galaxies || !taps || !out || n_gal < 1 || n_rows < 0 || n_target < 1 ||
      n_taps < 1 || (axis != 0 && axis != 1))
    return fail(RBX_EINVAL, "rbx_conv_batch_dot: bad arguments");
  const int64_t total = int64_t(n_rows) * n_target;
  const int nblk = dot_blocks(total);
  if (!workspace || workspace_bytes < size_t(nblk) * sizeof(double))
    return fail(RBX_EWORKSPACE, "rbx_conv_batch_dot: workspace too small");
  hipStream_t s = as_stream(stream);
  double* partial = static_cast<double*>(workspace);
  if (int rc = batch_dot_partials(a, b, galaxies, n_gal, n_rows, n_target, axis, taps, n_taps, start,
                                  partial, nblk, s))
    return rc;
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kDotThreads), 0, s, partial, nblk,
                     nullptr, out, nullptr);
  return check_launch("rbx_conv_batch_dot");
}

int rbx_conv_batch_bwd(const float* dout, const float* in, float* din, const rbx_galaxy* galaxies,
                       int32_t n_gal, int32_t n_rows, int32_t n_target, int32_t axis,
                       const float* reversed, const double* dtaps, int32_t n_taps, int32_t start,
                       const double* add, double* result, float* result32, void* workspace,
                       size_t workspace_bytes, void* stream) {
  using namespace rbx;
  if (!dout || !in || !din || !galaxies || !reversed || !dtaps || !result || n_gal < 1 ||
      n_rows < 0 || n_target < 1 || n_taps < 1 || (axis != 0 && axis != 1))
    return fail(RBX_EINVAL, "rbx_conv_batch_bwd: bad arguments");
  if (din == dout || din == in)
    return fail(RBX_EINVAL, "rbx_conv_batch_bwd: in-place convolution not supported");
  const int nblk = dot_blocks(int64_t(n_rows) * n_target);
  if (!workspace || workspace_bytes < size_t(nblk) * sizeof(double))
    return fail(RBX_EWORKSPACE, "rbx_conv_batch_bwd: workspace too small");
  hipStream_t s = as_stream(stream);
  double* partial = static_cast<double*>(workspace);
  const bool one_pass =
      n_gal <= kBatchGalMax && 2 * start == n_taps - 1 && n_taps <= 15 && with_taps(n_taps, [&](auto mc) {
        constexpr int M = decltype(mc)::value;
        if constexpr (M <= 15)
          hipLaunchKernelGGL(conv_batch_bwd_cols_kernel<M>, dim3(nblk), dim3(kDotThreads), 0, s, dout,
                             in, din, galaxies, n_gal, n_rows, n_target, axis, reversed, dtaps,
                             partial);
      });
  if (!one_pass) {
    int rc = rbx_conv_batch(dout, din, galaxies, n_gal, n_rows, n_target, axis, reversed, n_taps,
                            n_taps - 1 - start, stream);
    if (rc) return rc;
    rc = batch_dot_partials(dout, in, galaxies, n_gal, n_rows, n_target, axis, dtaps, n_taps, start,
                            partial, nblk, s);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kDotThreads), 0, s, partial, nblk, add, result,
                     result32);
  return check_launch("rbx_conv_batch_bwd");
}

}  // extern "C"
