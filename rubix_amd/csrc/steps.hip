// Plain per-step kernels: one kernel (and one hand-written adjoint) per
// rubix.core step, each writing the same RubixData field the reference step
// writes.  They materialise the per-star spectra exactly like the reference
// chain does, so they are HBM-bound by design; the fused path in cube.hip
// replaces calculate_spectra .. calculate_datacube for throughput.
//
//   calculate_spectra             rbx_ssp_lookup      (rubix/core/ifu.py:63-121)
//   scale_spectrum_by_mass        rbx_scale_rows      (rubix/core/ifu.py:149-157)
//   doppler_shift_and_resampling  rbx_resample        (rubix/core/ifu.py:269-293,
//                                                      rubix/spectra/ifu.py:190,223-266)
//   calculate_datacube            rbx_segment_cube    (rubix/spectra/ifu.py:269-288)
#include <float.h>

#include "rbx_common.h"
#include "ssp_device.h"

namespace rbx {

constexpr int kStepThreads = 256;
constexpr int kBins = 4;          // target bins a thread of resample_kernel has in flight
constexpr int kBwdBins = 2;       // and of resample_bwd_kernel, which then fits 80 VGPRs
constexpr int kBwdThreads = 512;  // most of resample_bwd: 3 workgroups a CU by LDS at 3721 bins, 24 wavefronts

// Fixed-order block reduction (deterministic); every thread gets the sum.
template <class T>
__device__ inline T block_sum(T v, T* sm) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) sm[w] = v;
  __syncthreads();
  T s = T(0);
  const int nw = blockDim.x >> 6;
  for (int k = 0; k < nw; ++k) s += sm[k];
  __syncthreads();
  return s;
}

// Elementwise work on rows of length n at any 4-byte alignment: f(k) on whole
// groups of four elements (one 16-byte access each), g(k) on the last few.
template <class F, class G>
__device__ inline void row_quads(int n, int first, int step, F&& f, G&& g) {
  for (int k = 4 * first; k + 4 <= n; k += 4 * step) f(k);
  const int tail = n & ~3;
  if (first < n - tail) g(tail + first);
}

__device__ inline void st_quad(float* base, uint32_t idx, const Quad& q) {
  *reinterpret_cast<Quad*>(reinterpret_cast<char*>(base) + idx * 4u) = q;
}

// ------------------------------------------------------------ lookup

// One workgroup per star.  Bound by the template rows' way through L2 (16
// bytes read per float written) and the writes; slabs of the wavelengths
// pinned to XCDs, so that each L2 holds its share of the templates, measured
// the same (1.8 ms at 200 k x 5000).
__global__ void __launch_bounds__(kStepThreads) lookup_kernel(SspView g, const float* __restrict__ met,
                                                             const float* __restrict__ age, int64_t n,
                                                             float* __restrict__ out) {
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const Cell c = make_cell(g, met[r], age[r]);
    const int nw = g.n_wave;
    const int row = __builtin_amdgcn_readfirstlane(c.row);
    const float* f[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) f[q] = g.flux + int64_t(corner_row(row, q, g.n_age)) * nw;
    float* o = out + r * nw;
    auto mix = [&](float f0, float f1, float f2, float f3) {
      return c.inside ? c.w[0] * f0 + c.w[1] * f1 + c.w[2] * f2 + c.w[3] * f3 : 0.f;
    };
    row_quads(
        nw, threadIdx.x, kStepThreads,
        [&](int k) {
          Quad v[4], res;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = ld_quad(f[q], uint32_t(k));
#pragma unroll
          for (int e = 0; e < 4; ++e) res.v[e] = mix(v[0].v[e], v[1].v[e], v[2].v[e], v[3].v[e]);
          st_quad(o, uint32_t(k), res);
        },
        [&](int k) { o[k] = mix(f[0][k], f[1][k], f[2][k], f[3][k]); });
  }
}

__global__ void __launch_bounds__(kStepThreads) lookup_bwd_kernel(
    SspView g, const float* __restrict__ met, const float* __restrict__ age, int64_t n,
    const float* __restrict__ dspec, float* __restrict__ dmet, float* __restrict__ dage) {
  __shared__ float sm[kStepThreads / 64];
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const float Z = met[r], t = age[r];
    const Cell c = make_cell(g, Z, t);
    if (!c.inside) {
      if (threadIdx.x == 0) {
        if (dmet) dmet[r] = 0.f;
        if (dage) dage[r] = 0.f;
      }
      continue;
    }
    const int nw = g.n_wave;
    const int row = __builtin_amdgcn_readfirstlane(c.row);
    const float* f[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) f[q] = g.flux + int64_t(corner_row(row, q, g.n_age)) * nw;
    const float* d = dspec + r * nw;
    float su = 0.f, ss = 0.f;
    auto add = [&](float dk, float v00, float v10, float v01, float v11) {
      su += dk * (c.gu[0] * v00 + c.gu[1] * v10 + c.gu[2] * v01 + c.gu[3] * v11);
      ss += dk * (c.gs[0] * v00 + c.gs[1] * v10 + c.gs[2] * v01 + c.gs[3] * v11);
    };
    row_quads(
        nw, threadIdx.x, kStepThreads,
        [&](int k) {
          const Quad dk = ld_quad(d, uint32_t(k));
          Quad v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = ld_quad(f[q], uint32_t(k));
#pragma unroll
          for (int e = 0; e < 4; ++e) add(dk.v[e], v[0].v[e], v[1].v[e], v[2].v[e], v[3].v[e]);
        },
        [&](int k) { add(d[k], f[0][k], f[1][k], f[2][k], f[3][k]); });
    su = block_sum(su, sm);
    ss = block_sum(ss, sm);
    if (threadIdx.x == 0) {
      if (dmet) dmet[r] = su * c.du_dZ;
      if (dage) dage[r] = ss * c.ds_dt;
    }
  }
}

// ------------------------------------------------------------ mass scaling

// One workgroup per row.  kDot: also dot[r] = sum_k in[r, k] other[r, k], so
// that the adjoint reads the incoming gradient once (200 k x 5000: 3.3 ms as
// two passes, 2.36 now, 5.1 TB/s).
template <bool kScale, bool kDot>
__global__ void __launch_bounds__(kStepThreads) scale_rows_kernel(
    const float* __restrict__ in, const float* __restrict__ scale, const float* __restrict__ other,
    int64_t n, int nw, float* __restrict__ out, float* __restrict__ dot) {
  __shared__ float sm[kStepThreads / 64];
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const float m = kScale ? scale[r] : 0.f;
    const float* x = in + r * nw;
    const float* y = kDot ? other + r * nw : nullptr;
    float* o = kScale ? out + r * nw : nullptr;
    float sum = 0.f;
    row_quads(
        nw, threadIdx.x, kStepThreads,
        [&](int k) {
          const Quad v = ld_quad(x, uint32_t(k));
          if (kDot) {
            const Quad w = ld_quad(y, uint32_t(k));
#pragma unroll
            for (int e = 0; e < 4; ++e) sum += v.v[e] * w.v[e];
          }
          if (kScale) {
            Quad res;
#pragma unroll
            for (int e = 0; e < 4; ++e) res.v[e] = v.v[e] * m;
            st_quad(o, uint32_t(k), res);
          }
        },
        [&](int k) {
          if (kDot) sum += x[k] * y[k];
          if (kScale) o[k] = x[k] * m;
        });
    if (kDot) {
      sum = block_sum(sum, sm);
      if (threadIdx.x == 0) dot[r] = sum;
    }
  }
}

// ------------------------------------------------------------ resampling

// Thread t's share of T = sum of S_k fl(w_k - w_{k-1}) over the in-range knots
// k >= 1, wmin <= w_k <= wmax.  The range of knots looked at comes from the
// locator guesses of its ends with their error bound (the whole grid on a
// coarse locator); the exact predicate decides each.
struct KnotRange {
  int lo, hi;
};

__device__ inline KnotRange mask_range(const SspView& g, const rbx_target& tg, const Shift& h) {
  const int n = g.n_wave;
  if (g.loc_multi) return {1, n - 1};
  auto guess = [&](float x) {
    const float fm = fminf(fmaxf(fmaf(x, h.c1, h.c0), 0.f), float(g.n_loc - 1));
    return ld_at(g.loc + 4 * int64_t(g.n_loc), uint32_t(fm));
  };
  const int a = guess(tg.wmin) - 3, b = guess(tg.wmax) + 5;
  return {a < 1 ? 1 : a, b > n - 1 ? n - 1 : b};
}

__device__ inline bool in_range(const rbx_target& tg, float w) { return w >= tg.wmin && w <= tg.wmax; }

__device__ inline float source_total(const SspView& g, const rbx_target& tg,
                                     const float* __restrict__ S, const KnotRange& kr, float a) {
  constexpr int U = 4;  // knots in flight per thread
  float T = 0.f;
  for (int kb = kr.lo + threadIdx.x; kb <= kr.hi; kb += U * blockDim.x) {
    Pair l[U];
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kb + u * int(blockDim.x);
      const uint32_t kc = uint32_t(k <= kr.hi ? k : kr.hi);
      l[u] = ld_pair(g.wave, kc - 1);
      v[u] = ld_at(S, kc);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float wl = mul_nocontract(l[u].lo, a), w = mul_nocontract(l[u].hi, a);
      T += in_range(tg, w) && kb + u * int(blockDim.x) <= kr.hi ? v[u] * (w - wl) : 0.f;
    }
  }
  return T;
}

// Wave total of v in a fixed order through DPP moves (rows of 16, then the rows
// in order); every lane of the wave active.
__device__ inline float wave_total(float v) {
  auto plus = [](float x, int moved) { return x + __int_as_float(moved); };
  v = plus(v, __builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
  v = plus(v, __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));
  v = plus(v, __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xF, 0xF, false));
  v = plus(v, __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, false));
  float t = 0.f;
#pragma unroll
  for (int r = 0; r < 64; r += 16)
    t += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), r));
  return t;
}

// The totals over the workgroup of K values, the waves in order; every thread
// gets them.  sm: K times the wavefronts, free since a barrier.
template <int K>
__device__ inline void block_totals(float (&v)[K], float* sm) {
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int q = 0; q < K; ++q) v[q] = wave_total(v[q]);
  if ((threadIdx.x & 63) == 0)
    for (int q = 0; q < K; ++q) sm[w * K + q] = v[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q) {
    float t = 0.f;
    for (int k = 0; k < nw; ++k) t += sm[k * K + q];
    v[q] = t;
  }
}

__device__ inline float nan_to_num(float v) {
  if (isnan(v)) return 0.f;
  return isinf(v) ? (v > 0.f ? FLT_MAX : -FLT_MAX) : v;
}

// One workgroup per star.  kLds: the P_j wait in LDS for their common factor
// (targets of up to 16384 bins) and each output is written once.  200 k stars,
// 5000 -> 3721: 6.3 ms with an exact walk to every segment from its locator
// cell, a division per bin and the outputs written twice; 2.65 now.
template <bool kLds>
__global__ void __launch_bounds__(kStepThreads) resample_kernel(
    SspView g, rbx_target tg, const float* __restrict__ spectra, const float* __restrict__ vel,
    int64_t vstride, int vcomp, float c, int64_t n, float* __restrict__ out) {
  extern __shared__ float Ps[];
  __shared__ float sm[2 * (kStepThreads / 64)];
  const int ns = g.n_wave, nt = tg.n;
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const float* S = spectra + r * ns;
    float* o = out + r * nt;
    const float a = doppler_factor(vel[r * vstride + vcomp], c);
    const Shift h = shift_of(g, a, 1.0f / a);
    float Nn = 0.f;
    for (int jb = threadIdx.x; jb < nt; jb += kBins * kStepThreads) {
      // kBins bins at a time: each waits on a chain of three loads
      float x[kBins], d[kBins];
#pragma unroll
      for (int u = 0; u < kBins; ++u) {
        const int j = jb + u * kStepThreads;
        const uint32_t jc = uint32_t(j < nt ? j : nt - 1);
        x[u] = ld_at(tg.wave, jc);
        d[u] = j < nt ? ld_at(tg.dwave, jc) : 0.f;
      }
      Knots K[kBins];
      knots_group<kBins, false>(g, x, h, K);
      Pair s[kBins];
#pragma unroll
      for (int u = 0; u < kBins; ++u) s[u] = ld_pair(S, K[u].i0);
#pragma unroll
      for (int u = 0; u < kBins; ++u) {
        const int j = jb + u * kStepThreads;
        const float P = s[u].lo + K[u].theta * (s[u].hi - s[u].lo);
        if (j < nt) {
          (kLds ? Ps : o)[j] = P;
          Nn += P * d[u];
        }
      }
    }
    float sums[2] = {source_total(g, tg, S, mask_range(g, tg, h), a), Nn};
    __syncthreads();  // the star before is done with sm
    block_totals<2>(sums, sm);
    const float sf = nan_to_num(sums[0] / sums[1]);
    // each thread rescales the bins it wrote itself
    for (int j = threadIdx.x; j < nt; j += blockDim.x) o[j] = (kLds ? Ps : o)[j] * sf;
  }
}

// Adjoint of resample_kernel for one star per workgroup.
//   P_j from the input spectrum S, out_j = P_j sf, sf = T / Nn.
//   sbar = sum_j g_j P_j; Pbar_j = g_j sf + Nbar d_j with Nbar = -sbar T / Nn^2
//   (0 when T / Nn is not finite), Tbar = sbar / Nn.
//   Sbar_k gathers the interpolation weights of every target bin whose
//   segment touches knot k (first[k] = first target bin with segment index
//   >= k, built without conflicts because segment indices are monotone in
//   j), plus Tbar (w_k - w_{k-1}) inside the mask window.
//   abar = sum_j Pbar_j dP_j/da + Tbar T / a; dv = abar a / c.
// One pass over the bins forms everything that is summed: T, Nn, sbar and
// dP_j/da weighted by g_j and by d_j apart (their combination follows from
// the first three; they cancel strongly and are added in double).  It leaves
// each bin's weight theta and g_j in LDS, then Pbar_j takes g_j's place and
// the knots gather.  LDS: theta, g (float) and seg (uint16) per target bin,
// first[] (uint16) per knot; first[] is reset to n_target before it is
// filled, so every index read from it stays in [0, n_target] whatever the
// target ordering.  200 k stars, 5000 -> 3721: 28.0 ms with two walks to every
// segment, two passes of divisions, 4 wavefronts a workgroup and one thread
// filling first[] below the first bin; 6.0 now (VALU issue alone: 3.3).
__global__ void __launch_bounds__(kBwdThreads) __attribute__((amdgpu_waves_per_eu(6)))
resample_bwd_kernel(
    SspView g, rbx_target tg, const float* __restrict__ spectra, const float* __restrict__ vel,
    int64_t vstride, int vcomp, float c, int64_t n, const float* __restrict__ dout,
    float* __restrict__ dspec, float* __restrict__ dv) {
  extern __shared__ char lds[];
  __shared__ float sm[3 * (kBwdThreads / 64)];
  __shared__ double sma[2 * (kBwdThreads / 64)];
  const int ns = g.n_wave, nt = tg.n;
  float* th = reinterpret_cast<float*>(lds);
  float* gp = th + nt;
  uint16_t* seg = reinterpret_cast<uint16_t*>(gp + nt);
  uint16_t* first = seg + nt;  // ns + 2 entries
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const float* S = spectra + r * ns;
    const float* gj = dout + r * nt;
    float* dS = dspec ? dspec + r * ns : nullptr;
    const float a = doppler_factor(vel[r * vstride + vcomp], c);
    const Shift h = shift_of(g, a, 1.0f / a);
    __syncthreads();  // the star before is done with th, gp and first
    const KnotRange kr = mask_range(g, tg, h);
    float Nn = 0.f, sbar = 0.f;
    double Ag = 0.0, Ad = 0.0;
    const int step = int(blockDim.x);
    for (int jb = threadIdx.x; jb < nt; jb += kBwdBins * step) {
      float x[kBwdBins], d[kBwdBins], gv[kBwdBins];
#pragma unroll
      for (int u = 0; u < kBwdBins; ++u) {
        const int j = jb + u * step;
        const uint32_t jc = uint32_t(j < nt ? j : nt - 1);
        x[u] = ld_at(tg.wave, jc);
        d[u] = ld_at(tg.dwave, jc);
        gv[u] = ld_at(gj, jc);
      }
      Knots K[kBwdBins];
      knots_group<kBwdBins, true>(g, x, h, K);
      Pair s[kBwdBins];
#pragma unroll
      for (int u = 0; u < kBwdBins; ++u) s[u] = ld_pair(S, K[u].i0);
#pragma unroll
      for (int u = 0; u < kBwdBins; ++u) {
        const int j = jb + u * step;
        if (j >= nt) continue;
        const float ds = s[u].hi - s[u].lo;
        const float P = s[u].lo + K[u].theta * ds;
        Nn += P * d[u];
        sbar += gv[u] * P;
        const double q = -double(ds) * double(K[u].kappa);  // dP_j / da
        Ag += double(gv[u]) * q;
        Ad += double(d[u]) * q;
        th[j] = K[u].theta;
        gp[j] = gv[u];
        seg[j] = uint16_t(K[u].i0 + 1);
      }
    }
    if (dS)
      for (int k = threadIdx.x; k <= ns + 1; k += blockDim.x) first[k] = uint16_t(nt);
    float sums[3] = {source_total(g, tg, S, kr, a), Nn, sbar};
    Ag = wave_sum(Ag);
    Ad = wave_sum(Ad);
    if ((threadIdx.x & 63) == 0) {
      sma[2 * (threadIdx.x >> 6)] = Ag;
      sma[2 * (threadIdx.x >> 6) + 1] = Ad;
    }
    block_totals<3>(sums, sm);  // also a barrier: seg[] and first[] are complete
    const float T = sums[0], N = sums[1];
    const float raw = T / N;
    const bool live = isfinite(raw);
    const float sf = nan_to_num(raw);
    const double Nbar = live ? -double(sums[2]) * T / (double(N) * N) : 0.0;
    const double Tbar = live ? double(sums[2]) / N : 0.0;
    if (dS) {
      for (int j = threadIdx.x; j < nt; j += blockDim.x) {
        gp[j] = float(double(gp[j]) * sf + Nbar * ld_at(tg.dwave, uint32_t(j)));
        if (j > 0)
          for (int k = int(seg[j - 1]) + 1; k <= int(seg[j]); ++k) first[k] = uint16_t(j);
      }
      // the knots before the first bin (a third of a grid that starts well
      // below the targets) by all threads
      for (int k = threadIdx.x; k <= int(seg[0]); k += blockDim.x) first[k] = 0;
      __syncthreads();
      const float Tb = float(Tbar);
      for (int k = threadIdx.x; k < ns; k += blockDim.x) {
        float acc = 0.f;
        const int f0 = first[k], f1 = first[k + 1], f2 = first[k + 2];
        for (int j = f0; j < f1; ++j) acc += gp[j] * th[j];          // segments i = k
        for (int j = f1; j < f2; ++j) acc += gp[j] * (1.f - th[j]);  // segments i = k + 1
        if (k >= kr.lo && k <= kr.hi) {
          const Pair l = ld_pair(g.wave, uint32_t(k - 1));
          const float wl = mul_nocontract(l.lo, a), w = mul_nocontract(l.hi, a);
          if (in_range(tg, w)) acc += Tb * (w - wl);
        }
        dS[k] = acc;
      }
    }
    if (threadIdx.x == 0 && dv) {
      double Agt = 0.0, Adt = 0.0;
      for (int w = 0; w < int(blockDim.x >> 6); ++w) {
        Agt += sma[2 * w];
        Adt += sma[2 * w + 1];
      }
      const double ab = double(sf) * Agt + Nbar * Adt + Tbar * (double(T) / a);
      dv[r] = float(ab * a / c);
    }
  }
}

// ------------------------------------------------------------ segment cube

// Item: (chunk, tile of 256 bins), a wavefront with four consecutive bins per
// lane (200 k x 3721: 0.96 ms with one bin per lane, 0.71 now).
constexpr int kSegTile = 256;

__global__ void __launch_bounds__(64) segment_accum_kernel(
    const float* __restrict__ spectra, const int32_t* __restrict__ perm, int nt,
    const ChunkDesc* __restrict__ desc, const int32_t* __restrict__ n_chunks_ptr, int n_tiles,
    double* __restrict__ partial) {
  const int tile = blockIdx.x % n_tiles;
  const int chunk = blockIdx.x / n_tiles;
  if (chunk >= *n_chunks_ptr) return;
  const ChunkDesc dd = desc[chunk];
  const int j = tile * kSegTile + 4 * int(threadIdx.x);
  if (j >= nt) return;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  double* o = partial + int64_t(chunk) * nt + j;
  if (j + 4 <= nt) {
    const float* col = spectra + j;
#pragma unroll 4
    for (int r = dd.begin; r < dd.end; ++r) {
      const Quad v = *reinterpret_cast<const Quad*>(col + int64_t(perm[r]) * nt);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += v.v[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = acc[e];
  } else {
    for (int e = 0; j + e < nt; ++e) {
      double t = 0.0;
      for (int r = dd.begin; r < dd.end; ++r) t += spectra[int64_t(perm[r]) * nt + j + e];
      o[e] = t;
    }
  }
}

// One workgroup per star: its spaxel's row, or zeros (200 k x 3721: 1.43 ms
// with an index division per element, 0.77 now).
__global__ void __launch_bounds__(kStepThreads) segment_bwd_kernel(
    const float* __restrict__ dcube, const int32_t* __restrict__ ids, int64_t n, int n_spaxel,
    int nt, float* __restrict__ dspec) {
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const int32_t p = ids[r];
    const bool ok = p >= 0 && p < n_spaxel;
    const float* src = dcube + int64_t(ok ? p : 0) * nt;
    float* o = dspec + r * nt;
    row_quads(
        nt, threadIdx.x, kStepThreads,
        [&](int k) {
          Quad v = ld_quad(src, uint32_t(k));
          if (!ok) v = {{0.f, 0.f, 0.f, 0.f}};
          st_quad(o, uint32_t(k), v);
        },
        [&](int k) { o[k] = ok ? src[k] : 0.f; });
  }
}

struct SegLayout {
  int32_t *perm, *offsets, *chunk_off, *scan_blocks;
  ChunkDesc* desc;
  double* partial;
  void* sort_ws;
  size_t sort_ws_bytes;
  int64_t max_chunks;
};

template <class C>
static void seg_layout(C& c, int64_t n, int32_t n_keys, int32_t nt, SegLayout* L) {
  const int64_t max_chunks = (n + kChunk - 1) / kChunk + n_keys;
  const size_t sort_bytes = sort_workspace_size(n, n_keys);
  auto* perm = c.template take<int32_t>(n > 0 ? n : 1);
  auto* offs = c.template take<int32_t>(size_t(n_keys) + 1);
  auto* coff = c.template take<int32_t>(size_t(n_keys) + 1);
  auto* blocks = c.template take<int32_t>((size_t(n_keys) + 1) / 4096 + 2);
  auto* desc = c.template take<ChunkDesc>(max_chunks);
  auto* part = c.template take<double>(size_t(max_chunks) * nt);
  auto* sws = c.template take<char>(sort_bytes);
  if (L) {
    L->perm = reinterpret_cast<int32_t*>(perm);
    L->offsets = reinterpret_cast<int32_t*>(offs);
    L->chunk_off = reinterpret_cast<int32_t*>(coff);
    L->scan_blocks = reinterpret_cast<int32_t*>(blocks);
    L->desc = reinterpret_cast<ChunkDesc*>(desc);
    L->partial = reinterpret_cast<double*>(part);
    L->sort_ws = sws;
    L->sort_ws_bytes = sort_bytes;
    L->max_chunks = max_chunks;
  }
}

struct SizeOnly2 {
  Sizer s;
  template <class T>
  T* take(size_t count) {
    s.take<T>(count);
    return nullptr;
  }
};

static int blocks_for_rows(int64_t n) { return int(n < (1 << 20) ? (n > 0 ? n : 1) : (1 << 20)); }

static int grid_for(int64_t n, int threads) {
  int64_t gsz = (n + threads - 1) / threads;
  if (gsz < 1) gsz = 1;
  if (gsz > (1 << 20)) gsz = 1 << 20;
  return int(gsz);
}

static bool ssp_ok(const rbx_ssp* s, bool need_wave) {
  if (!s || !s->flux || !s->ax_met || !s->ax_age || s->n_met < 2 || s->n_age < 2 || s->n_wave < 2)
    return false;
  if (need_wave && (!s->wave_obs || !s->locate || s->n_locate < 1 || !(s->locate_inv_h > 0.f)))
    return false;
  return true;
}

// Two bins in flight a thread at least, so a short axis takes fewer threads.
static int bwd_threads(int nt) { return nt <= 1024 ? 256 : kBwdThreads; }

static size_t resample_bwd_lds(int nt, int ns) {
  return size_t(nt) * 2 * 4 + size_t(nt) * 2 + size_t(ns + 2) * 2;
}

}  // namespace rbx

extern "C" {

int rbx_ssp_lookup(const rbx_ssp* ssp, const float* met, const float* age, int64_t n,
                   float* spectra, void* stream) {
  using namespace rbx;
  if (!ssp_ok(ssp, false) || n < 0 || (n > 0 && (!met || !age || !spectra)))
    return fail(RBX_EINVAL, "rbx_ssp_lookup: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL(lookup_kernel, dim3(blocks_for_rows(n)), dim3(kStepThreads), 0,
                     as_stream(stream), view_of(*ssp), met, age, n, spectra);
  return check_launch("rbx_ssp_lookup");
}

int rbx_ssp_lookup_bwd(const rbx_ssp* ssp, const float* met, const float* age, int64_t n,
                       const float* dspectra, float* dmet, float* dage, void* stream) {
  using namespace rbx;
  if (!ssp_ok(ssp, false) || n < 0 || (n > 0 && (!met || !age || !dspectra)))
    return fail(RBX_EINVAL, "rbx_ssp_lookup_bwd: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL(lookup_bwd_kernel, dim3(blocks_for_rows(n)), dim3(kStepThreads), 0,
                     as_stream(stream), view_of(*ssp), met, age, n, dspectra, dmet, dage);
  return check_launch("rbx_ssp_lookup_bwd");
}

int rbx_scale_rows(const float* in, const float* scale, int64_t n, int32_t nw, float* out,
                   void* stream) {
  using namespace rbx;
  if (n < 0 || nw < 1 || (n > 0 && (!in || !scale || !out)))
    return fail(RBX_EINVAL, "rbx_scale_rows: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL((scale_rows_kernel<true, false>), dim3(blocks_for_rows(n)), dim3(kStepThreads),
                     0, as_stream(stream), in, scale, nullptr, n, nw, out, nullptr);
  return check_launch("rbx_scale_rows");
}

int rbx_row_dot(const float* a, const float* b, int64_t n, int32_t nw, float* out, void* stream) {
  using namespace rbx;
  if (n < 0 || nw < 1 || (n > 0 && (!a || !b || !out)))
    return fail(RBX_EINVAL, "rbx_row_dot: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL((scale_rows_kernel<false, true>), dim3(blocks_for_rows(n)), dim3(kStepThreads),
                     0, as_stream(stream), a, nullptr, b, n, nw, nullptr, out);
  return check_launch("rbx_row_dot");
}

int rbx_scale_rows_bwd(const float* dout, const float* scale, const float* in, int64_t n,
                       int32_t nw, float* din, float* dscale, void* stream) {
  using namespace rbx;
  if (n < 0 || nw < 1 || (n > 0 && (!dout || !scale || !in || !din || !dscale)))
    return fail(RBX_EINVAL, "rbx_scale_rows_bwd: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL((scale_rows_kernel<true, true>), dim3(blocks_for_rows(n)), dim3(kStepThreads), 0,
                     as_stream(stream), dout, scale, in, n, nw, din, dscale);
  return check_launch("rbx_scale_rows_bwd");
}

int rbx_resample(const rbx_ssp* ssp, const rbx_target* tg, const float* spectra,
                 const float* velocity, int64_t vel_stride, int32_t vel_comp, float c, int64_t n,
                 float* out, void* stream) {
  using namespace rbx;
  if (!ssp_ok(ssp, true) || !tg || tg->n < 1 || !tg->wave || !tg->dwave || n < 0 ||
      vel_comp < 0 || vel_comp >= vel_stride || !(c > 0.f) ||
      (n > 0 && (!spectra || !velocity || !out)))
    return fail(RBX_EINVAL, "rbx_resample: bad arguments");
  if (n == 0) return RBX_OK;
  const size_t lds = size_t(tg->n) * sizeof(float);
  if (lds <= 64 * 1024)
    hipLaunchKernelGGL(resample_kernel<true>, dim3(blocks_for_rows(n)), dim3(kStepThreads), lds,
                       as_stream(stream), view_of(*ssp), *tg, spectra, velocity, vel_stride,
                       vel_comp, c, n, out);
  else
    hipLaunchKernelGGL(resample_kernel<false>, dim3(blocks_for_rows(n)), dim3(kStepThreads), 0,
                       as_stream(stream), view_of(*ssp), *tg, spectra, velocity, vel_stride,
                       vel_comp, c, n, out);
  return check_launch("rbx_resample");
}

int rbx_resample_bwd(const rbx_ssp* ssp, const rbx_target* tg, const float* spectra,
                     const float* velocity, int64_t vel_stride, int32_t vel_comp, float c,
                     int64_t n, const float* dout, float* dspectra, float* dvlos, void* stream) {
  using namespace rbx;
  if (!ssp_ok(ssp, true) || !tg || tg->n < 1 || !tg->wave || !tg->dwave || n < 0 ||
      vel_comp < 0 || vel_comp >= vel_stride || !(c > 0.f) ||
      (n > 0 && (!spectra || !velocity || !dout)))
    return fail(RBX_EINVAL, "rbx_resample_bwd: bad arguments");
  const size_t lds = resample_bwd_lds(tg->n, ssp->n_wave);
  if (lds > 64 * 1024 || tg->n > 65535 || ssp->n_wave > 65533)
    return fail(RBX_EINVAL, "rbx_resample_bwd: 10*n_target + 2*n_wave bytes must fit 64 KiB of LDS");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL(resample_bwd_kernel, dim3(blocks_for_rows(n)), dim3(bwd_threads(tg->n)), lds,
                     as_stream(stream), view_of(*ssp), *tg, spectra, velocity, vel_stride, vel_comp,
                     c, n, dout, dspectra, dvlos);
  return check_launch("rbx_resample_bwd");
}

size_t rbx_segment_cube_workspace_size(int64_t n, int32_t n_keys, int32_t n_wave) {
  using namespace rbx;
  if (n < 0 || n_keys < 1 || n_wave < 1) return 0;
  SizeOnly2 so;
  seg_layout(so, n, n_keys, n_wave, nullptr);
  return so.s.used;
}

int rbx_segment_cube(const float* spectra, const int32_t* ids, int64_t n, int32_t n_spaxel,
                     int32_t n_keys, int32_t n_wave, float* cube, void* workspace,
                     size_t workspace_bytes, void* stream) {
  using namespace rbx;
  if (n < 0 || n_spaxel < 1 || n_keys < n_spaxel || n_wave < 1 || !cube ||
      (n > 0 && (!spectra || !ids)))
    return fail(RBX_EINVAL, "rbx_segment_cube: bad arguments");
  if (n > INT32_MAX - 1) return fail(RBX_EINVAL, "rbx_segment_cube: n must fit int32");
  hipStream_t s = as_stream(stream);
  Carver cv(workspace, workspace_bytes);
  SegLayout L;
  seg_layout(cv, n, n_keys, n_wave, &L);
  if (!cv.ok) return fail(RBX_EWORKSPACE, "rbx_segment_cube: workspace too small");
  int rc = spaxel_sort_impl(ids, n, n_keys, L.perm, nullptr, L.offsets, L.sort_ws, L.sort_ws_bytes, s);
  if (rc) return rc;
  rc = build_chunks(L.offsets, n_spaxel, kChunk, L.chunk_off, L.scan_blocks, L.desc, s);
  if (rc) return rc;
  const int n_tiles = (n_wave + kSegTile - 1) / kSegTile;
  const int64_t max_chunks = (n + kChunk - 1) / kChunk + n_spaxel;
  if (n > 0) {
    const int64_t blocks = int64_t(n_tiles) * max_chunks;
    if (blocks > INT32_MAX) return fail(RBX_EINVAL, "rbx_segment_cube: problem too large");
    hipLaunchKernelGGL(segment_accum_kernel, dim3(blocks), dim3(64), 0, s, spectra, L.perm, n_wave,
                       L.desc, L.chunk_off + n_spaxel, n_tiles, L.partial);
  }
  combine_chunks(L.partial, L.chunk_off, n_spaxel, n_wave, cube, s);
  return check_launch("rbx_segment_cube");
}

int rbx_segment_cube_bwd(const float* dcube, const int32_t* ids, int64_t n, int32_t n_spaxel,
                         int32_t n_wave, float* dspectra, void* stream) {
  using namespace rbx;
  if (n < 0 || n_spaxel < 1 || n_wave < 1 || (n > 0 && (!dcube || !ids || !dspectra)))
    return fail(RBX_EINVAL, "rbx_segment_cube_bwd: bad arguments");
  if (n == 0) return RBX_OK;
  hipLaunchKernelGGL(segment_bwd_kernel, dim3(blocks_for_rows(n)), dim3(kStepThreads), 0,
                     as_stream(stream), dcube, ids, n, n_spaxel, n_wave, dspectra);
  return check_launch("rbx_segment_cube_bwd");
}

}  // extern "C"
