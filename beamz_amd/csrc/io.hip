// Source injection and DFT-monitor accumulation kernels for gfx950.
//
//   slab sources: beamz/simulation/execute.py:374-461 (field[start:start+size]
//                 += coeff * waveform[clip(step, 0, T-1)]); post-update timings
//                 skip PEC-constrained cells (equivalent to re-masking,
//                 execute.py:488-521)
//   DFT monitors: beamz/simulation/observe.py:315-357 (gating, window),
//                 observe.py:529-585 (weighted gather and accumulation)
//
// The DFT accumulators and their phase factors are float64: the phase
// 2*pi*f*t_phys is evaluated in float64 from t_phys = t + (k + 1) dt.

#include <algorithm>
#include <climits>

#include "common.h"

namespace bzh {
namespace {

template <typename T>
__global__ void __launch_bounds__(256) source_kernel(SourceParams p) {
  const int cx = blockIdx.x * 64 + threadIdx.x;
  const int cy = blockIdx.y * 4 + threadIdx.y;
  const int cz = blockIdx.z;
  if (cx >= p.sdims[2] || cy >= p.sdims[1] || cz >= p.sdims[0]) return;
  int widx = *p.step0 + p.k;
  widx = widx < 0 ? 0 : (widx > p.T - 1 ? p.T - 1 : widx);
  const int slab_cells = p.sdims[0] * p.sdims[1] * p.sdims[2];
  const int c = (cz * p.sdims[1] + cy) * p.sdims[2] + cx;
  T* f = static_cast<T*>(p.field);
  for (int s = p.slab0; s < p.slab0 + p.nslabs; ++s) {
    const int z = p.starts[s * 3 + 0] + cz;
    const int y = p.starts[s * 3 + 1] + cy;
    const int x = p.starts[s * 3 + 2] + cx;
    if (z < 0 || y < 0 || x < 0 || z >= p.fdims[0] || y >= p.fdims[1] || x >= p.fdims[2]) continue;
    if ((p.mlo[0] && z == 0) || (p.mhi[0] && z == p.fdims[0] - 1) ||
        (p.mlo[1] && y == 0) || (p.mhi[1] && y == p.fdims[1] - 1) ||
        (p.mlo[2] && x == 0) || (p.mhi[2] && x == p.fdims[2] - 1))
      continue;
    const int o = (z * p.fdims[1] + y) * p.fdims[2] + x;
    const float add = p.coeff[static_cast<int64_t>(s) * slab_cells + c] *
                      p.wave[static_cast<int64_t>(s) * p.T + widx] * p.scale;
    store_f(f, o, load_f(f, o) + add);
  }
}

constexpr int kDftBlock = 128;
constexpr int kMaxFreq = 256;

// Weighted gather of one monitor sample (observe.py:360-370, 529-585),
// from the field or, when ``p.cap`` is set, from the capture of the
// monitored cells (the corner's cell mapped into its component's box).
//
// Four corners at a time: their indices and weights, then their cells, are
// loaded before the first is summed (one corner after another cost three
// dependent round trips each).  Corners outside the component add nothing, and
// are read at element 0 instead.
template <typename T>
__device__ __forceinline__ float gather(const DftParams& p, const T* fld, const float* cap, int m,
                                        int c, int pt) {
  const int64_t base = ((static_cast<int64_t>(m) * 6 + c) * p.Pmax + pt) * p.K;
  const int32_t* t = p.capbox + (m * 6 + c) * 8;
  const int sy = p.fdims[c][1], sx = p.fdims[c][2];
  float v = 0.0f;
  for (int q0 = 0; q0 < p.K; q0 += 4) {
    int idx[4];
    float w[4], x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int q = min(q0 + e, p.K - 1);
      idx[e] = p.indices[base + q];
      w[e] = q0 + e < p.K ? p.weights[base + q] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (idx[e] < 0 || idx[e] >= p.fsize[c]) w[e] = 0.0f;
      int cell = w[e] != 0.0f ? idx[e] : 0;
      if (cap != nullptr) {
        const int nzb = t[1] - t[0] + 1, nyb = t[3] - t[2] + 1;
        const int cz = cell / (sy * sx), r = cell - cz * (sy * sx);
        const int cy = r / sx, cx = r - cy * sx;
        if (cz < t[0] || cz > t[1] || cy < t[2] || cy > t[3] || cx < t[4] || cx > t[5]) w[e] = 0.0f;
        cell = w[e] != 0.0f ? t[6] + ((cx - t[4]) * nyb + (cy - t[2])) * nzb + (cz - t[0]) : 0;
        x[e] = cap[cell];
      } else {
        x[e] = load_f(fld, cell);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v = w[e] != 0.0f ? v + w[e] * x[e] : v;
  }
  return v;
}

// sin and cos of 2 pi x for x turns.  Dropping whole turns first is exact and
// spares sincos its reduction of arguments in the thousands, which took most
// of a flush (the product f t carries the same relative rounding either way).
__device__ __forceinline__ void phase_factor(double x, double& sn, double& cs) {
  sincospi(2.0 * (x - rint(x)), &sn, &cs);
}

// Gate, window and amplitude factor of step k of this call for monitor m
// (observe.py:315-357).  Returns false when the step is not sampled.
__device__ __forceinline__ bool dft_gate(const DftParams& p, int m, int k, double& t,
                                         double& window, double& scale) {
  const int interval = p.counts[m * 5 + 2] > 1 ? p.counts[m * 5 + 2] : 1;
  const int step = *p.step0 + k;
  const double t0 = p.time_f64 ? *static_cast<const double*>(p.time)
                               : static_cast<double>(*static_cast<const float*>(p.time));
  t = t0 + static_cast<double>(k + 1) * p.dt;
  const double ts = p.windows[m * 3 + 0];
  const double te = p.windows[m * 3 + 1];
  if (!(t >= ts && t <= te) || (step % interval) != 0) return false;
  window = 1.0;
  if (p.codes[m * 2 + 0] == 1 && isfinite(te) && te > ts) {
    double tau = (t - ts) / fmax(te - ts, 1e-30);
    tau = fmin(fmax(tau, 0.0), 1.0);
    window = 0.5 * (1.0 - cos(2.0 * M_PI * tau));
  }
  scale = fmax(window, 0.0);
  if (p.codes[m * 2 + 1] == 1) {
    const double lu = p.windows[m * 3 + 2];
    scale *= (p.dt * interval * 299792458.0 / lu) / sqrt(2.0 * M_PI);
  }
  return true;
}

// Buffered path, step k: stage the gathered sample (f32) in ring slot k % slots;
// with p.pair also step k + 1's, from field2 (blockIdx.y 1).  A strided plane
// is bound by the lines of its cells, a small one by the launch: three
// 128 x 256 planes normal to x take 26 us for both steps (two launches: 34),
// two 64 x 96 ones 5.5 us (11).
template <typename T>
__global__ void __launch_bounds__(kDftBlock) dft_stage_kernel(DftParams p) {
  const int m = blockIdx.z / 6;
  const int c = blockIdx.z % 6;
  const bool second = blockIdx.y != 0;
  const int k = p.k + blockIdx.y;
  const int P = p.counts[m * 5 + 1];
  double t, window, scale;
  if (!dft_gate(p, m, k, t, window, scale)) return;
  const int pt = blockIdx.x * kDftBlock + threadIdx.x;
  const T* fld = static_cast<const T*>(second ? p.field2[c] : p.field[c]);
  if (p.masks[m * 6 + c] == 0.0f || pt >= P || pt >= p.Pmax || fld == nullptr) return;
  const int64_t slot = k % p.slots;
  p.stage[((slot * p.M + m) * 6 + c) * p.Pmax + pt] =
      gather<T>(p, fld, second ? nullptr : p.cap, m, c, pt);
}

// Fold steps k0 .. k0+nk-1 into the accumulators of frequencies f0 .. f0+kFt-1
// (blockIdx.y picks the tile), given each step's gathered sample v[j].  A
// step's term is formed exactly as in the direct path (f32 sample times
// 1/scale, mask and amplitude in f64, times the f64 phase factor); the nk
// terms of one (frequency, point) are summed in f64 and added once.
constexpr int kFt = 8;
struct FlushLds {
  double t[kDftMaxSlots], scale[kDftMaxSlots], win[kDftMaxSlots];
  int on[kDftMaxSlots];
  double cs[kDftMaxSlots][kFt], sn[kDftMaxSlots][kFt];
  float v[kDftMaxSlots][kDftBlock];  // each thread's samples (its own column)
};
// The steps' gates, the window sums and the phase factors of this block.
template <typename A>
__device__ __forceinline__ void flush_begin(const DftParams& p, int m, int c, FlushLds& l) {
  const int nk = p.nk < kDftMaxSlots ? p.nk : kDftMaxSlots;
  const int F = p.counts[m * 5 + 0], nf = F < p.Fmax ? F : p.Fmax;
  const int64_t woff = p.counts[m * 5 + 4];
  const int f0 = blockIdx.y * kFt;
  // this thread's frequency (its table entries e = threadIdx.x + i kDftBlock
  // all have column e % kFt)
  const int ft = f0 + static_cast<int>(threadIdx.x) % kFt;
  double fr = 0.0;
  if (ft < nf)
    fr = p.freqs_f64 ? static_cast<const double*>(p.freqs)[m * p.Fmax + ft]
                     : static_cast<double>(static_cast<const float*>(p.freqs)[m * p.Fmax + ft]);
  if (threadIdx.x < kDftMaxSlots) {
    double t = 0.0, window = 0.0, scale = 0.0;
    const bool on = threadIdx.x < nk && dft_gate(p, m, p.k0 + threadIdx.x, t, window, scale);
    l.t[threadIdx.x] = t;
    l.scale[threadIdx.x] = on ? scale : 0.0;
    l.win[threadIdx.x] = on ? window : 0.0;
    l.on[threadIdx.x] = on ? 1 : 0;
  }
  __syncthreads();
  if (c == 0 && blockIdx.x == 0 && blockIdx.y == 0) {
    A* w = static_cast<A*>(p.wsum);
    for (int f = threadIdx.x; f < nf; f += kDftBlock) {
      double acc = 0.0;
      for (int j = 0; j < nk; ++j) acc += l.win[j];
      if (woff + f < p.w_len) w[woff + f] += static_cast<A>(acc);
    }
  }
  static_assert(kDftBlock % kFt == 0, "a thread's entries share one frequency");
  for (int e = threadIdx.x; e < kDftMaxSlots * kFt; e += kDftBlock) {
    const int j = e / kFt;
    double sn = 0.0, cs = 0.0;
    if (ft < nf && j < nk) phase_factor(fr * l.t[j], sn, cs);
    l.cs[j][e % kFt] = cs;
    l.sn[j][e % kFt] = sn;
  }
  __syncthreads();
}
// The accumulators of (component, frequencies f0 .. f0 + kFt - 1, point),
// loaded before the phase factors are formed: read one frequency after another
// at the end, they were the kernel's longest chain.
template <typename A>
struct FlushAcc {
  A re[kFt], im[kFt];
  int64_t o;       // index of the first; frequency f sits P further per step
  int P, n;        // n live frequencies (0: none)
};
template <typename A>
__device__ __forceinline__ void flush_load(const DftParams& p, int m, int c, int pt, bool live,
                                           FlushAcc<A>& a) {
  const int P = p.counts[m * 5 + 1], F = p.counts[m * 5 + 0], nf = F < p.Fmax ? F : p.Fmax;
  const int f0 = blockIdx.y * kFt;
  a.P = P;
  a.o = p.counts[m * 5 + 3] + (static_cast<int64_t>(c) * F + f0) * P + pt;
  a.n = live ? max(0, min(kFt, nf - f0)) : 0;
#pragma unroll
  for (int f = 0; f < kFt; ++f) {
    const int64_t o = a.o + static_cast<int64_t>(f) * P;
    const bool in = f < a.n && o < p.re_len;
    a.re[f] = in ? static_cast<const A*>(p.re)[o] : A(0);
    a.im[f] = in ? static_cast<const A*>(p.im)[o] : A(0);
  }
}
// (No step or frequency is skipped by a branch: steps past nk and frequencies
// past the last carry zero factors, so that the reads and the 16 independent
// sums pipeline.  The samples wait in LDS: with the step loop unrolled over a
// register array the scheduler spilled.)
template <typename A>
__device__ __forceinline__ void flush_add(const DftParams& p, int m, int c, const FlushLds& l,
                                          const FlushAcc<A>& acc) {
  const float cmask = p.masks[m * 6 + c], inv = p.inv_scale[c];
  double ar[kFt] = {}, ai[kFt] = {};
#pragma unroll 2
  for (int j = 0; j < kDftMaxSlots; ++j) {
    const double t = static_cast<double>(l.v[j][threadIdx.x]) * inv * cmask * l.scale[j];
    const double dv = l.on[j] ? t : 0.0;
#pragma unroll
    for (int f = 0; f < kFt; ++f) {
      ar[f] += dv * l.cs[j][f];
      ai[f] += dv * l.sn[j][f];
    }
  }
  A* re = static_cast<A*>(p.re);
  A* im = static_cast<A*>(p.im);
#pragma unroll
  for (int f = 0; f < kFt; ++f) {
    const int64_t o = acc.o + static_cast<int64_t>(f) * acc.P;
    if (f < acc.n && o < p.re_len) {
      re[o] = acc.re[f] + static_cast<A>(ar[f]);
      im[o] = acc.im[f] + static_cast<A>(ai[f]);
    }
  }
}

// Buffered path: fold the ring's staged samples.  The frequency tiles are
// separate blocks: 96 x 232-point planes of 11 frequencies took 108 us when
// one block walked them all.
template <typename A>
__global__ void __launch_bounds__(kDftBlock) dft_flush_kernel(DftParams p) {
  const int m = blockIdx.z / 6, c = blockIdx.z % 6;
  const int P = p.counts[m * 5 + 1];
  const int pt = blockIdx.x * kDftBlock + threadIdx.x;
  const bool any = p.masks[m * 6 + c] != 0.0f && p.field[c] != nullptr;
  if (!any && c != 0) return;  // (component 0 also adds the window sums)
  const bool live = any && pt < P && pt < p.Pmax;
  FlushAcc<A> acc;
  flush_load<A>(p, m, c, pt, live, acc);
  __shared__ FlushLds l;
  flush_begin<A>(p, m, c, l);
  if (!live) return;
#pragma unroll 8
  for (int j = 0; j < kDftMaxSlots; ++j) {
    const int slot = (p.k0 + min(j, p.nk - 1)) % p.slots;
    l.v[j][threadIdx.x] = p.stage[((static_cast<int64_t>(slot) * p.M + m) * 6 + c) * p.Pmax + pt];
  }
  flush_add<A>(p, m, c, l, acc);
}

// 2D multi-step calls: gather each step's sample from the captured cells and
// fold it, without a launch per step.
template <typename A>
__global__ void __launch_bounds__(kDftBlock) dft_capture_kernel(DftCapParams p) {
  const DftParams& d = p.d;
  const int m = blockIdx.z / 6, c = blockIdx.z % 6;
  const int P = d.counts[m * 5 + 1];
  const int pt = blockIdx.x * kDftBlock + threadIdx.x;
  const int q = c == 2 ? 2 : c - 3;  // (DFT order Ez 2, Hx 3, Hy 4)
  const bool any = (c >= 2 && c <= 4) && d.masks[m * 6 + c] != 0.0f && d.field[c] != nullptr;
  if (!any && c != 0) return;
  // (the gather's loads, four corners at a time, are issued before the phase
  // factors are formed: one corner after another behind them took 32 us for
  // two 180-point lines)
  float v[kDftMaxSlots];
#pragma unroll
  for (int j = 0; j < kDftMaxSlots; ++j) v[j] = 0.0f;
  const bool live = any && pt < P && pt < d.Pmax;
  FlushAcc<A> acc;
  flush_load<A>(d, m, c, pt, live, acc);
  if (live) {
    const TmBox b = p.box[m][q];
    const int64_t base = ((static_cast<int64_t>(m) * 6 + c) * d.Pmax + pt) * d.K;
    const int sx = d.fdims[c][2];
    for (int e0 = 0; e0 < d.K; e0 += 4) {
      int idx[4];
      float w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = e0 + e < d.K;
        idx[e] = in ? d.indices[base + e0 + e] : -1;
        w[e] = in ? d.weights[base + e0 + e] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int y = idx[e] / sx, x = idx[e] - y * sx;
        if (w[e] == 0.0f || idx[e] < 0 || idx[e] >= d.fsize[c] || y < b.y0 || y > b.y1 || x < b.x0 ||
            x > b.x1)
          continue;
        const float* cell = p.cap + b.off + (y - b.y0) * (b.x1 - b.x0 + 1) + (x - b.x0);
#pragma unroll
        for (int j = 0; j < kDftMaxSlots; ++j)
          v[j] += w[e] * cell[static_cast<int64_t>(min(j, d.nk - 1)) * p.cap_cells];
      }
    }
  }
  __shared__ FlushLds l;
#pragma unroll
  for (int j = 0; j < kDftMaxSlots; ++j) l.v[j][threadIdx.x] = v[j];
  flush_begin<A>(d, m, c, l);
  if (!live) return;
  flush_add<A>(d, m, c, l, acc);
}

template <typename T, typename A>
__global__ void __launch_bounds__(kDftBlock) dft_kernel(DftParams p) {
  const int m = blockIdx.z / 6;
  const int c = blockIdx.z % 6;
  const int P = p.counts[m * 5 + 1];
  const int F = p.counts[m * 5 + 0];
  const int interval = p.counts[m * 5 + 2] > 1 ? p.counts[m * 5 + 2] : 1;
  const int64_t voff = p.counts[m * 5 + 3];
  const int64_t woff = p.counts[m * 5 + 4];
  const int step = *p.step0 + p.k;
  const double t0 = p.time_f64 ? *static_cast<const double*>(p.time)
                               : static_cast<double>(*static_cast<const float*>(p.time));
  const double t = t0 + static_cast<double>(p.k + 1) * p.dt;
  const double ts = p.windows[m * 3 + 0];
  const double te = p.windows[m * 3 + 1];
  // observe.py:315-338: gate on the time window and the sampling interval
  if (!(t >= ts && t <= te) || (step % interval) != 0) return;
  double window = 1.0;
  if (p.codes[m * 2 + 0] == 1 && isfinite(te) && te > ts) {
    double tau = (t - ts) / fmax(te - ts, 1e-30);
    tau = fmin(fmax(tau, 0.0), 1.0);
    window = 0.5 * (1.0 - cos(2.0 * M_PI * tau));
  }
  double scale = fmax(window, 0.0);
  if (p.codes[m * 2 + 1] == 1) {
    // observe.py:341-357 physical normalization
    const double lu = p.windows[m * 3 + 2];
    scale *= (p.dt * interval * 299792458.0 / lu) / sqrt(2.0 * M_PI);
  }
  __shared__ double s_cos[kMaxFreq];
  __shared__ double s_sin[kMaxFreq];
  const int nf = F < p.Fmax ? F : p.Fmax;
  for (int f = threadIdx.x; f < nf && f < kMaxFreq; f += kDftBlock) {
    const double fr = p.freqs_f64 ? static_cast<const double*>(p.freqs)[m * p.Fmax + f]
                                  : static_cast<double>(static_cast<const float*>(p.freqs)[m * p.Fmax + f]);
    double sn, cs;
    phase_factor(fr * t, sn, cs);
    s_cos[f] = cs;
    s_sin[f] = sn;
  }
  __syncthreads();
  // weight sum: one thread per monitor adds the window for each frequency
  if (c == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
    A* w = static_cast<A*>(p.wsum);
    for (int f = 0; f < nf; ++f)
      if (woff + f < p.w_len) w[woff + f] += static_cast<A>(window);
  }
  const float cmask = p.masks[m * 6 + c];
  const int pt = blockIdx.x * kDftBlock + threadIdx.x;
  if (cmask == 0.0f || pt >= P || pt >= p.Pmax || p.field[c] == nullptr) return;
  const float v = gather<T>(p, static_cast<const T*>(p.field[c]), p.cap, m, c, pt);
  const double dv = static_cast<double>(v) * p.inv_scale[c] * cmask * scale;
  A* re = static_cast<A*>(p.re);
  A* im = static_cast<A*>(p.im);
  for (int f = 0; f < nf && f < kMaxFreq; ++f) {
    const int64_t o = voff + (static_cast<int64_t>(c) * F + f) * P + pt;
    if (o < p.re_len) {
      re[o] += static_cast<A>(dv * s_cos[f]);
      im[o] += static_cast<A>(dv * s_sin[f]);
    }
  }
}

template <typename T>
void dft_dispatch(hipStream_t s, const DftParams& p) {
  dim3 block(kDftBlock, 1, 1);
  dim3 grid((p.Pmax + kDftBlock - 1) / kDftBlock, 1, p.M * 6);
  if (p.mode == 1) {
    grid.y = p.pair != 0 ? 2 : 1;
    hipLaunchKernelGGL((dft_stage_kernel<T>), grid, block, 0, s, p);
  } else if (p.mode == 2) {
    grid.y = std::max(1, (p.Fmax + kFt - 1) / kFt);  // (no frequency: nothing to add)
    if (p.acc_f64) hipLaunchKernelGGL((dft_flush_kernel<double>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((dft_flush_kernel<float>), grid, block, 0, s, p);
  } else {
    if (p.acc_f64) hipLaunchKernelGGL((dft_kernel<T, double>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((dft_kernel<T, float>), grid, block, 0, s, p);
  }
}


// Bounding boxes of the monitors' gather points, for the pair step's
// intermediate bank: box m = [zmin, zmax, ymin, ymax, xmin, xmax] over every
// point the gather reads (weight != 0, index inside the component).  The
// init kernel empties the boxes; blocks (b, m) fold slices of monitor m's
// points in with atomics.
__global__ void __launch_bounds__(64) monbox_init_kernel(MonBoxParams p) {
  const int i = threadIdx.x;
  if (i < p.M * 6) p.box[i] = (i % 2 == 0) ? INT_MAX : INT_MIN;
}

constexpr int kBoxBlock = 256;
constexpr int kBoxSlices = 64;

__global__ void __launch_bounds__(kBoxBlock) monbox_kernel(MonBoxParams p) {
  __shared__ int red[6][kBoxBlock];
  const int m = blockIdx.y;
  int v[6] = {INT_MAX, INT_MIN, INT_MAX, INT_MIN, INT_MAX, INT_MIN};
  const int64_t per = static_cast<int64_t>(p.Pmax) * p.K;
  for (int c = 0; c < 6; ++c) {
    const int Sz = p.dims[c][0], Sy = p.dims[c][1], Sx = p.dims[c][2];
    const int64_t n = static_cast<int64_t>(Sz) * Sy * Sx;
    if (n <= 0) continue;
    const int64_t base = (static_cast<int64_t>(m) * 6 + c) * per;
    for (int64_t i = blockIdx.x * int64_t{kBoxBlock} + threadIdx.x; i < per;
         i += int64_t{kBoxBlock} * gridDim.x) {
      const int idx = p.indices[base + i];
      if (p.weights[base + i] == 0.0f || idx < 0 || idx >= n) continue;
      const int z = idx / (Sy * Sx);
      const int r = idx - z * (Sy * Sx);
      const int y = r / Sx;
      const int x = r - y * Sx;
      v[0] = min(v[0], z);
      v[1] = max(v[1], z);
      v[2] = min(v[2], y);
      v[3] = max(v[3], y);
      v[4] = min(v[4], x);
      v[5] = max(v[5], x);
    }
  }
  for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = v[q];
  __syncthreads();
  for (int h = kBoxBlock / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) {
      for (int q = 0; q < 6; ++q) {
        const int a = red[q][threadIdx.x], b = red[q][threadIdx.x + h];
        red[q][threadIdx.x] = (q % 2 == 0) ? min(a, b) : max(a, b);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int q = 0; q < 6; q += 2) {
      if (red[q][0] != INT_MAX) atomicMin(&p.box[m * 6 + q], red[q][0]);
      if (red[q + 1][0] != INT_MIN) atomicMax(&p.box[m * 6 + q + 1], red[q + 1][0]);
    }
  }
}

}  // namespace

void launch_source(hipStream_t s, const SourceParams& p) {
  if (p.sdims[0] <= 0 || p.sdims[1] <= 0 || p.sdims[2] <= 0 || p.nslabs <= 0) return;
  dim3 block(64, 4, 1);
  dim3 grid((p.sdims[2] + 63) / 64, (p.sdims[1] + 3) / 4, p.sdims[0]);
  switch (p.dtype) {
    case BZH_F32: hipLaunchKernelGGL((source_kernel<float>), grid, block, 0, s, p); break;
    case BZH_BF16: hipLaunchKernelGGL((source_kernel<bf16_t>), grid, block, 0, s, p); break;
    case BZH_F16: hipLaunchKernelGGL((source_kernel<__half>), grid, block, 0, s, p); break;
    default: throw Failure{"unsupported source field dtype"};
  }
  BZH_HIP(hipGetLastError());
}

void launch_dft(hipStream_t s, const DftParams& p) {
  if (p.M <= 0 || p.Pmax <= 0) return;
  BZH_REQUIRE(p.Fmax <= kMaxFreq, "DFT monitors support at most 256 frequencies");
  if (p.mode != 0) {
    BZH_REQUIRE(p.stage != nullptr && p.slots >= 1 && p.slots <= kDftMaxSlots,
                "buffered DFT needs a staging ring of 1..32 slots");
    BZH_REQUIRE(p.pair == 0 || (p.mode == 1 && (p.k + 1) % p.slots != 0),
                "a pair of DFT samples needs two slots of one ring round");
    BZH_REQUIRE(p.mode != 2 || (p.nk >= 1 && p.nk <= p.slots), "DFT flush range exceeds the ring");
  }
  switch (p.dtype) {
    case BZH_F32: dft_dispatch<float>(s, p); break;
    case BZH_BF16: dft_dispatch<bf16_t>(s, p); break;
    case BZH_F16: dft_dispatch<__half>(s, p); break;
    default: throw Failure{"unsupported DFT field dtype"};
  }
  BZH_HIP(hipGetLastError());
}


void launch_dft_capture(hipStream_t s, const DftCapParams& p) {
  const DftParams& d = p.d;
  if (d.M <= 0 || d.Pmax <= 0) return;
  BZH_REQUIRE(d.Fmax <= kMaxFreq, "DFT monitors support at most 256 frequencies");
  BZH_REQUIRE(d.M <= kMaxMonBoxes && d.nk >= 1 && d.nk <= kDftMaxSlots && p.cap != nullptr,
              "captured DFT is malformed");
  const dim3 block(kDftBlock),
      grid((d.Pmax + kDftBlock - 1) / kDftBlock, std::max(1, (d.Fmax + kFt - 1) / kFt), d.M * 6);
  if (d.acc_f64) hipLaunchKernelGGL((dft_capture_kernel<double>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((dft_capture_kernel<float>), grid, block, 0, s, p);
  BZH_HIP(hipGetLastError());
}

void launch_monbox(hipStream_t s, const MonBoxParams& p) {
  BZH_REQUIRE(p.M >= 1 && p.M <= kMaxMonBoxes && p.box != nullptr, "monitor boxes are malformed");
  if (p.Pmax <= 0 || p.K <= 0) return;
  hipLaunchKernelGGL(monbox_init_kernel, dim3(1), dim3(64), 0, s, p);
  hipLaunchKernelGGL(monbox_kernel, dim3(kBoxSlices, p.M), dim3(kBoxBlock), 0, s, p);
  BZH_HIP(hipGetLastError());
}

}  // namespace bzh
