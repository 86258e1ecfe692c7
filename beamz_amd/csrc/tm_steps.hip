// Several TMxy (2D) leapfrog steps per launch: temporal blocking in registers.
//
// A 2D step of the per-phase kernels is three to five launches of 2.6-5 us
// each whose arrays mostly sit in cache, so it is bound by launches and
// latency, not bytes.  Here one launch reads bank A and writes bank B after T
// steps.
//
// Tile: a workgroup of NW waves holds 64 columns by NW * RPT rows, each lane
// RPT rows of one column in registers (Ez, Hx, Hy, the E coefficients and,
// near the faces, the CPML memories).  A step makes one cell ring at the
// region's edge invalid, so with T steps the block owns the inner
// (64 - 2T) x (NW RPT - 2T) cells.  x neighbours come from DPP wave shifts
// (full-rate vector moves, no LDS), y neighbours from the lane's own registers
// and, across waves, from two published rows: each wave carries the Hx row
// below its own (recomputed from the neighbour's Ez), so a step needs one
// barrier instead of two.
//
// Blocks and waves clear of every x or y face and slab run leaner bodies.  A
// step is short (a few hundred instructions of a wave), so scalar loads and
// branches inside it cost as much as its arithmetic: slab rows' coefficients,
// the first source slab of each timing and the first two capture boxes are
// resolved before the steps.  Source slabs of every timing are applied inside
// (execute.py:467-541 order: pre-E, H, h, E, e), and the cells that monitors
// gather are captured after every step, so that the DFT needs no launch per
// step (dft_capture_kernel folds up to 32 steps).
//
// Numerical contract: identical to phase.hip, operation for operation
// (kernels.py:731-811, 1217-1290; lattice.py:523-575; kernels.py:184-264;
// _boundary_compile.py:118-160; execute.py:374-461): each update reads the
// same inputs and rounds in the same places, so results are bitwise those of
// the per-phase kernels.

#include "common.h"

// every fused operation below is written out
#pragma clang fp contract(off)

namespace bzh {
namespace {

using tfloat = const __attribute__((address_space(4))) float;
__device__ __forceinline__ float scalar_at(const float* p, int i) { return ((tfloat*)(p))[i]; }

// The value of lane + 1 (x + 1) and of lane - 1; 0 past the wave's ends.
__device__ __forceinline__ float from_right(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_left(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
}

__device__ __forceinline__ int tm_slab(int c, int n, int L) {
  return c < L ? c : (c >= n - L ? c - (n - 2 * L) : -1);
}

// Contiguous tile ranges per XCD (workgroups are dealt round-robin to the 8
// XCDs), so that neighbouring tiles share their halo in one L2.
__device__ __forceinline__ int tm_remap(int g, int n) {
  const int c = g % 8, m = g / 8, base = n / 8, rem = n % 8;
  return c * base + min(c, rem) + m;
}

// Descriptors are read through the constant address space (scalar loads) and
// re-read where they are needed: held across the step loop, their pointers and
// the per-row conditions spill scalar registers to vector lanes.
template <typename T>
using kptr = const __attribute__((address_space(4))) T*;
template <typename P>
__device__ __forceinline__ P fresh(P p) {
  asm volatile("" : "+s"(p));
  return p;
}

__device__ __forceinline__ int fresh(int v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ uint32_t fresh(uint32_t v) { return fresh(static_cast<int>(v)); }
// The same for a per-lane value (row masks, whose tests would otherwise be
// held as lane masks).
__device__ __forceinline__ uint32_t fresh_lane(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A source slab with its origin resolved.
struct TmSlabAt {
  kptr<TmSlab> s;
  const float* coeff;
  int y0, x0;
};
__device__ __forceinline__ bool tm_slab_at(kptr<TmSlab> s, TmSlabAt& o) {
  o.s = s;
  o.coeff = s->coeff;
  o.y0 = s->y0;
  o.x0 = s->x0;
  if (s->start != nullptr) {
    kptr<int32_t> st = (kptr<int32_t>)(s->start);
    const int cz = -st[0];  // a 2D field is plane z = 0
    if (cz < 0 || cz >= s->sz) return false;
    o.coeff += static_cast<int64_t>(cz) * s->sy * s->sx;
    o.y0 = st[1];
    o.x0 = st[2];
  }
  return true;
}

// v + c w, the product rounded first (as the source launches add it).
__device__ __forceinline__ float plus_product(float v, float c, float w) {
  const float t = c * w;
  return v + t;
}

// Rows v[0 .. N) start at grid row j; adds the slab's terms of one step.
// ``timed``: a post-update slab, fused multiply-add as the folded phase
// sources; else the separately rounded product of the source launches.
template <int N>
__device__ __forceinline__ void tm_add(const TmSlabAt& a, int step, int j, int x, bool timed,
                                       float (&v)[N]) {
  kptr<TmSlab> s = a.s;
  const int T = s->T, sy = s->sy, sx = s->sx, fy = s->fy, fx = s->fx;
  const int wi = step < 0 ? 0 : (step > T - 1 ? T - 1 : step);
  const float wv = scalar_at(s->wave, wi);
  const int cx = x - a.x0;
  const bool in = cx >= 0 && cx < sx && x >= 0 && x < fx && !(s->ml && x == 0) &&
                  !(s->mr && x == fx - 1);
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const int y = j + r, cy = y - a.y0;
    if (cy < 0 || cy >= sy || y < 0 || y >= fy || (s->mb && y == 0) || (s->mt && y == fy - 1))
      continue;
    if (!in) continue;
    const float c = a.coeff[static_cast<int64_t>(cy) * sx + cx];
    v[r] = timed ? __builtin_fmaf(c, wv, v[r]) : plus_product(v[r], c, wv);
  }
}

// A slab's coefficients on the wave's rows, held in registers across the steps:
// ``bits`` marks the rows (per lane) it covers, ``wave`` lane k step k's
// waveform sample.
template <int N>
struct TmHeld {
  float c[N];
  uint32_t bits;
  float wave;
};
template <int N>
__device__ __forceinline__ void tm_hold(const TmSlabAt& a, int step, int T, int j, int x, int lane,
                                        TmHeld<N>& h) {
  kptr<TmSlab> s = a.s;
  const int n = s->T, sy = s->sy, sx = s->sx, fy = s->fy, fx = s->fx;
  const int cx = x - a.x0;
  const bool in = cx >= 0 && cx < sx && x >= 0 && x < fx && !(s->ml && x == 0) &&
                  !(s->mr && x == fx - 1);
  h.bits = 0;
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const int y = j + r, cy = y - a.y0;
    h.c[r] = 0.0f;
    if (cy < 0 || cy >= sy || y < 0 || y >= fy || (s->mb && y == 0) || (s->mt && y == fy - 1))
      continue;
    if (!in) continue;
    h.c[r] = a.coeff[static_cast<int64_t>(cy) * sx + cx];
    h.bits |= 1u << r;
  }
  const int k = step + min(lane, T - 1);
  h.wave = s->wave[k < 0 ? 0 : (k > n - 1 ? n - 1 : k)];
}
template <int N>
__device__ __forceinline__ void tm_held_add(const TmHeld<N>& h, int k, bool timed, float (&v)[N]) {
  const float wv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(h.wave), k));
  const uint32_t bits = fresh_lane(h.bits);
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const float t = timed ? __builtin_fmaf(h.c[r], wv, v[r]) : plus_product(v[r], h.c[r], wv);
    v[r] = (bits >> r) & 1u ? t : v[r];
  }
}

// The march of one wave: columns x = i0 + lane, rows j .. j + RPT - 1.
// kXE: the block reaches an x face or x slab; kYE: the wave a y face or slab.
// Waves of one block may run different versions: each step of each version
// meets the block's barrier once.
template <int NW, int RPT, bool kDec, bool kCpml, bool kOut, bool kXE, bool kYE>
__device__ __forceinline__ void tm_march(kptr<TmSim> S0, int bank, kptr<TmParams> O0,
                                         float (*rows)[NW][2][64], int T, int step, int i0, int j0,
                                         int w) {
  const int lane = threadIdx.x & 63;
  const int ny = S0->ny, nx = S0->nx, W = nx + 1, L = S0->L, m = S0->metallic;
  const bool ml = m & kLeft, mr = m & kRight;
  const float idx = S0->inv_dx;
  const float hd0 = scalar_at(S0->h_dec[0], 0), hd1 = scalar_at(S0->h_dec[1], 0);
  const float hs0 = scalar_at(S0->h_src[0], 0), hs1 = scalar_at(S0->h_src[1], 0);
  const int x = i0 + lane, j = j0 + w * RPT;
  const bool vez = !kXE || (x >= 0 && x <= nx), vhy = !kXE || (x >= 0 && x < nx);
  const bool xpec = kXE && ((ml && x == 0) || (mr && x == nx));
  // owned cells: T from every side of the region
  const bool own_x = lane >= T && lane < 64 - T && vez;
  const int r_lo = max(0, T - w * RPT), r_hi = min(RPT, NW * RPT - T - w * RPT);  // owned rows
  auto own_row = [&](int r) { return r >= r_lo && r < r_hi; };

  // ---- which slabs and capture boxes reach this wave: lane q tests entry q
  // (read before the fields, whose loads then overlap it) ----
  bool shit = false, chit = false;
  if (lane < S0->nslab) {
    const TmSlab* s = (const TmSlab*)(&S0->slab[lane]);
    int y0 = s->y0, x0 = s->x0;
    if (s->start != nullptr) {
      y0 = s->start[1];
      x0 = s->start[2];
    }
    shit = y0 < j + RPT && y0 + s->sy > j - 1 && x0 < i0 + 64 && x0 + s->sx > i0;
  }
  if constexpr (kOut) {
    if (lane < O0->nbox) {
      const TmBox* q = (const TmBox*)(&O0->box[lane]);
      chit = q->y0 < j + r_hi && q->y1 >= j + r_lo && r_lo < r_hi && q->x0 < i0 + 64 - T &&
             q->x1 >= i0 + T;
    }
  }

  // ---- loads ----
  float ez[RPT], hy[RPT], hx[RPT + 1], se[RPT], de[kDec ? RPT : 1];
  {
    const float *eza = S0->ez[bank], *hxa = S0->hx[bank], *hya = S0->hy[bank], *es = S0->e_src;
    const float* ed = S0->e_dec;
    const bool sarr = S0->src_st != 0;
    const float se_u = scalar_at(es, 0);
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int y = j + r;
      const bool vr = !kYE || (y >= 0 && y <= ny);
      ez[r] = hy[r] = 0.0f;
      se[r] = se_u;
      if constexpr (kDec) de[r] = 1.0f;
      if (vr && vez) {
        ez[r] = eza[y * W + x];
        if (sarr) se[r] = es[y * W + x];
        if constexpr (kDec) de[r] = ed[y * W + x];
      }
      if (vr && vhy) hy[r] = hya[y * nx + x];
    }
    if constexpr (!kDec) de[0] = scalar_at(ed, 0);
#pragma unroll
    for (int r = 0; r <= RPT; ++r) {
      const int y = j - 1 + r;
      hx[r] = ((!kYE || (y >= 0 && y < ny)) && vez) ? hxa[y * W + x] : 0.0f;
    }
  }
  // CPML: x terms per lane, y terms per row (uniform; bit r of ymh / yme when
  // Hx row j - 1 + r / Ez row j + r lies in a y slab)
  constexpr bool kXS = kXE && kCpml, kYS = kYE && kCpml;
  int q1 = -1, q2 = -1;
  float a1 = 0, b1 = 0, k1 = 0, a2 = 0, b2 = 0, k2 = 0;
  float p1[kXS ? RPT : 1], p2[kXS ? RPT : 1];
  float p0[kYS ? RPT + 1 : 1], p3[kYS ? RPT : 1];
  float ha[kYS ? RPT + 1 : 1], hb[kYS ? RPT + 1 : 1], hk[kYS ? RPT + 1 : 1];
  float ea[kYS ? RPT : 1], eb[kYS ? RPT : 1], ek[kYS ? RPT : 1];
  uint32_t ymh = 0, yme = 0;
  auto row_h = [&](int y) { return y >= 0 && y < ny ? tm_slab(y, ny, L) : -1; };
  auto row_e = [&](int y) { return y >= 0 && y <= ny ? tm_slab(y, ny + 1, L) : -1; };
  if constexpr (kXS) {
    q1 = vhy ? tm_slab(x, nx, L) : -1;
    q2 = vez ? tm_slab(x, nx + 1, L) : -1;
    if (q1 >= 0) {
      a1 = S0->ta[1][q1];
      b1 = S0->tb[1][q1];
      k1 = S0->tk[1][q1];
    }
    if (q2 >= 0) {
      a2 = S0->ta[2][q2];
      b2 = S0->tb[2][q2];
      k2 = S0->tk[2][q2];
    }
    const float *pa1 = S0->psi[bank][1], *pa2 = S0->psi[bank][2];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int y = j + r;
      const bool vr = !kYE || (y >= 0 && y <= ny);
      p1[r] = (vr && q1 >= 0) ? pa1[y * 2 * L + q1] : 0.0f;
      p2[r] = (vr && q2 >= 0) ? pa2[y * 2 * L + q2] : 0.0f;
    }
  }
  if constexpr (kYS) {
    const float *pa0 = S0->psi[bank][0], *pa3 = S0->psi[bank][3];
#pragma unroll
    for (int r = 0; r <= RPT; ++r) {
      const int q = row_h(j - 1 + r), qq = max(q, 0);
      if (q >= 0) ymh |= 1u << r;
      p0[r] = (q >= 0 && vez) ? pa0[q * W + x] : 0.0f;
      ha[r] = scalar_at(S0->ta[0], qq);
      hb[r] = scalar_at(S0->tb[0], qq);
      hk[r] = scalar_at(S0->tk[0], qq);
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int q = row_e(j + r), qq = max(q, 0);
      if (q >= 0) yme |= 1u << r;
      p3[r] = (q >= 0 && vez) ? pa3[q * W + x] : 0.0f;
      ea[r] = scalar_at(S0->ta[3], qq);
      eb[r] = scalar_at(S0->tb[3], qq);
      ek[r] = scalar_at(S0->tk[3], qq);
    }
  }
  const bool yface = kYE && ((0 >= j && 0 < j + RPT) || (ny >= j && ny < j + RPT));

  const uint32_t smask = static_cast<uint32_t>(__ballot(shit));
  const uint32_t cmask = kOut ? static_cast<uint32_t>(__ballot(chit)) : 0u;
  const uint32_t spre = smask & ((1u << S0->nslab_pre) - 1u);
  const uint32_t sh = smask & ((1u << S0->nslab_h) - 1u) & ~spre;
  const uint32_t spost = smask & ~(spre | sh);
  // the first slab of each timing is held in registers, further ones are
  // added from memory
  TmHeld<RPT> hpre, hpost;
  TmHeld<RPT + 1> hmid;   // an Hx slab on rows j - 1 .., an Hy slab on rows j ..
  bool mid_x = false;
  hpre.bits = hpost.bits = hmid.bits = 0;
  {
    TmSlabAt s;
    if (spre != 0 && tm_slab_at(&S0->slab[__builtin_ctz(spre)], s))
      tm_hold<RPT>(s, step, T, j, x, lane, hpre);
    if (spost != 0 && tm_slab_at(&S0->slab[__builtin_ctz(spost)], s))
      tm_hold<RPT>(s, step, T, j, x, lane, hpost);
    if (sh != 0 && tm_slab_at(&S0->slab[__builtin_ctz(sh)], s)) {
      mid_x = s.s->comp == 0;
      tm_hold<RPT + 1>(s, step, T, mid_x ? j - 1 : j, x, lane, hmid);
    }
  }
  auto e_sources = [&](uint32_t bits, int k, bool timed) {
    bits &= bits - 1;
    while (bits != 0) {
      TmSlabAt s;
      const int q = __builtin_ctz(bits);
      bits &= bits - 1;
      if (tm_slab_at(&fresh(S0)->slab[q], s)) tm_add<RPT>(s, step + k, fresh(j), x, timed, ez);
    }
  };
  // capture: the first two boxes' cells as an index and a row mask per lane
  int ci0 = 0, ci1 = 0, cw0 = 0, cw1 = 0, cc0 = 0, cc1 = 0;
  uint32_t cb0 = 0, cb1 = 0, crest = 0;
  float* cap = nullptr;
  int64_t cap_cells = 0;
  if constexpr (kOut) {
    if (cmask != 0) {
      cap_cells = O0->cap_cells;
      cap = O0->cap + O0->cap_slot * cap_cells;
      auto hold = [&](int b, int& ci, int& cw, int& cc, uint32_t& cb) {
        kptr<TmBox> q = &O0->box[b];
        const int y0 = q->y0, y1 = q->y1, x0 = q->x0, x1 = q->x1;
        cw = x1 - x0 + 1;
        cc = q->comp;
        ci = q->off + (j - y0) * cw + (x - x0);
#pragma unroll
        for (int r = 0; r < RPT; ++r)
          if (own_row(r) && own_x && j + r >= y0 && j + r <= y1 && x >= x0 && x <= x1) cb |= 1u << r;
      };
      hold(__builtin_ctz(cmask), ci0, cw0, cc0, cb0);
      crest = cmask & (cmask - 1);
      if (crest != 0) {
        hold(__builtin_ctz(crest), ci1, cw1, cc1, cb1);
        crest &= crest - 1;
      }
    }
  }
  // the adjoint's forward curl over the design box, likewise
  int ri = 0, rw = 0;
  uint32_t rb = 0;
  float* rec = nullptr;
  int64_t rec_cells = 0;
  if constexpr (kOut) {
    if (O0->record != nullptr) {
      const int y0 = O0->design[0], y1 = O0->design[1], x0 = O0->design[2], x1 = O0->design[3];
      rw = x1 - x0;
      rec_cells = static_cast<int64_t>(y1 - y0) * rw;
      ri = (j - y0) * rw + (x - x0);
#pragma unroll
      for (int r = 0; r < RPT; ++r)
        if (own_row(r) && own_x && j + r >= y0 && j + r < y1 && x >= x0 && x < x1) rb |= 1u << r;
      if (__builtin_amdgcn_readfirstlane(__any(rb != 0)) != 0)
        rec = O0->record + O0->record_slot * rec_cells;
    }
  }
  auto put = [&](float* at, int ci, int cw, int cc, uint32_t mask) {
    const uint32_t cb = fresh_lane(mask);
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      // (by value: a conditional of two lvalues indexes them in scratch)
      const float ve = ez[r], vx = hx[r + 1], vy = hy[r];
      const float v = cc == 2 ? ve : (cc == 0 ? vx : vy);
      if ((cb >> r) & 1u) at[ci + r * cw] = v;
    }
  };

  for (int k = 0; k < T; ++k) {
    const int b = k & 1;
    if (spre != 0) {
      tm_held_add<RPT>(hpre, k, false, ez);
      e_sources(spre, k, false);
    }
    rows[b][w][0][lane] = ez[0];
    rows[b][w][1][lane] = ez[RPT - 1];
    __syncthreads();
    const float ez_up = w + 1 < NW ? rows[b][w + 1][0][lane] : 0.0f;
    const float ez_dn = w > 0 ? rows[b][w - 1][1][lane] : 0.0f;
    // Hy
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      float d = (from_right(ez[r]) - ez[r]) * idx;
      if constexpr (kXS) {
        const float t = __builtin_fmaf(b1, p1[r], a1 * d);
        p1[r] = q1 >= 0 ? t : 0.0f;
        d = q1 >= 0 ? __builtin_fmaf(d, k1, t) : d;
      }
      hy[r] = __builtin_fmaf(hd1, hy[r], hs1 * d);
    }
    // Hx
    const uint32_t yh = kYS ? fresh(ymh) : 0u, ye = kYS ? fresh(yme) : 0u;
#pragma unroll
    for (int r = 0; r <= RPT; ++r) {
      const float hi = r < RPT ? +ez[r < RPT ? r : 0] : ez_up;
      const float lo = r > 0 ? +ez[r > 0 ? r - 1 : 0] : ez_dn;
      float d = (hi - lo) * idx;
      if constexpr (kYS) {
        if ((yh >> r) & 1u) {
          p0[r] = __builtin_fmaf(hb[r], p0[r], ha[r] * d);
          d = __builtin_fmaf(d, hk[r], p0[r]);
        }
      }
      hx[r] = __builtin_fmaf(hd0, hx[r], -(hs0 * d));
      if (xpec) hx[r] = 0.0f;
    }
    if constexpr (kYE) {
      if (yface) {
        const int jj = fresh(j), mm = fresh(m);
#pragma unroll
        for (int r = 0; r < RPT; ++r)
          if (((mm & kBottom) && jj + r == 0) || ((mm & kTop) && jj + r == ny)) hy[r] = 0.0f;
      }
    }
    if (sh != 0) {
      if (mid_x) {
        tm_held_add<RPT + 1>(hmid, k, true, hx);
      } else {
        const float wv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hmid.wave), k));
        const uint32_t hb = fresh_lane(hmid.bits);
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const float t = __builtin_fmaf(hmid.c[r], wv, hy[r]);
          hy[r] = (hb >> r) & 1u ? t : hy[r];
        }
      }
      uint32_t bits = sh & (sh - 1);
      while (bits != 0) {
        TmSlabAt s;
        const int q = __builtin_ctz(bits);
        bits &= bits - 1;
        if (!tm_slab_at(&fresh(S0)->slab[q], s)) continue;
        if (s.s->comp == 0) tm_add<RPT + 1>(s, step + k, fresh(j) - 1, x, true, hx);
        else tm_add<RPT>(s, step + k, fresh(j), x, true, hy);
      }
    }
    // E
    float v[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) v[r] = hx[r + 1] - hx[r];
    if constexpr (kYE) {
      // ghost rule: zero past a metallic face, the edge sample past others
      if (yface) {
        const int jj = fresh(j), mm = fresh(m);
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          if (jj + r == 0) v[r] = hx[r + 1] - ((mm & kBottom) ? 0.0f : hx[r + 1]);
          if (jj + r == ny) v[r] = ((mm & kTop) ? 0.0f : hx[r]) - hx[r];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      float hyl = from_left(hy[r]), hyc = hy[r];
      if constexpr (kXE) {
        hyl = x == 0 ? (ml ? 0.0f : hyc) : hyl;
        hyc = x == nx ? (mr ? 0.0f : hyl) : hyc;
      }
      const float u = hyc - hyl;
      float d0 = u * idx, d1 = v[r] * idx;
      if constexpr (kOut) {
        // (no slab and no face in the design box)
        if (rec != nullptr && ((fresh_lane(rb) >> r) & 1u)) rec[ri + r * rw] = __builtin_fmaf(idx, u, -d1);
      }
      if constexpr (kXS) {
        const float t = __builtin_fmaf(b2, p2[r], a2 * d0);
        p2[r] = q2 >= 0 ? t : 0.0f;
        d0 = q2 >= 0 ? __builtin_fmaf(d0, k2, t) : d0;
      }
      if constexpr (kYS) {
        if ((ye >> r) & 1u) {
          p3[r] = __builtin_fmaf(eb[r], p3[r], ea[r] * d1);
          d1 = __builtin_fmaf(d1, ek[r], p3[r]);
        }
      }
      // (without CPML the phase kernel's curl is one fused operation)
      const float curl = kCpml ? d0 - d1 : __builtin_fmaf(u, idx, -d1);
      ez[r] = __builtin_fmaf(de[kDec ? r : 0], ez[r], se[r] * curl);
      if (xpec) ez[r] = 0.0f;
    }
    if constexpr (kYE) {
      if (yface) {
        const int jj = fresh(j), mm = fresh(m);
#pragma unroll
        for (int r = 0; r < RPT; ++r)
          if (((mm & kBottom) && jj + r == 0) || ((mm & kTop) && jj + r == ny)) ez[r] = 0.0f;
      }
    }
    if (spost != 0) {
      tm_held_add<RPT>(hpost, k, true, ez);
      e_sources(spost, k, true);
    }
    if constexpr (kOut) {
      if (rec != nullptr) rec += rec_cells;
      if (cmask != 0) {
        put(cap, ci0, cw0, cc0, cb0);
        if (cw1 != 0) put(cap, ci1, cw1, cc1, cb1);
        uint32_t bits = crest;
        while (bits != 0) {
          kptr<TmBox> q = &fresh(O0)->box[__builtin_ctz(bits)];
          bits &= bits - 1;
          const int j = fresh(j0 + w * RPT), r_lo = max(0, fresh(T) - w * RPT);
          const int r_hi = min(RPT, NW * RPT - fresh(T) - w * RPT);
          const int y0 = q->y0, y1 = q->y1, x0 = q->x0, x1 = q->x1;
          uint32_t cb = 0;
#pragma unroll
          for (int r = 0; r < RPT; ++r)
            if (r >= r_lo && r < r_hi && own_x && j + r >= y0 && j + r <= y1 && x >= x0 && x <= x1)
              cb |= 1u << r;
          put(cap, q->off + (j - y0) * (x1 - x0 + 1) + (x - x0), x1 - x0 + 1, q->comp, cb);
        }
        cap += cap_cells;
      }
    }
  }

  // ---- stores ----
  kptr<TmSim> S = fresh(S0);
  const int je = fresh(j), nb = bank ^ 1;
  float *ezb = S->ez[nb], *hxb = S->hx[nb], *hyb = S->hy[nb];
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int y = je + r;
    if (!own_row(r) || !own_x || (kYE && (y < 0 || y > ny))) continue;
    ezb[y * W + x] = ez[r];
    if (vhy) hyb[y * nx + x] = hy[r];
    if (!kYE || y < ny) hxb[y * W + x] = hx[r + 1];
    if constexpr (kXS) {
      if (q1 >= 0) S->psi[nb][1][y * 2 * L + q1] = p1[r];
      if (q2 >= 0) S->psi[nb][2][y * 2 * L + q2] = p2[r];
    }
    if constexpr (kYS) {
      if ((ymh >> (r + 1)) & 1u) S->psi[nb][0][row_h(y) * W + x] = p0[r + 1];
      if ((yme >> r) & 1u) S->psi[nb][3][row_e(y) * W + x] = p3[r];
    }
  }
}

// One wave of a block at (i0, j0): the version its position needs.
template <int NW, int RPT, bool kDec, bool kCpml, bool kOut>
__device__ __forceinline__ void tm_wave(kptr<TmSim> S, int bank, kptr<TmParams> O,
                                        float (*rows)[NW][2][64], int T, int step, int i0, int j0) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = max(S->L, 1), j = j0 + w * RPT;
  const bool xin = i0 >= M && i0 + 63 <= S->nx - M - 1;
  const bool yin = j - 1 >= M && j + RPT <= S->ny - M - 1;
  if (xin && yin) tm_march<NW, RPT, kDec, kCpml, kOut, false, false>(S, bank, O, rows, T, step, i0, j0, w);
  else if (xin) tm_march<NW, RPT, kDec, kCpml, kOut, false, true>(S, bank, O, rows, T, step, i0, j0, w);
  else if (yin) tm_march<NW, RPT, kDec, kCpml, kOut, true, false>(S, bank, O, rows, T, step, i0, j0, w);
  else tm_march<NW, RPT, kDec, kCpml, kOut, true, true>(S, bank, O, rows, T, step, i0, j0, w);
}

template <int NW, int RPT, bool kDec, bool kCpml>
__global__ void __launch_bounds__(64 * NW) tm_steps(TmParams) {
  __shared__ float rows[2][NW][2][64];
  kptr<TmParams> p = (kptr<TmParams>)(__builtin_amdgcn_kernarg_segment_ptr());
  kptr<TmSim> S = &p->sim;
  const int t = tm_remap(blockIdx.x, gridDim.x), ntx = p->ntx;
  const int ty = t / ntx, tx = t - ty * ntx;
  const int T = p->T;
  const int i0 = tx * (64 - 2 * T) - T, j0 = ty * (NW * RPT - 2 * T) - T;
  kptr<int32_t> st = (kptr<int32_t>)(p->step0);
  const int step = (st != nullptr ? *st : 0) + p->k;
  tm_wave<NW, RPT, kDec, kCpml, true>(S, p->bank, p, rows, T, step, i0, j0);
}

// Batched simulations: one block per tile of any member, the members'
// descriptors in device memory.  64 simulations of 26 M cells: 424 GCUPS; one
// wave per 62-column item with one step per launch reached 121.  Members
// without CPML run the CPML form too, whose curl rounds both terms.
template <int NW, int RPT>
__global__ void __launch_bounds__(64 * NW) tm_batch(TmBatchParams p) {
  __shared__ float rows[2][NW][2][64];
  kptr<int32_t> td = (kptr<int32_t>)(p.tiles + tm_remap(blockIdx.x, gridDim.x));
  const int sim = td[0], ty = td[1], tx = td[2];
  const int T = p.T;
  const int i0 = tx * (64 - 2 * T) - T, j0 = ty * (NW * RPT - 2 * T) - T;
  const int step = *(kptr<int32_t>)(p.step0) + p.k;
  tm_wave<NW, RPT, false, true, false>((kptr<TmSim>)(p.sims + sim), p.bank, (kptr<TmParams>)(nullptr),
                                       rows, T, step, i0, j0);
}

template <int NW, int RPT>
void launch_tm_rows(hipStream_t s, const TmParams& p) {
  static_assert(NW * RPT == kTmRows, "tile height");
  const int own = kTmRows - 2 * p.T;
  const int nty = (p.sim.ny + 1 + own - 1) / own;
  const dim3 grid(static_cast<unsigned>(p.ntx) * nty), block(64 * NW);
  if (p.sim.dec_st) {
    if (p.sim.L > 0) hipLaunchKernelGGL((tm_steps<NW, RPT, true, true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((tm_steps<NW, RPT, true, false>), grid, block, 0, s, p);
  } else {
    if (p.sim.L > 0) hipLaunchKernelGGL((tm_steps<NW, RPT, false, true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((tm_steps<NW, RPT, false, false>), grid, block, 0, s, p);
  }
}

}  // namespace

void launch_tm(hipStream_t s, const TmParams& p) {
  BZH_REQUIRE(p.T >= 1 && p.T <= kTmMaxSteps && p.sim.nslab <= kMaxTmSlabs && p.nbox <= kMaxTmBoxes &&
                  (p.rpt == 2 || p.rpt == 4),
              "2D multi-step launch is malformed");
  BZH_REQUIRE(p.ntx * (64 - 2 * p.T) >= p.sim.nx + 1, "2D multi-step tiles do not cover the grid");
  if (p.rpt == 2) launch_tm_rows<16, 2>(s, p);
  else launch_tm_rows<8, 4>(s, p);
  BZH_HIP(hipGetLastError());
}

void launch_tm_batch(hipStream_t s, const TmBatchParams& p) {
  BZH_REQUIRE(p.T >= 1 && p.T <= kTmMaxSteps && (p.rpt == 2 || p.rpt == 4) && p.ntiles >= 1 &&
                  p.sims != nullptr && p.tiles != nullptr && p.step0 != nullptr,
              "batched launch is malformed");
  const dim3 grid(p.ntiles);
  if (p.rpt == 2) hipLaunchKernelGGL((tm_batch<16, 2>), grid, dim3(64 * 16), 0, s, p);
  else hipLaunchKernelGGL((tm_batch<8, 4>), grid, dim3(64 * 8), 0, s, p);
  BZH_HIP(hipGetLastError());
}

}  // namespace bzh
