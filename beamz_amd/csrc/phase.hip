// Per-phase Yee updates for gfx950: one launch advances the three H (or E)
// components of a 3D grid, or the TMxy pair / Ez of a 2D plane, including the
// packed CPML recurrences and the PEC face rule.
//
// Numerical contract (reference files):
//   3D H: beamz/simulation/kernels.py:458-503, 267-290; lattice.py:467-473
//   3D E: kernels.py:554-626, 326-388; ghost rule lattice.py:523-575
//   TMxy: kernels.py:731-811, 1217-1290
//   CPML: kernels.py:184-264 (packed slabs), PEC: _boundary_compile.py:118-160
//
// Mapping: wave64 along x (fastest storage axis), block 64x4, one thread per
// (k, j, i) of the union of the three component supports; each thread updates
// every component whose support contains it.  All field indices are 32-bit:
// the host rejects arrays of 2^31 elements or more.

#include "common.h"

namespace bzh {
namespace {

constexpr int kBX = 64;
constexpr int kBY = 4;

template <typename T>
__device__ __forceinline__ float ld(const void* p, int i) {
  return load_f(static_cast<const T*>(p), i);
}

__device__ __forceinline__ float metric_at(const PhaseParams& p, int axis, int c) {
  const float* m = p.metric[axis];
  return m == nullptr ? p.inv_dx : m[c * p.met_st[axis]];
}

// Packed CPML correction of one derivative (kernels.py:184-264).  ``c`` is the
// coordinate along the term's axis, ``lin_of`` maps a packed coordinate to the
// psi linear index.  Returns d/kappa + psi inside the slab and d outside.
template <typename F>
__device__ __forceinline__ float cpml_correct(const PhaseParams& p, int t, float d,
                                              int c, F lin_of) {
  const DevTerm& tm = p.term[t];
  int low, high;
  if (p.uniform_l > 0) {
    low = high = p.uniform_l;
  } else {
    low = p.meta[t * 5 + 2];
    high = p.meta[t * 5 + 3];
  }
  int packed = -1;
  if (c < low) {
    packed = c;
  } else if (c >= tm.n - high) {
    packed = low + c - (tm.n - high);
  }
  // tm.low/tm.high carry the psi extent split validated on the host; a packed
  // index outside [0, low + high) is never dereferenced.
  if (packed < 0 || packed >= tm.low + tm.high) return d;
  const int q = lin_of(packed);
  float psi;
  if (tm.psi_bf16) {
    psi = load_f(static_cast<const bf16_t*>(tm.psi), q);
  } else {
    psi = static_cast<const float*>(tm.psi)[q];
  }
  psi = tm.b[packed] * psi + tm.a[packed] * d;
  if (tm.psi_bf16) {
    store_f(static_cast<bf16_t*>(tm.psi), q, psi);
  } else {
    static_cast<float*>(tm.psi)[q] = psi;
  }
  return d * tm.ik[packed] + psi;
}

__device__ __forceinline__ float coef(const float* arr, int st, float s, int i) {
  return arr == nullptr ? s : arr[i * st];
}
// E source coefficient c of cell o: scf is a table indexed by the cell's
// 8-bit ID (four IDs per int32 word, lowest byte first; compile.py:146-168)
// when scf_ids[c] is set, else as coef
__device__ __forceinline__ float scf_at(const PhaseParams& p, int c, int o) {
  if (p.scf_ids[c] != nullptr) {
    const uint32_t word = static_cast<uint32_t>(p.scf_ids[c][o >> 2]);
    return p.scf[c][(word >> ((o & 3) * 8)) & 0xFFu];
  }
  return coef(p.scf[c], p.scf_st[c], p.scf_s[c], o);
}

// What folded source group ``s`` adds to its target's cell (k, j, i), the
// slabs in declaration order after v (as successive source launches add them,
// to rounding); float32 fields only.
__device__ __forceinline__ float group_add(const PhaseParams& p, const PhaseSrc& s, int k, int j,
                                           int i, float v) {
  if ((s.mlo[0] && k == 0) || (s.mhi[0] && k == s.fz - 1) || (s.mlo[1] && j == 0) ||
      (s.mhi[1] && j == s.fy - 1) || (s.mlo[2] && i == 0) || (s.mhi[2] && i == s.fx - 1))
    return v;
  int widx = *p.step0 + p.k;
  widx = widx < 0 ? 0 : (widx > s.T - 1 ? s.T - 1 : widx);
  for (int q = 0; q < s.n; ++q) {
    const int cz = k - s.starts[q * 3 + 0], cy = j - s.starts[q * 3 + 1];
    const int cx = i - s.starts[q * 3 + 2];
    if (cz < 0 || cz >= s.sz || cy < 0 || cy >= s.sy || cx < 0 || cx >= s.sx) continue;
    const int64_t c = ((static_cast<int64_t>(q) * s.sz + cz) * s.sy + cy) * s.sx + cx;
    v = v + s.coeff[c] * s.wave[static_cast<int64_t>(q) * s.T + widx];
  }
  return v;
}
// the groups of a 3D phase's three targets.  Few waves meet a source, so the
// parameters are re-read from the argument block through a pointer the
// compiler cannot see into: read as ordinary arguments they were all loaded
// at the kernel's start and spilled (4591 against 3930 us per 64 lossy steps
// at 72x120x200).
__device__ __forceinline__ void sources_3d(int k, int j, int i, float& x, float& y, float& z) {
  using KP = __attribute__((address_space(4))) const PhaseParams;
  KP* a = (KP*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  for (int c = 0; c < 3; ++c) {
    const auto& s = a->psrc[c];
    if (s.n == 0) continue;
    float add = 0.0f;
    for (int q = 0; q < s.n; ++q) {
      const int cz = k - s.starts[q * 3 + 0], cy = j - s.starts[q * 3 + 1];
      if (cz < 0 || cz >= s.sz || cy < 0 || cy >= s.sy) continue;
      if ((s.mlo[0] && k == 0) || (s.mhi[0] && k == s.fz - 1) || (s.mlo[1] && j == 0) ||
          (s.mhi[1] && j == s.fy - 1))
        continue;
      const int cx = i - s.starts[q * 3 + 2];
      const bool open = !((s.mlo[2] && i == 0) || (s.mhi[2] && i == s.fx - 1));
      int widx = *a->step0 + a->k;
      widx = widx < 0 ? 0 : (widx > s.T - 1 ? s.T - 1 : widx);
      const float wv = s.wave[static_cast<int64_t>(q) * s.T + widx];
      if (open && cx >= 0 && cx < s.sx)
        add += s.coeff[((static_cast<int64_t>(q) * s.sz + cz) * s.sy + cy) * s.sx + cx] * wv;
    }
    x += c == 0 ? add : 0.0f;
    y += c == 1 ? add : 0.0f;
    z += c == 2 ? add : 0.0f;
  }
}

// ---------------------------------------------------------------------------
// 3D phases
//
// A wave owns 64 cells of one row, one cell per thread: k and j are uniform.
// What bounds these kernels is latency and instruction issue (a wave lives
// 2.9 us; the scalar unit of a CU serves all its waves), then the L2 misses.
// So each wave takes one of three bodies: plain (no face, slab or ghost
// anywhere in it), x-edge (only x faces and slabs) and general, the first two
// free of clamps and tests (72x120x200 with per-cell decay, per step: 73 us
// with the general body alone, 68 with the three); every array is reached at
// its base plus one per-lane byte offset, and all loads are issued before the
// first store, since the compiler cannot move them over stores that may alias
// (a load-update-store sequence per component took 79 us for the two phases,
// this 50).  Marching each column over 2 to 12 planes with the next plane's
// loads in flight was slower at every depth: 95 us and more per step.
// ---------------------------------------------------------------------------

// element at byte offset ``off`` of an array; Off is 32-bit when every array
// spans less than 4 GiB
template <typename T, typename Off>
__device__ __forceinline__ float ldb(const void* p, Off off) {
  return load_f(reinterpret_cast<const T*>(static_cast<const char*>(p) + off), 0);
}
template <typename T, typename Off>
__device__ __forceinline__ void stb(void* p, Off off, float v) {
  store_f(reinterpret_cast<T*>(static_cast<char*>(p) + off), 0, v);
}

// One CPML term at this cell: packed coordinate (-1 outside the slabs), psi
// index, recurrence coefficients and memory (kernels.py:184-264).
struct Slab {
  int pk, q;
  float a, b, ik, psi;
};
template <bool kOn, typename F>
__device__ __forceinline__ Slab slab_load(const PhaseParams& p, int t, bool ok, int c, F lin_of) {
  Slab s{-1, 0, 0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (kOn) {
    const DevTerm& tm = p.term[t];
    const int low = p.uniform_l > 0 ? p.uniform_l : p.meta[t * 5 + 2];
    const int high = p.uniform_l > 0 ? p.uniform_l : p.meta[t * 5 + 3];
    const int pk = c < low ? c : (c >= tm.n - high ? low + c - (tm.n - high) : -1);
    // tm.low + tm.high is the psi extent validated on the host; a packed
    // index outside it is never dereferenced
    if (ok && pk >= 0 && pk < tm.low + tm.high) {
      s.pk = pk;
      s.q = lin_of(tm.low + tm.high, pk);
      s.a = tm.a[pk];
      s.b = tm.b[pk];
      s.ik = tm.ik[pk];
      s.psi = tm.psi_bf16 ? load_f(static_cast<const bf16_t*>(tm.psi), s.q)
                          : static_cast<const float*>(tm.psi)[s.q];
    }
  }
  return s;
}
// d / kappa + psi' inside the slab (storing psi' = b psi + a d), d outside
template <bool kOn>
__device__ __forceinline__ float slab_apply(const PhaseParams& p, int t, const Slab& s, float d) {
  if constexpr (kOn) {
    if (s.pk >= 0) {
      const DevTerm& tm = p.term[t];
      const float psi = s.b * s.psi + s.a * d;
      if (tm.psi_bf16) store_f(static_cast<bf16_t*>(tm.psi), s.q, psi);
      else static_cast<float*>(tm.psi)[s.q] = psi;
      return d * s.ik + psi;
    }
  }
  return d;
}

// Coefficients of element e: kCoefScalar, every one a device scalar;
// kCoefArray, arrays or device scalars (read at element 0: no branch);
// kCoefAny, also host scalars and tables by 8-bit ID.
enum { kCoefScalar = 0, kCoefArray, kCoefAny };
template <int kCoef, typename Off>
__device__ __forceinline__ float dec_at(const PhaseParams& p, int c, Off e) {
  if constexpr (kCoef == kCoefScalar) return p.dec[c][0];
  else if constexpr (kCoef == kCoefArray) return ldb<float>(p.dec[c], p.dec_st[c] != 0 ? e * 4 : Off{0});
  else return coef(p.dec[c], p.dec_st[c], p.dec_s[c], static_cast<int>(e));
}
template <int kCoef, typename Off>
__device__ __forceinline__ float src_at(const PhaseParams& p, int c, Off e) {
  if constexpr (kCoef == kCoefScalar) return p.scf[c][0] * p.ratio;
  else if constexpr (kCoef == kCoefArray) return ldb<float>(p.scf[c], p.scf_st[c] != 0 ? e * 4 : Off{0}) * p.ratio;
  else return scf_at(p, c, static_cast<int>(e)) * p.ratio;
}

// What a wave's cells reach: with M = max(L, 1), plain waves lie in [M, n - M)
// of every axis, where no CPML term, face, ghost or validity cut applies.
// (Slabs that differ by face are read from device metadata: general.)
enum { kWavePlain = 0, kWaveXEdge, kWaveGeneral };
__device__ __forceinline__ int wave_kind(const PhaseParams& p, int i0, int j, int k) {
  if (p.nterms > 0 && p.uniform_l <= 0) return kWaveGeneral;
  const int M = p.nterms > 0 ? max(p.uniform_l, 1) : 1;
  if (k < M || k >= p.nz - M || j < M || j >= p.ny - M) return kWaveGeneral;
  return i0 >= M && i0 + kBX <= p.nx - M ? kWavePlain : kWaveXEdge;
}

template <typename T, typename Off, int kKind, bool kCpml, int kCoef>
__device__ __forceinline__ void h_cell(const PhaseParams& p, int i, int j, int k) {
  constexpr bool kX = kKind != kWavePlain, kYZ = kKind == kWaveGeneral;
  const int nz = p.nz, ny = p.ny, nx = p.nx;
  const int iX = kX ? min(i, nx - 1) : i, iY = kX ? min(i, nx) : i, i1 = kX ? min(i + 1, nx) : i + 1;
  const int jY = kYZ ? min(j, ny - 1) : j, j1 = kYZ ? min(j + 1, ny) : j + 1;
  const int kz = kYZ ? min(k, nz - 1) : k, k1 = kYZ ? min(k + 1, nz) : k + 1;
  // elements: A of Ex, Hy (.., ny+1, nx); B of Ey, Hx (.., ny, nx+1); C of Ez
  // (.., ny+1, nx+1); D of Hz (.., ny, nx)
  auto A = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * (ny + 1) + jj) * nx + ii); };
  auto B = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * ny + jj) * (nx + 1) + ii); };
  auto C = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * (ny + 1) + jj) * (nx + 1) + ii); };
  auto D = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * ny + jj) * nx + ii); };
  constexpr Off sz = sizeof(T);
  const float ex = ldb<T>(p.src[0], A(k, j, iX) * sz), exz = ldb<T>(p.src[0], A(k1, j, iX) * sz);
  const float exy = ldb<T>(p.src[0], A(k, j1, iX) * sz);
  const float ey = ldb<T>(p.src[1], B(k, jY, iY) * sz), eyz = ldb<T>(p.src[1], B(k1, jY, iY) * sz);
  const float eyx = ldb<T>(p.src[1], B(k, jY, i1) * sz);
  const float ez = ldb<T>(p.src[2], C(kz, j, iY) * sz), ezy = ldb<T>(p.src[2], C(kz, j1, iY) * sz);
  const float ezx = ldb<T>(p.src[2], C(kz, j, i1) * sz);
  const Off ox = B(kz, jY, iY), oy = A(kz, j, iX), oz = D(k, jY, iX);
  const float hx0 = ldb<T>(p.tin[0], ox * sz), hy0 = ldb<T>(p.tin[1], oy * sz), hz0 = ldb<T>(p.tin[2], oz * sz);
  const float cx = dec_at<kCoef>(p, 0, ox), cy = dec_at<kCoef>(p, 1, oy), cz = dec_at<kCoef>(p, 2, oz);
  const float sx = src_at<kCoef>(p, 0, ox), sy = src_at<kCoef>(p, 1, oy), sz_ = src_at<kCoef>(p, 2, oz);
  const float mz = metric_at(p, 0, kz), my = metric_at(p, 1, jY), mx = metric_at(p, 2, iX);
  const bool vk = !kYZ || k < nz, vj = !kYZ || j < ny, vX = !kX || i < nx, vY = !kX || i <= nx;
  constexpr bool kTx = kCpml && kX, kTyz = kCpml && kYZ;
  const Slab s0 = slab_load<kTyz>(p, 0, vk && vj && vY, jY, [&](int n, int q) { return (kz * n + q) * (nx + 1) + iY; });
  const Slab s1 = slab_load<kTyz>(p, 1, vk && vj && vY, kz, [&](int, int q) { return static_cast<int>(B(q, jY, iY)); });
  const Slab s2 = slab_load<kTyz>(p, 2, vk && vX, kz, [&](int, int q) { return static_cast<int>(A(q, j, iX)); });
  const Slab s3 = slab_load<kTx>(p, 3, vk && vX, iX, [&](int n, int q) { return (kz * (ny + 1) + j) * n + q; });
  const Slab s4 = slab_load<kTx>(p, 4, vj && vX, iX, [&](int n, int q) { return (k * ny + jY) * n + q; });
  const Slab s5 = slab_load<kTyz>(p, 5, vj && vX, jY, [&](int n, int q) { return (k * n + q) * nx + iX; });

  const float d0 = slab_apply<kTyz>(p, 0, s0, (ezy - ez) * my);  // dEz/dy
  const float d1 = slab_apply<kTyz>(p, 1, s1, (eyz - ey) * mz);  // dEy/dz
  const float d2 = slab_apply<kTyz>(p, 2, s2, (exz - ex) * mz);  // dEx/dz
  const float d3 = slab_apply<kTx>(p, 3, s3, (ezx - ez) * mx);   // dEz/dx
  const float d4 = slab_apply<kTx>(p, 4, s4, (eyx - ey) * mx);   // dEy/dx
  const float d5 = slab_apply<kTyz>(p, 5, s5, (exy - ex) * my);  // dEx/dy
  const int m = p.metallic;
  float hx = cx * hx0 - sx * (d0 - d1);
  float hy = cy * hy0 - sy * (d2 - d3);
  float hz = cz * hz0 - sz_ * (d4 - d5);
  if (kX && (((m & kLeft) && i == 0) || ((m & kRight) && i == nx))) hx = 0.0f;
  if (kYZ && (((m & kBottom) && j == 0) || ((m & kTop) && j == ny))) hy = 0.0f;
  if (kYZ && (((m & kFront) && k == 0) || ((m & kBack) && k == nz))) hz = 0.0f;
  if (p.npsrc > 0) sources_3d(k, j, i, hx, hy, hz);
  if (vk && vj && vY) stb<T>(p.tout[0], ox * sz, hx);
  if (vk && vX) stb<T>(p.tout[1], oy * sz, hy);
  if (vj && vX) stb<T>(p.tout[2], oz * sz, hz);
}

// Backward difference of ghost-padded H along one axis (lattice.py:523-575)
// at node c of 0..N: ``cur`` is the value at min(c, N - 1), ``prev`` at
// max(c - 1, 0).  kGhost false: 0 < c < N.
template <bool kGhost>
__device__ __forceinline__ float ghost_diff(float cur, float prev, int c, int N, bool metal_lo,
                                            bool metal_hi) {
  if constexpr (!kGhost) return cur - prev;
  const float up = c < N ? cur : (metal_hi ? 0.0f : prev);
  const float lo = c > 0 ? prev : (metal_lo ? 0.0f : cur);
  return up - lo;
}

template <typename T, typename Off, int kKind, bool kCpml, int kCoef>
__device__ __forceinline__ void e_cell(const PhaseParams& p, int i, int j, int k) {
  constexpr bool kX = kKind != kWavePlain, kYZ = kKind == kWaveGeneral;
  const int nz = p.nz, ny = p.ny, nx = p.nx;
  const int m = p.metallic;
  const int iX = kX ? min(i, nx - 1) : i, iY = kX ? min(i, nx) : i;
  const int i1 = kX ? min(max(i - 1, 0), nx - 1) : i - 1;
  const int jY = kYZ ? min(j, ny - 1) : j, j1 = kYZ ? max(j - 1, 0) : j - 1;
  const int kz = kYZ ? min(k, nz - 1) : k, k1 = kYZ ? max(k - 1, 0) : k - 1;
  auto A = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * (ny + 1) + jj) * nx + ii); };
  auto B = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * ny + jj) * (nx + 1) + ii); };
  auto C = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * (ny + 1) + jj) * (nx + 1) + ii); };
  auto D = [&](int kk, int jj, int ii) { return static_cast<Off>((kk * ny + jj) * nx + ii); };
  constexpr Off sz = sizeof(T);
  const float hx = ldb<T>(p.src[0], B(kz, jY, iY) * sz), hxz = ldb<T>(p.src[0], B(k1, jY, iY) * sz);
  const float hxy = ldb<T>(p.src[0], B(kz, j1, iY) * sz);
  const float hy = ldb<T>(p.src[1], A(kz, j, iX) * sz), hyz = ldb<T>(p.src[1], A(k1, j, iX) * sz);
  const float hyx = ldb<T>(p.src[1], A(kz, j, i1) * sz);
  const float hz = ldb<T>(p.src[2], D(k, jY, iX) * sz), hzy = ldb<T>(p.src[2], D(k, j1, iX) * sz);
  const float hzx = ldb<T>(p.src[2], D(k, jY, i1) * sz);
  const Off ox = A(k, j, iX), oy = B(k, jY, iY), oz = C(kz, j, iY);
  const float ex0 = ldb<T>(p.tin[0], ox * sz), ey0 = ldb<T>(p.tin[1], oy * sz), ez0 = ldb<T>(p.tin[2], oz * sz);
  const float cx = dec_at<kCoef>(p, 0, ox), cy = dec_at<kCoef>(p, 1, oy), cz = dec_at<kCoef>(p, 2, oz);
  const float sx = src_at<kCoef>(p, 0, ox), sy = src_at<kCoef>(p, 1, oy), sz_ = src_at<kCoef>(p, 2, oz);
  const float mz = metric_at(p, 0, k), my = metric_at(p, 1, j), mx = metric_at(p, 2, iY);
  const bool vk = !kYZ || k < nz, vj = !kYZ || j < ny, vX = !kX || i < nx, vY = !kX || i <= nx;
  constexpr bool kTx = kCpml && kX, kTyz = kCpml && kYZ;
  const Slab s0 = slab_load<kTyz>(p, 0, vX, j, [&](int n, int q) { return (k * n + q) * nx + iX; });
  const Slab s1 = slab_load<kTyz>(p, 1, vX, k, [&](int, int q) { return static_cast<int>(A(q, j, iX)); });
  const Slab s2 = slab_load<kTyz>(p, 2, vj && vY, k, [&](int, int q) { return static_cast<int>(B(q, jY, iY)); });
  const Slab s3 = slab_load<kTx>(p, 3, vj && vY, iY, [&](int n, int q) { return (k * ny + jY) * n + q; });
  const Slab s4 = slab_load<kTx>(p, 4, vk && vY, iY, [&](int n, int q) { return (kz * (ny + 1) + j) * n + q; });
  const Slab s5 = slab_load<kTyz>(p, 5, vk && vY, j, [&](int n, int q) { return (kz * n + q) * (nx + 1) + iY; });

  const float d0 = slab_apply<kTyz>(p, 0, s0, ghost_diff<kYZ>(hz, hzy, j, ny, m & kBottom, m & kTop) * my);  // dHz/dy
  const float d1 = slab_apply<kTyz>(p, 1, s1, ghost_diff<kYZ>(hy, hyz, k, nz, m & kFront, m & kBack) * mz);  // dHy/dz
  const float d2 = slab_apply<kTyz>(p, 2, s2, ghost_diff<kYZ>(hx, hxz, k, nz, m & kFront, m & kBack) * mz);  // dHx/dz
  const float d3 = slab_apply<kTx>(p, 3, s3, ghost_diff<kX>(hz, hzx, iY, nx, m & kLeft, m & kRight) * mx);   // dHz/dx
  const float d4 = slab_apply<kTx>(p, 4, s4, ghost_diff<kX>(hy, hyx, iY, nx, m & kLeft, m & kRight) * mx);   // dHy/dx
  const float d5 = slab_apply<kTyz>(p, 5, s5, ghost_diff<kYZ>(hx, hxy, j, ny, m & kBottom, m & kTop) * my);  // dHx/dy
  float ex = cx * ex0 + sx * (d0 - d1);
  float ey = cy * ey0 + sy * (d2 - d3);
  float ez = cz * ez0 + sz_ * (d4 - d5);
  const bool zf = kYZ && (((m & kFront) && k == 0) || ((m & kBack) && k == nz));
  const bool yf = kYZ && (((m & kBottom) && j == 0) || ((m & kTop) && j == ny));
  const bool xf = kX && (((m & kLeft) && i == 0) || ((m & kRight) && i == nx));
  if (zf || yf) ex = 0.0f;
  if (zf || xf) ey = 0.0f;
  if (yf || xf) ez = 0.0f;
  if (p.npsrc > 0) sources_3d(k, j, i, ex, ey, ez);
  if (vX) stb<T>(p.tout[0], ox * sz, ex);
  if (vj && vY) stb<T>(p.tout[1], oy * sz, ey);
  if (vk && vY) stb<T>(p.tout[2], oz * sz, ez);
}

// Blocks in x, y, z order, in runs of p.run that are dealt to the XCDs in turn
// (workgroup g runs on XCD g % 8).  Dealt one by one, a row, read by the
// blocks of its own, the next row and the next plane, was fetched by three L2s;
// eight long runs keep it in one but give the z-slab planes, with their CPML
// terms, to two XCDs.  72x120x200 with per-cell decay, per step with its
// source and DFT: one by one 78 us, 8 runs 77 us, 24 to 128 runs 67 to 68 us.
constexpr int kPhaseRounds = 6;
template <typename T, typename Off, bool kH, bool kCpml, int kCoef>
__global__ void __launch_bounds__(kBX * kBY)
phase_3d(PhaseParams p) {
  const int nbx = (p.nx + kBX) / kBX, nby = (p.ny + kBY) / kBY;
  const int t = (blockIdx.y * 8 + (blockIdx.x & 7)) * p.run + (blockIdx.x >> 3);
  const int row = t / nbx, bx = t - row * nbx;
  const int k = row / nby, by = row - k * nby;
  if (k > p.nz) return;
  const int i = bx * kBX + threadIdx.x;
  const int j = __builtin_amdgcn_readfirstlane(by * kBY + threadIdx.y);
  if (j > p.ny) return;
  const int kind = wave_kind(p, bx * kBX, j, k);
  if constexpr (kH) {
    if (kind == kWavePlain) h_cell<T, Off, kWavePlain, kCpml, kCoef>(p, i, j, k);
    else if (kind == kWaveXEdge) h_cell<T, Off, kWaveXEdge, kCpml, kCoef>(p, i, j, k);
    else h_cell<T, Off, kWaveGeneral, kCpml, kCoef>(p, i, j, k);
  } else {
    if (kind == kWavePlain) e_cell<T, Off, kWavePlain, kCpml, kCoef>(p, i, j, k);
    else if (kind == kWaveXEdge) e_cell<T, Off, kWaveXEdge, kCpml, kCoef>(p, i, j, k);
    else e_cell<T, Off, kWaveGeneral, kCpml, kCoef>(p, i, j, k);
  }
}

// ---------------------------------------------------------------------------
// 2D TMxy (Ez, Hx, Hy) on (ny, nx): kernels.py:731-811, 1217-1290
// ---------------------------------------------------------------------------

template <typename T, bool kCpml>
__global__ void __launch_bounds__(kBX * kBY)
h_phase_tm(PhaseParams p) {
  const int i = blockIdx.x * kBX + threadIdx.x;
  const int j = blockIdx.y * kBY + threadIdx.y;
  const int ny = p.ny, nx = p.nx;
  const int m = p.metallic;
  const void* Ez = p.src[2];  // (ny+1, nx+1)
  // Hx (ny, nx+1): corrected(+dEz/dy)
  if (j < ny && i <= nx) {
    const int o = j * (nx + 1) + i;
    const int ez = j * (nx + 1) + i;
    float d = (ld<T>(Ez, ez + nx + 1) - ld<T>(Ez, ez)) * metric_at(p, 1, j);
    if constexpr (kCpml) {
      d = cpml_correct(p, 0, d, j, [&](int q) { return q * (nx + 1) + i; });
    }
    float h = coef(p.dec[0], p.dec_st[0], p.dec_s[0], o) * ld<T>(p.tin[0], o) -
              coef(p.scf[0], p.scf_st[0], p.scf_s[0], o) * p.ratio * d;
    if (((m & kLeft) && i == 0) || ((m & kRight) && i == nx)) h = 0.0f;
    if (p.psrc[0].n > 0) h = group_add(p, p.psrc[0], 0, j, i, h);
    store_f(static_cast<T*>(p.tout[0]), o, h);
  }
  // Hy (ny+1, nx): corrected(-dEz/dx)
  if (j <= ny && i < nx) {
    const int o = j * nx + i;
    const int ez = j * (nx + 1) + i;
    float d = (ld<T>(Ez, ez + 1) - ld<T>(Ez, ez)) * metric_at(p, 2, i);
    if constexpr (kCpml) {
      d = cpml_correct(p, 1, d, i, [&](int q) { return j * (p.term[1].low + p.term[1].high) + q; });
    }
    float h = coef(p.dec[1], p.dec_st[1], p.dec_s[1], o) * ld<T>(p.tin[1], o) +
              coef(p.scf[1], p.scf_st[1], p.scf_s[1], o) * p.ratio * d;
    if (((m & kBottom) && j == 0) || ((m & kTop) && j == ny)) h = 0.0f;
    if (p.psrc[1].n > 0) h = group_add(p, p.psrc[1], 0, j, i, h);
    store_f(static_cast<T*>(p.tout[1]), o, h);
  }
}

// Backward difference of ghost-padded H along one axis (lattice.py:523-575):
// as ghost_diff, loading:
// ``idx`` is the linear index of coordinate ``c`` (valid only when c < N).
template <typename T>
__device__ __forceinline__ float ghost_bdiff(const void* h, int idx, int stride, int c,
                                             int N, bool metal_lo, bool metal_hi) {
  const float up = (c < N) ? ld<T>(h, idx) : (metal_hi ? 0.0f : ld<T>(h, idx - stride));
  const float lo = (c > 0) ? ld<T>(h, idx - stride) : (metal_lo ? 0.0f : ld<T>(h, idx));
  return up - lo;
}

template <typename T, bool kCpml>
__global__ void __launch_bounds__(kBX * kBY)
e_phase_tm(PhaseParams p) {
  const int i = blockIdx.x * kBX + threadIdx.x;
  const int j = blockIdx.y * kBY + threadIdx.y;
  const int ny = p.ny, nx = p.nx;
  const int m = p.metallic;
  if (j > ny || i > nx) return;
  const void* Hx = p.src[0];  // (ny, nx+1)
  const void* Hy = p.src[1];  // (ny+1, nx)
  const int o = j * (nx + 1) + i;
  float d0 = ghost_bdiff<T>(Hy, j * nx + i, 1, i, nx, m & kLeft, m & kRight) * metric_at(p, 2, i);
  float d1 = ghost_bdiff<T>(Hx, j * (nx + 1) + i, nx + 1, j, ny, m & kBottom, m & kTop) *
             metric_at(p, 1, j);
  if constexpr (kCpml) {
    d0 = cpml_correct(p, 0, d0, i, [&](int q) { return j * (p.term[0].low + p.term[0].high) + q; });
    d1 = cpml_correct(p, 1, d1, j, [&](int q) { return q * (nx + 1) + i; });
  }
  const float curl = d0 - d1;
  float e = coef(p.dec[2], p.dec_st[2], p.dec_s[2], o) * ld<T>(p.tin[2], o) +
            scf_at(p, 2, o) * p.ratio * curl;
  if (((m & kBottom) && j == 0) || ((m & kTop) && j == ny) ||
      ((m & kLeft) && i == 0) || ((m & kRight) && i == nx))
    e = 0.0f;
  if (p.psrc[2].n > 0) e = group_add(p, p.psrc[2], 0, j, i, e);
  store_f(static_cast<T*>(p.tout[2]), o, e);
}

template <typename T, typename Off, bool kH, int kCoef>
void launch3d(hipStream_t s, PhaseParams p) {
  const int64_t n = int64_t{(p.nx + kBX) / kBX} * ((p.ny + kBY) / kBY) * (p.nz + 1);
  BZH_REQUIRE(p.nz < 65535 && (p.ny + kBY) / kBY <= 65535, "3D phase grid too large");
  const int64_t rounds = std::max<int64_t>(kPhaseRounds, n >> 22);  // a launch dimension holds 2^32 threads
  p.run = static_cast<int32_t>((n + 8 * rounds - 1) / (8 * rounds));
  const dim3 block(kBX, kBY, 1), grid(8 * p.run, static_cast<uint32_t>(rounds), 1);
  if (p.nterms > 0) hipLaunchKernelGGL((phase_3d<T, Off, kH, true, kCoef>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((phase_3d<T, Off, kH, false, kCoef>), grid, block, 0, s, p);
}

template <typename T>
void dispatch3d(hipStream_t s, const PhaseParams& p, int phase) {
  const bool h = phase == BZH_PHASE_H;
  // H coefficients are nearly always scalars, E coefficients arrays or scalars
  // (variants without the general choices per component: 68 -> 64 us per step
  // at 72x120x200 with per-cell decay)
  bool any = false;
  for (int c = 0; c < 3; ++c)
    any = any || p.dec[c] == nullptr || p.scf[c] == nullptr || p.scf_ids[c] != nullptr ||
          (h && (p.dec_st[c] != 0 || p.scf_st[c] != 0));
  // the largest byte offset of any field or coefficient array
  if (int64_t{p.nz + 1} * (p.ny + 1) * (p.nx + 1) * 4 >= (int64_t{1} << 32)) {
    if (h) launch3d<T, uint64_t, true, kCoefAny>(s, p);
    else launch3d<T, uint64_t, false, kCoefAny>(s, p);
  } else if (h) {
    if (any) launch3d<T, uint32_t, true, kCoefAny>(s, p);
    else launch3d<T, uint32_t, true, kCoefScalar>(s, p);
  } else {
    if (any) launch3d<T, uint32_t, false, kCoefAny>(s, p);
    else launch3d<T, uint32_t, false, kCoefArray>(s, p);
  }
}

template <typename T>
void dispatch_tm(hipStream_t s, const PhaseParams& p, int phase) {
  dim3 block(kBX, kBY, 1);
  dim3 grid((p.nx + 1 + kBX - 1) / kBX, (p.ny + 1 + kBY - 1) / kBY, 1);
  const bool cpml = p.nterms > 0;
  if (phase == BZH_PHASE_H) {
    if (cpml) hipLaunchKernelGGL((h_phase_tm<T, true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((h_phase_tm<T, false>), grid, block, 0, s, p);
  } else {
    if (cpml) hipLaunchKernelGGL((e_phase_tm<T, true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((e_phase_tm<T, false>), grid, block, 0, s, p);
  }
}

}  // namespace

void launch_phase3d(hipStream_t s, const PhaseParams& p, int phase, int dtype) {
  BZH_REQUIRE(!p.scf_f16, "f16 coefficient arrays are read only by the fused step");
  BZH_REQUIRE(p.npsrc == 0 || p.step0 != nullptr,
              "folded source slabs are malformed");
  BZH_REQUIRE(p.npsrc == 0 || dtype == BZH_F32, "folded source slabs need float32 fields");
  switch (dtype) {
    case BZH_F32: dispatch3d<float>(s, p, phase); break;
    case BZH_BF16: dispatch3d<bf16_t>(s, p, phase); break;
    case BZH_F16: dispatch3d<__half>(s, p, phase); break;
    default: throw Failure{"unsupported field dtype"};
  }
  BZH_HIP(hipGetLastError());
}

void launch_phase_tm(hipStream_t s, const PhaseParams& p, int phase, int dtype) {
  BZH_REQUIRE(!p.scf_f16, "f16 coefficient arrays are read only by the fused step");
  BZH_REQUIRE(p.npsrc == 0 || p.step0 != nullptr,
              "folded source slabs are malformed");
  BZH_REQUIRE(p.npsrc == 0 || dtype == BZH_F32, "folded source slabs need float32 fields");
  switch (dtype) {
    case BZH_F32: dispatch_tm<float>(s, p, phase); break;
    case BZH_BF16: dispatch_tm<bf16_t>(s, p, phase); break;
    case BZH_F16: dispatch_tm<__half>(s, p, phase); break;
    default: throw Failure{"unsupported field dtype"};
  }
  BZH_HIP(hipGetLastError());
}

}  // namespace bzh
