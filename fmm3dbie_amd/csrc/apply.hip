// Layer-potential apply on gfx950 (lpcomp_{helm,lap}_comb_dir_addsub,
// helm_comb_dir.f:856-1208; lap_comb_dir.f90:806-1188):
//
//   pot = sum_{all oversampled j} K(x_i, y_j) s_j      (FMM3D call in the reference)
//       + sum_{near pairs} wnear . sigma                 (CSR correction, :1138-1151)
//       - sum_{near pairs} sum_{j in patch} K(x_i,y_j) s_j (subtraction, :1156-1193)
// with s_j = sigma_over_j * whtsover_j and K the combined kernel (alpha S + beta D).
//
// The FMM is replaced by an all-pairs sum, one density on the vector units (k_farsum) and
// blocks of densities on the matrix cores (k_farsum_mfma, k_farsum_split).  Two modes:
//   ADDSUB : all sources, then the near patches' contributions subtracted (the reference's
//            algebra);
//   MASKED : sources of the target's near patches are skipped inside the sum
//            (algebraically identical, no cancellation; used for FP32).
// Sources are sorted by patch, so the near-patch test is a moving pointer into the
// target's sorted near list.  Sources with |x-y| <= thresh are skipped in every sum
// (get_fmm_thresh, src/common/get_fmm_thresh.f:81).
// Laplace densities may be complex too: a real kernel applied to both parts.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

#include "apply.hpp"
#include "common.hpp"
#include "host_basis.hpp"

namespace {

constexpr int TPB = 256;

template <typename T>
struct V2 {
  T x, y;
};

// Source geometry record: x, y, z, nx, ny, nz (FP32: padded to 32 bytes).
template <typename T>
constexpr int GEO = sizeof(T) == 8 ? 6 : 8;

// Right-hand sides of a group on the matrix cores.
constexpr int MG = 16;

// Strengths of the far sum: sigma_over = I * sigma per patch, s = phase * sigma_over * w,
// one complex value per oversampled node and right-hand side, stored by groups of nr
// right-hand sides: group g, node i, right-hand side r of the group at (g nptso + i) nr + r.
// Right-hand sides from nrhs to the end of the last group are zero.
// A thread takes RB right-hand sides of one node (grid y).
// bmax (FP32, optional): the largest |Re s|, |Im s| of the workgroup's nodes for each right-hand
// side, at workgroup * right-hand sides (padded) + right-hand side.
template <typename T, int RB>
__global__ void __launch_bounds__(256) k_oversample(int64_t nptso, const int* __restrict__ opatch, const int64_t* __restrict__ ixyzs,
                             const int64_t* __restrict__ ixyzso, const int64_t* __restrict__ ioff,
                             const int* __restrict__ np_of, const double* __restrict__ imat,
                             const V2<T>* __restrict__ sigma, int nrhs, int64_t ldsig,
                             const T* __restrict__ wover, double pr, double pi, int nr, V2<T>* __restrict__ str,
                             float* __restrict__ bmax) {
  const int64_t it = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const bool in = it < nptso;
  const int64_t i = in ? it : nptso - 1;
  const int r0 = blockIdx.y * RB;
  const int ip = opatch[i];
  const int p = np_of[ip];
  const int64_t li = i - (ixyzso[ip] - 1);
  const double* row = imat + ioff[ip] + li * p;
  const int64_t s0 = ixyzs[ip] - 1;
  const double w = (double)wover[i];
  double sr[RB], si[RB];
  const V2<T>* sg[RB];
#pragma unroll
  for (int r = 0; r < RB; r++) {
    sr[r] = si[r] = 0.0;
    sg[r] = sigma + (int64_t)(r0 + r < nrhs ? r0 + r : 0) * ldsig + s0;
  }
  for (int l = 0; l < p; l++) {
    const double c = row[l];
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const V2<T> v = sg[r][l];
      sr[r] = fma(c, (double)v.x, sr[r]);
      si[r] = fma(c, (double)v.y, si[r]);
    }
  }
  const int g = r0 / nr;
  V2<T>* o = str + ((int64_t)g * nptso + i) * nr + (r0 - g * nr);
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const double a = sr[r] * w, b = si[r] * w;
    const bool live = r0 + r < nrhs;
    const V2<T> v = {live ? (T)(pr * a - pi * b) : (T)0, live ? (T)(pr * b + pi * a) : (T)0};
    if (in) o[r] = v;
    sr[r] = v.x;
    si[r] = v.y;
  }
  if constexpr (sizeof(T) == 4) {
    if (!bmax) return;
    __shared__ float wmax[4][RB];
#pragma unroll
    for (int r = 0; r < RB; r++) {
      float m = fmaxf(fabsf((float)sr[r]), fabsf((float)si[r]));  // (past the last node: that node's)
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
      if (threadIdx.x % 64 == 0) wmax[threadIdx.x / 64][r] = m;
    }
    __syncthreads();
    if (threadIdx.x < RB) {
      const int r = threadIdx.x;
      bmax[(int64_t)blockIdx.x * (gridDim.y * RB) + r0 + r] =
          fmaxf(fmaxf(wmax[0][r], wmax[1][r]), fmaxf(wmax[2][r], wmax[3][r]));
    }
  }
}

// Values that k_oversample leaves after the strengths of nr right-hand sides (bmax)
static int64_t bmax_values(int64_t nptso, int nr) { return (nptso + 255) / 256 * nr; }

// ---- kernel values of the far sum
// The combined kernel is K = (alpha + beta t (1 - ikr)) e^{ikr} / (4 pi r), t = (x - y).n / r^2.
// The plan factors it as phase * (a + t' (1 - ikr)) e^{ikr} / r with |a| <= 1 and the source
// normals scaled (apply_plan_scale): one complex strength per node instead of a charge and a
// dipole, and G = a + t' (1 - ikr) takes two fused multiply-adds.
// KIND 0: k = 0 (Laplace): a real kernel, no sine and cosine.  KIND 1: real wavenumber.  KIND
// 2: complex wavenumber, or (FP32) phases beyond the hardware sine's range, which are
// reduced to one revolution first; otherwise the FP32 phase k r / (2 pi) goes to the hardware
// sine and cosine directly (they take revolutions, valid below 256, which the plan checks
// against its bounding box): with KIND 1 the FP32 coordinates are stored in units of the
// wavelength (scaled before they are rounded to FP32), so that r is the phase; a and the normals
// carry the unit's powers, strengths and kernel values are those of the caller's units.
template <typename T>
struct FarPar {
  T ar, ai;    // a
  T kr, ki;    // wavenumber
  T khi, klo;  // FP64: k / pi as a sum of two doubles; FP32, KIND 2: khi = k / (2 pi)
};

// 1 / sqrt(x)
__device__ __forceinline__ float far_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double far_rsqrt(double x) { return rsqrt_halley(x); }

// From r^2, 1/r and d = (x - y).n': G and (c, s, q) with e^{ikr} / r = (c + i s) q.  A pair to
// be skipped passes rinv = 0: r is then 0, every factor finite and q zero, so that its
// contribution is an exact zero.
template <typename T, int KIND>
__device__ __forceinline__ void pair_factors(T r2, T rinv, T d, const FarPar<T>& P, T& gr, T& gi, T& c, T& s, T& q) {
  const T u = d * rinv;
  q = rinv;
  if constexpr (KIND == 0) {
    gr = fma(u, rinv, P.ar);
    gi = (T)0;
    c = (T)1;
    s = (T)0;
  } else {
    const T r = r2 * rinv;
    if constexpr (sizeof(T) == 4) {
      T rev = r;
      if constexpr (KIND == 2) {
        rev *= P.khi;
        rev -= rintf(rev);
      }
      s = __builtin_amdgcn_sinf(rev);
      c = __builtin_amdgcn_cosf(rev);
    } else {
      bool neg;
      sincos_turns(r, P.khi, P.klo, s, c, neg);
      q = neg ? -rinv : rinv;
    }
    if constexpr (KIND == 2) {
      T mag;
      if constexpr (sizeof(T) == 4) mag = __expf(-P.ki * r);
      else mag = exp(-P.ki * r);
      q *= mag;
      gr = fma(u * rinv, fma(P.ki, r, (T)1), P.ar);
    } else {
      gr = fma(u, rinv, P.ar);
    }
    gi = fma(-P.kr, u, P.ai);
  }
}

// The complex kernel value from the factors.
template <typename T, int KIND>
__device__ __forceinline__ void pair_value(T gr, T gi, T c, T s, T q, T& kr, T& ki) {
  if constexpr (KIND == 0) {
    kr = gr * q;
    ki = (T)0;
  } else {
    const T cq = c * q, sq = s * q;
    kr = gr * cq - gi * sq;
    ki = gr * sq + gi * cq;
  }
}

// The sources of a target's near patches, in source order: sources are sorted by patch and
// the near list of each target too, so [ea, eb) is the interval of the next near patch
// (patch p owns sources ixyzso[p]-1 .. ixyzso[p+1]-2), moved on by seek(j) to the first
// that ends after source j.
struct NearCursor {
  static constexpr int NONE = 0x7fffffff;
  const int* list;
  const int64_t* ixyzso;
  int64_t ptr = 0, end = 0;
  int ea = NONE, eb = NONE;
  __device__ __forceinline__ void seek(int j) {
    ea = NONE;
    eb = NONE;
    while (ptr < end) {
      const int p = list[ptr];
      const int e = (int)(ixyzso[p + 1] - 1);
      if (e > j) {
        ea = (int)(ixyzso[p] - 1);
        eb = e;
        break;
      }
      ptr++;
    }
  }
};

// Far sum on the vector units, one target per lane, one wavefront per workgroup:
// part[i] = sum over the sources of split blockIdx.y of K(x_i, y_j) s_j, for the NRHS
// right-hand sides of group blockIdx.z (the kernel value is computed once per group).
// Every lane works on the same source, whose geometry and strengths are wave-uniform: they
// come by scalar loads into scalar registers, and one operand of each vector instruction
// may be one of those, so that no LDS, barrier or vector register is spent on them.
// Bound by vector instruction issue: a pair takes 61 instructions in the add/subtract form of FP64
// with a real wavenumber (counted; 76 with a charge and a dipole strength per source, sincos_red
// and a Newton step more; 266 cycles of a SIMD per 64 pairs, before 330; the apply of 344064
// points 412 -> 337 ms, of 25920 points 4.44 -> 3.55 ms) and 27.5 in FP32 (93 cycles, before 103:
// 1.95 -> 1.85 ms for 43008 points), three of them hardware functions of 10 cycles.  Laplace,
// which ran the Helmholtz kernel with k = 0, takes 117 cycles in FP64 and 65 in FP32.
// MASK: sources of the target's near patches are skipped; tiles of STILE sources that hold
// none for any lane of the wavefront (nearly all) run without a test.
// !MASK: sources within thresh of the target are skipped: each pair is compared, and only
// if a lane of a block of UB sources finds one is the block summed again with the test.
// VALUE (one density): the kernel value first, then its product with the strength (2 instructions
// more).  In FP32 and wavelengths G alone is its true size times the unit, and a product with the
// strength could leave FP32's range where kernel value and result do not: units beyond
// UNIT32_MILD take this form (43008 points, k = 0.01: 1.89 ms against 1.83, error 4.8e-7 as before).
constexpr int STILE = 32;
constexpr double UNIT32_MILD = 16.0;
template <typename T, bool MASK, int KIND, int NRHS, bool VALUE = false>
__global__ void __launch_bounds__(64) k_farsum(int ntarg, const T* __restrict__ tx, const T* __restrict__ ty,
                                               const T* __restrict__ tz, int nsrc, const T* __restrict__ geo,
                                               const int64_t* __restrict__ ixyzso, const V2<T>* __restrict__ str,
                                               const int64_t* __restrict__ row_ptr, const int* __restrict__ near_sorted,
                                               FarPar<T> P, T thresh2, int chunk, int nrhs,
                                               V2<T>* __restrict__ part, int64_t ldpart) {
  const int64_t rg = blockIdx.z;
  str += rg * NRHS * nsrc;
  const int i = blockIdx.x * 64 + threadIdx.x;
  const bool act = i < ntarg;
  const T x = act ? tx[i] : (T)0, y = act ? ty[i] : (T)0, z = act ? tz[i] : (T)0;
  T accr[NRHS], acci[NRHS];
#pragma unroll
  for (int r = 0; r < NRHS; r++) { accr[r] = 0; acci[r] = 0; }
  const int jbeg = blockIdx.y * chunk;
  const int jend = chunk < nsrc - jbeg ? jbeg + chunk : nsrc;
  // source j: r^2 and, unless skip, its contribution
  auto pair = [&](int j, auto test) -> T {
    const T* g = geo + (int64_t)j * GEO<T>;
    const T dx = x - g[0], dy = y - g[1], dz = z - g[2];
    const T r2 = dx * dx + dy * dy + dz * dz;
    const T d = dx * g[3] + dy * g[4] + dz * g[5];
    T rinv = far_rsqrt(r2);
    if constexpr (!std::is_same<decltype(test), std::nullptr_t>::value) rinv = test(r2) ? rinv : (T)0;
    T gr, gi, c, s, q;
    pair_factors<T, KIND>(r2, rinv, d, P, gr, gi, c, s, q);
    const V2<T>* v = str + (int64_t)j * NRHS;
    if constexpr (NRHS == 1 && KIND != 0 && !VALUE) {
      const T ir = v[0].x * gr - v[0].y * gi, ii = v[0].x * gi + v[0].y * gr;
      accr[0] = fma(ir * c - ii * s, q, accr[0]);
      acci[0] = fma(ir * s + ii * c, q, acci[0]);
    } else {
      T vr, vi;
      pair_value<T, KIND>(gr, gi, c, s, q, vr, vi);
#pragma unroll
      for (int r = 0; r < NRHS; r++) {
        if constexpr (KIND == 0) {
          accr[r] = fma(vr, v[r].x, accr[r]);
          acci[r] = fma(vr, v[r].y, acci[r]);
        } else if constexpr (VALUE) {
          accr[r] += fma(vr, v[r].x, -(vi * v[r].y));
          acci[r] += fma(vr, v[r].y, vi * v[r].x);
        } else {
          accr[r] = fma(vr, v[r].x, fma(-vi, v[r].y, accr[r]));
          acci[r] = fma(vr, v[r].y, fma(vi, v[r].x, acci[r]));
        }
      }
    }
    return r2;
  };
  if constexpr (MASK) {
    // unrolled by 2 against rolled, cycles per 64 pairs: FP64 262 and 295, FP32 98 and 95
    constexpr int UN = sizeof(T) == 8 ? 2 : 1;
    NearCursor nc{near_sorted, ixyzso};
    if (act && jbeg < jend) {
      nc.ptr = row_ptr[i] - 1;
      nc.end = row_ptr[i + 1] - 1;
      nc.seek(jbeg);
    }
    for (int base = jbeg; base < jend; base += STILE) {
      const int cnt = jend - base < STILE ? jend - base : STILE;
      if (base >= nc.eb) nc.seek(base);
      if (__all(nc.ea >= base + cnt)) {
#pragma unroll UN
        for (int k = 0; k < cnt; k++) pair(base + k, nullptr);
      } else {
#pragma unroll 1
        for (int k = 0; k < cnt; k++) {
          const int j = base + k;
          if (j >= nc.eb) nc.seek(j);
          pair(j, [&](T) { return j < nc.ea; });
        }
      }
    }
  } else {
    constexpr int UB = 4;
    int j = jbeg;
    for (; j + UB <= jend; j += UB) {
      T sr[NRHS], si[NRHS];
#pragma unroll
      for (int r = 0; r < NRHS; r++) { sr[r] = accr[r]; si[r] = acci[r]; }
      bool close = false;
#pragma unroll
      for (int k = 0; k < UB; k++) close |= !(pair(j + k, nullptr) > thresh2);
      if (__any(close)) {
#pragma unroll
        for (int r = 0; r < NRHS; r++) { accr[r] = sr[r]; acci[r] = si[r]; }
#pragma unroll 1
        for (int k = 0; k < UB; k++) pair(j + k, [&](T r2) { return r2 > thresh2; });
      }
    }
    for (; j < jend; j++) pair(j, [&](T r2) { return r2 > thresh2; });
  }
  if (act) {
#pragma unroll
    for (int r = 0; r < NRHS; r++)
      if (rg * NRHS + r < nrhs)
        part[(int64_t)blockIdx.y * ldpart + (rg * NRHS + r) * ntarg + i] = {accr[r], acci[r]};
  }
}

// Far sum of a group of 16 right-hand sides on the matrix cores, FP64: the group's potentials
// are the complex product pot = K S of the target x source kernel matrix with the source x 16
// strength matrix.  A wavefront takes MT tiles of 16 targets; in a step of 4 sources lane l
// evaluates the pairs (target l % 16 of each tile, source l / 16) once on the vector units,
// and the 16x16x4 product of the matrix cores multiplies the 16 x 4 kernel blocks by the 4 x
// 16 strength blocks (lane l supplies source l / 16, right-hand side l % 16).  The complex
// product takes four real ones (Laplace: two, K being real).  Three (Gauss) would save 64 of
// these cycles, but leave the imaginary part an error relative to the real one: 1.9e-14 of
// itself for a real density at k = 0.01, where this form has 4.3e-16.
// The workgroup stages FT sources at a time in LDS, geometry and strengths; MT tiles share
// each LDS read.
// Bound by issue: on this chip FP64 matrix instructions do not overlap with vector ones of the
// same SIMD (measured: the times of wavefronts of either kind add up), so that the products' 4
// x 64 cycles and the kernel values of 64 pairs add.  The 16-density apply of 86016 points
// (139206 sources): 40.7 ms, with three products 38.3.
// Tiles of 128 sources, 1, 3 or 4 target tiles and an unrolled loop were all 1 to 15% slower.
typedef double dbl4 __attribute__((ext_vector_type(4)));
constexpr int FT = 64;  // sources per LDS tile
constexpr int FW = 4;   // wavefronts per workgroup
constexpr int MT = 2;   // tiles of 16 targets per wavefront
template <bool MASK, int KIND>
__global__ void __launch_bounds__(64 * FW)
    k_farsum_mfma(int ntarg, const double* __restrict__ tx, const double* __restrict__ ty,
                  const double* __restrict__ tz, int nsrc, const double* __restrict__ geo,
                  const int64_t* __restrict__ ixyzso, const V2<double>* __restrict__ str,
                  const int64_t* __restrict__ row_ptr, const int* __restrict__ near_sorted, FarPar<double> P,
                  double thresh2, int chunk, int nrhs, V2<double>* __restrict__ part, int64_t ldpart) {
  using T = double;
  constexpr int NT = MT, G = GEO<T>;
  __shared__ __align__(16) T lgeo[FT * G];
  __shared__ __align__(16) V2<T> lstr[FT * MG];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t rg = blockIdx.z;
  str += rg * MG * nsrc;
  const int t0 = (blockIdx.x * FW + wv) * (16 * NT);
  const int ks = lane >> 4;  // this lane's source within a step of 4
  T x[NT], y[NT], z[NT];
  dbl4 re[NT], im[NT];
  const int jbeg = blockIdx.y * chunk;
  const int jend = chunk < nsrc - jbeg ? jbeg + chunk : nsrc;
  NearCursor nc[NT];
  bool act[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = t0 + 16 * t + (lane & 15);
    act[t] = i < ntarg;
    x[t] = act[t] ? tx[i] : (T)0;
    y[t] = act[t] ? ty[i] : (T)0;
    z[t] = act[t] ? tz[i] : (T)0;
    re[t] = im[t] = dbl4{0.0, 0.0, 0.0, 0.0};
    nc[t] = NearCursor{near_sorted, ixyzso};
    if (MASK && act[t] && jbeg < jend) {
      nc[t].ptr = row_ptr[i] - 1;
      nc[t].end = row_ptr[i + 1] - 1;
      nc[t].seek(jbeg);
    }
  }
  for (int base = jbeg; base < jend; base += FT) {
    const int cnt = jend - base < FT ? jend - base : FT;
    __syncthreads();
    // sources past the tile's count: zero geometry and strengths (and skipped below)
    for (int e = threadIdx.x; e < FT * G; e += 64 * FW) lgeo[e] = e < cnt * G ? geo[(int64_t)base * G + e] : (T)0;
    for (int e = threadIdx.x; e < FT * MG; e += 64 * FW)
      lstr[e] = e < cnt * MG ? str[(int64_t)base * MG + e] : V2<T>{(T)0, (T)0};
    __syncthreads();
    // FULL: no source of the tile is skipped for any target of the wavefront
    auto step = [&](int k, auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      const int jl = k + ks, j = base + jl;
      const T* g = lgeo + jl * G;
      const T gx = g[0], gy = g[1], gz = g[2], nx = g[3], ny = g[4], nz = g[5];
      const V2<T> sv = lstr[jl * MG + (lane & 15)];  // source k + l / 16, right-hand side l % 16
      const T neg = -sv.y;
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const T dx = x[t] - gx, dy = y[t] - gy, dz = z[t] - gz;
        const T r2 = dx * dx + dy * dy + dz * dz;
        const T d = dx * nx + dy * ny + dz * nz;
        T rinv = far_rsqrt(r2);
        if constexpr (!FULL) {
          if (MASK && j >= nc[t].eb) nc[t].seek(j);
          rinv = (act[t] && jl < cnt && (MASK ? j < nc[t].ea : r2 > thresh2)) ? rinv : (T)0;
        }
        T gr, gi, c, s, q, vr, vi;
        pair_factors<T, KIND>(r2, rinv, d, P, gr, gi, c, s, q);
        pair_value<T, KIND>(gr, gi, c, s, q, vr, vi);
        re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vr, sv.x, re[t], 0, 0, 0);
        im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vr, sv.y, im[t], 0, 0, 0);
        if constexpr (KIND != 0) {
          re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vi, neg, re[t], 0, 0, 0);
          im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vi, sv.x, im[t], 0, 0, 0);
        }
      }
    };
    bool full = MASK && cnt == FT;
    if constexpr (MASK) {
      bool mine = true;
#pragma unroll
      for (int t = 0; t < NT; t++) {
        if (base >= nc[t].eb) nc[t].seek(base);
        mine = mine && act[t] && nc[t].ea >= base + cnt;
      }
      full = full && __all(mine);
    }
    if (full) {
#pragma unroll 1
      for (int k = 0; k < FT; k += 4) step(k, std::true_type{});
    } else {
#pragma unroll 1
      for (int k = 0; k < cnt; k += 4) step(k, std::false_type{});
    }
  }
  // accumulator element e of lane l: target l / 16 + 4 e of the tile, right-hand side l % 16
  const int r = (int)rg * MG + (lane & 15);
  if (r < nrhs) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int it = t0 + 16 * t + ks + 4 * e;
        if (it < ntarg) part[(int64_t)blockIdx.y * ldpart + (int64_t)r * ntarg + it] = {re[t][e], im[t][e]};
      }
  }
}

// Far sum of all NG groups of 16 right-hand sides of a block, FP32.  The kernel values are
// computed once for all groups, and the products run in bfloat16, where the matrix cores have
// sixteen times their FP32 rate, exact products and FP32 sums: each value is split into three
// bfloat16 terms (hi + mid + lo, rounded to nearest, is the FP32 value to its last bit), and six
// products of terms take the place of one (those left out are below 2^-26 of it), as in Henry, Tang
// and Heinecke, Leveraging the bfloat16 artificial intelligence datatype for higher-precision
// computations, ARITH 2019.
// A wavefront takes MT tiles of 16 targets; in a tile of ST = 32 sources lane l evaluates the pairs
// (target l % 16, sources 8 (l / 16) ..) on the vector units, which are the operand of the 16x16x32
// products as they stand.  The workgroup stages the sources' geometry and the split strengths in
// LDS, in the order in which the lanes read them; the next tile's are loaded while one is summed.
// The strengths of a right-hand side are scaled by the power of two that takes the largest to 1
// and its potentials back: the last term of an FP32 value, 2^-24 of it, is then above bfloat16's
// smallest value whatever the size of a density (unscaled, strengths of 1e-34 lose 1e-5).  The
// largest comes from k_oversample's workgroups.  (Scaled by tiles instead, with no such pass, 16
// densities took 18.1 ms and 64 37.4.)
// The complex product takes four real ones, as in k_farsum_mfma, and a tile's products are
// summed by themselves before they are added to the potentials: the matrix cores round each sum
// of a chain downwards, which over all sources would add up (error of the 64-density apply below
// against the FP64 one 3.1e-6; 3.8e-7 in this way).  Re K Re s and Im K Im s have a sum each,
// which costs less than to negate an operand.
// Bound by issue: per 64 pairs 3 matrix and 39 vector instructions with one group, 12 and 52 with
// four (kernel values and splits, sums, and the staging, which MT = 2 tiles share): 184 and 381
// cycles of a SIMD.  The apply of 86016 points (139206 sources): 16 densities 15.4 ms, 32 22.8, 48
// 30.6, 64 34.8; in FP32 products, a group at a time, 19.3 ms for each 16.
typedef float flt2 __attribute__((ext_vector_type(2)));
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
constexpr int ST = 32;  // sources per tile
struct Split8 {         // the terms of eight values
  union {
    bf8 v;
    bf2 p[4];
  } t[3];
};
// The next terms of a and b, which keep what is left
__device__ __forceinline__ bf2 next_term(float& a, float& b) {
  const bf2 h = __builtin_convertvector(flt2{a, b}, bf2);
  a -= (float)h.x;
  b -= (float)h.y;
  return h;
}

template <int KIND, int NG>
__global__ void __launch_bounds__(64 * FW, 2)
    k_farsum_split(int ntarg, const float* __restrict__ tx, const float* __restrict__ ty, const float* __restrict__ tz,
                   int nsrc, const float* __restrict__ geo, const int64_t* __restrict__ ixyzso,
                   const V2<float>* __restrict__ str, const float* __restrict__ bmax,
                   const int64_t* __restrict__ row_ptr, const int* __restrict__ near_sorted, FarPar<float> P, int chunk,
                   int nrhs, V2<float>* __restrict__ part, int64_t ldpart) {
  using T = float;
  constexpr int NM = KIND == 0 ? 1 : 2;  // kernel matrices: Re K, Im K
  constexpr int SI = NG == 1 ? 2 : (NG == 2 ? 4 : 8);  // sources that a thread stages, of one right-hand side
  constexpr int NT = MT;
  __shared__ __align__(16) T lgeo[ST * 8];
  __shared__ __align__(16) bf8 lstr[NG][2][3][64];  // Re s, Im s
  __shared__ int lexp[NG * MG];                     // exponent bits of a right-hand side's largest strength
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int t0 = (blockIdx.x * FW + wv) * (16 * NT);
  const int ks = lane >> 4;  // this lane's sources: 8 ks .. 8 ks + 7 of a tile
  const int jbeg = blockIdx.y * chunk;
  const int jend = chunk < nsrc - jbeg ? jbeg + chunk : nsrc;
  T x[NT], y[NT], z[NT];
  NearCursor nc[NT];
  bool act[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = t0 + 16 * t + (lane & 15);
    act[t] = i < ntarg;
    x[t] = act[t] ? tx[i] : (T)0;
    y[t] = act[t] ? ty[i] : (T)0;
    z[t] = act[t] ? tz[i] : (T)0;
    nc[t] = NearCursor{near_sorted, ixyzso};
    if (act[t] && jbeg < jend) {
      nc[t].ptr = row_ptr[i] - 1;
      nc[t].end = row_ptr[i + 1] - 1;
      nc[t].seek(jbeg);
    }
  }
  // this thread's part of a tile: right-hand side sr of group sg, sources sj .. sj + SI - 1
  const int sr = threadIdx.x & 15, sj = SI * ((threadIdx.x >> 4) % (ST / SI)), sg = (threadIdx.x >> 4) / (ST / SI);
  const bool stager = sg < NG;
  const V2<T>* sp = str + (int64_t)(stager ? sg : 0) * nsrc * MG + sr;
  for (int r = threadIdx.x; r < NG * MG; r += 64 * FW) lexp[r] = 0;
  __syncthreads();
  {
    constexpr int PER = 64 * FW / (NG * MG);  // threads per right-hand side
    const int r = threadIdx.x % (NG * MG), nb = (nsrc + 255) / 256;
    float m = 0.0f;
    if (threadIdx.x < PER * NG * MG)
      for (int b = threadIdx.x / (NG * MG); b < nb; b += PER) m = fmaxf(m, bmax[(int64_t)b * (NG * MG) + r]);
    atomicMax(lexp + r, __float_as_int(m) >> 23);
  }
  __syncthreads();
  // 2^(e - 127) is the unit of a right-hand side, 2^(127 - e) its inverse: both are normal
  auto unit_exp = [&](int r) {
    const int e = lexp[r];
    return e < 1 ? 1 : (e > 253 ? 253 : e);
  };
  const T scale = __int_as_float((254 - unit_exp(stager ? sg * MG + sr : 0)) << 23);
  V2<T> next[SI];
  T nextg;  // and one value of the geometry
  static_assert(ST * 8 == 64 * FW, "");
  // (loads without a condition, in flight together while a tile is summed; sources past the chunk
  // are zeroed below)
  auto load = [&](int base) {
#pragma unroll
    for (int u = 0; u < SI; u++) {
      const int j = base + sj + u;
      next[u] = sp[(int64_t)(j < nsrc ? j : nsrc - 1) * MG];
    }
    const int64_t e = (int64_t)base * 8 + threadIdx.x;
    nextg = geo[e < (int64_t)nsrc * 8 ? e : 0];
  };
  auto stage = [&](int base) {
    lgeo[threadIdx.x] = base + (int)(threadIdx.x / 8) < jend ? nextg : (T)0;
#pragma unroll
    for (int u = 0; u < SI; u++)
      if (base + sj + u >= jend) next[u] = V2<T>{0.0f, 0.0f};
    if (!stager) return;
    bf2* o = reinterpret_cast<bf2*>(&lstr[sg][0][0][sj / 8 * 16 + sr]) + (sj % 8) / 2;
#pragma unroll
    for (int m = 0; m < 2; m++) {
      bf2 v[3][SI / 2];
#pragma unroll
      for (int u = 0; u < SI; u += 2) {
        T a = scale * (m == 0 ? next[u].x : next[u].y);
        T b = scale * (m == 0 ? next[u + 1].x : next[u + 1].y);
#pragma unroll
        for (int k = 0; k < 3; k++) v[k][u / 2] = next_term(a, b);
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        bf2* q = o + (m * 3 + k) * 64 * 4;
        if constexpr (SI == 8) *reinterpret_cast<bf8*>(q) = *reinterpret_cast<const bf8*>(v[k]);
        else if constexpr (SI == 4) *reinterpret_cast<bf4*>(q) = *reinterpret_cast<const bf4*>(v[k]);
        else *q = v[k][0];
      }
    }
  };
  flt4 re[NT][NG], im[NT][NG];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int g = 0; g < NG; g++) re[t][g] = im[t][g] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
  if (jbeg < jend) load(jbeg);
#pragma unroll 1
  for (int base = jbeg; base < jend; base += ST) {
    __syncthreads();
    stage(base);
    __syncthreads();
    if (base + ST < jend) load(base + ST);
    bool mine = base + ST <= jend;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      if (base >= nc[t].eb) nc[t].seek(base);
      mine = mine && act[t] && nc[t].ea >= base + ST;
    }
    Split8 A[NT][NM];
    // FULL: no source of the step is skipped for any target of the wavefront
    auto eval = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        T gg[2][6];
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
          for (int e = 0; e < 6; e++) gg[v][e] = lgeo[(8 * ks + u + v) * 8 + e];
#pragma unroll
        for (int t = 0; t < NT; t++) {
          T vr[2], vi[2];
#pragma unroll
          for (int v = 0; v < 2; v++) {
            const T* g = gg[v];
            const T dx = x[t] - g[0], dy = y[t] - g[1], dz = z[t] - g[2];
            const T r2 = dx * dx + dy * dy + dz * dz;
            const T d = dx * g[3] + dy * g[4] + dz * g[5];
            T rinv = far_rsqrt(r2);
            if constexpr (!FULL) {
              const int j = base + 8 * ks + u + v;
              if (j >= nc[t].eb) nc[t].seek(j);
              rinv = (act[t] && j < jend && j < nc[t].ea) ? rinv : (T)0;
            }
            T gr, gi, c, s, q;
            pair_factors<T, KIND>(r2, rinv, d, P, gr, gi, c, s, q);
            pair_value<T, KIND>(gr, gi, c, s, q, vr[v], vi[v]);
          }
#pragma unroll
          for (int k = 0; k < 3; k++) {
            A[t][0].t[k].p[u / 2] = next_term(vr[0], vr[1]);
            if constexpr (NM == 2) A[t][1].t[k].p[u / 2] = next_term(vi[0], vi[1]);
          }
        }
      }
    };
    if (__all(mine)) eval(std::true_type{});
    else eval(std::false_type{});
#pragma unroll
    for (int g = 0; g < NG; g++) {
      flt4 rr[NT], ii[NT], mix[NT];  // sums of Re K Re s, Im K Im s, Re K Im s + Im K Re s
#pragma unroll
      for (int t = 0; t < NT; t++) rr[t] = ii[t] = mix[t] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int m = 0; m < 2; m++) {
        bf8 b[3];
#pragma unroll
        for (int k = 0; k < 3; k++) b[k] = lstr[g][m][k][lane];
        auto mul = [&](int km, flt4(&sum)[NT]) {
          constexpr int ka[6] = {2, 0, 1, 1, 0, 0}, kb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
          for (int e = 0; e < 6; e++)
#pragma unroll
            for (int t = 0; t < NT; t++)
              sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[t][km].t[ka[e]].v, b[kb[e]], sum[t], 0, 0, 0);
        };
        mul(0, m == 0 ? rr : mix);
        if constexpr (NM == 2) mul(1, m == 0 ? mix : ii);
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        re[t][g] += rr[t] - ii[t];
        im[t][g] += mix[t];
      }
    }
  }
  // accumulator element e of lane l: target 4 (l / 16) + e of the tile, right-hand side l % 16
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int g = 0; g < NG; g++) {
      const int r = g * MG + (lane & 15);
      if (r >= nrhs) continue;
      const T unit = __int_as_float(unit_exp(r) << 23);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int it = t0 + 16 * t + 4 * ks + e;
        if (it < ntarg)
          part[(int64_t)blockIdx.y * ldpart + (int64_t)r * ntarg + it] = {unit * re[t][g][e], unit * im[t][g][e]};
      }
    }
}

// pot[r][i] = (sum over source splits of part) / (4 pi)
template <typename T>
__global__ void k_farsum_reduce(int64_t ntarg, int nrhs, int nsplit, const V2<T>* __restrict__ part,
                                int64_t ldpart, V2<T>* __restrict__ pot, int64_t ldpot) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (i >= ntarg || r >= nrhs) return;
  T sr = 0, si = 0;
  for (int sp = 0; sp < nsplit; sp++) {
    const V2<T> v = part[(int64_t)sp * ldpart + r * ntarg + i];
    sr += v.x;
    si += v.y;
  }
  pot[r * ldpot + i] = {(T)(sr * (T)OVER4PI), (T)(si * (T)OVER4PI)};
}

// What the near subtraction (add/subtract form) needs: targets, sources and strengths.
struct SubArgs {
  const double *tx, *ty, *tz, *geo;
  const V2<double>* str;
  int64_t nptso;
  int nr;  // right-hand sides per strength group
  const int64_t *col_ind, *ixyzso;
  FarPar<double> P;
  double thresh2;
};

// Smooth-rule contributions of target i's near patches (CSR entries j0..j1), subtracted from
// the lane's sums of right-hand sides rb .. rb + RB - 1.  Four patches at a time, 16 lanes
// each: a patch's 15 to 45 oversampled nodes fill 16 lanes better than 64 (one patch at a
// time on all lanes took 24 us for 1920 and 182 us for 25920 targets).
template <int RB>
__device__ __forceinline__ void near_sub(const SubArgs& S, int64_t i, int64_t j0, int64_t j1, int rb, int nrhs,
                                         double (&ar)[RB], double (&ai)[RB]) {
  const int lane = threadIdx.x % 64;
  const double x = S.tx[i], y = S.ty[i], z = S.tz[i];
  for (int64_t jj = j0 + (lane >> 4); jj < j1; jj += 4) {
    const int64_t ip = S.col_ind[jj] - 1;
    const int64_t e = S.ixyzso[ip + 1] - 1;
    for (int64_t j = S.ixyzso[ip] - 1 + (lane & 15); j < e; j += 16) {
      const double* g = S.geo + 6 * j;
      const double dx = x - g[0], dy = y - g[1], dz = z - g[2];
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double d = dx * g[3] + dy * g[4] + dz * g[5];
      const double rinv = r2 > S.thresh2 ? far_rsqrt(r2) : 0.0;
      double gr, gi, c, s, q, vr, vi;
      if (S.P.ki != 0.0) pair_factors<double, 2>(r2, rinv, d, S.P, gr, gi, c, s, q);
      else if (S.P.kr != 0.0) pair_factors<double, 1>(r2, rinv, d, S.P, gr, gi, c, s, q);
      else pair_factors<double, 0>(r2, rinv, d, S.P, gr, gi, c, s, q), gi = S.P.ai;
      pair_value<double, 1>(gr, gi, c, s, -OVER4PI * q, vr, vi);
#pragma unroll
      for (int r = 0; r < RB; r++) {
        if (rb + r < nrhs) {
          const int g_ = (rb + r) / S.nr;
          const V2<double> v = S.str[((int64_t)g_ * S.nptso + j) * S.nr + (rb + r - g_ * S.nr)];
          ar[r] = fma(vr, v.x, fma(-vi, v.y, ar[r]));
          ai[r] = fma(vr, v.y, fma(vi, v.x, ai[r]));
        }
      }
    }
  }
}

// Near subtraction alone (after the general CSR kernel): one wavefront per target.
__global__ void k_near_sub(int64_t ntarg, const int64_t* __restrict__ row_ptr, SubArgs S, int nrhs,
                           V2<double>* __restrict__ pot, int64_t ldpot) {
  const int64_t i = blockIdx.x * (int64_t)(blockDim.x / 64) + threadIdx.x / 64;
  if (i >= ntarg) return;
  for (int r = 0; r < nrhs; r++) {
    double ar[1] = {0.0}, ai[1] = {0.0};
    near_sub<1>(S, i, row_ptr[i] - 1, row_ptr[i + 1] - 1, r, nrhs, ar, ai);
    const double sr = wave_sum(ar[0]), si = wave_sum(ai[0]);
    if (threadIdx.x % 64 == 0) {
      pot[r * ldpot + i].x += sr;
      pot[r * ldpot + i].y += si;
    }
  }
}

// General CSR correction (any patch sizes): one thread per target row.
template <typename T, typename TW>
__global__ void k_csr_gen(int64_t ntarg, const int64_t* __restrict__ row_ptr, const int64_t* __restrict__ col_ind,
                          const int64_t* __restrict__ iquad, const int64_t* __restrict__ ixyzs,
                          const V2<TW>* __restrict__ wnear, const V2<T>* __restrict__ sigma, int64_t ldsig,
                          int nrhs, V2<T>* __restrict__ pot, int64_t ldpot) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= ntarg) return;
  for (int r = 0; r < nrhs; r++) {
    double sr = 0.0, si = 0.0;
    for (int64_t jj = row_ptr[i] - 1; jj < row_ptr[i + 1] - 1; jj++) {
      const int64_t ip = col_ind[jj] - 1;
      const int64_t s0 = ixyzs[ip] - 1, p = ixyzs[ip + 1] - ixyzs[ip], q0 = iquad[jj] - 1;
      for (int64_t l = 0; l < p; l++) {
        const V2<TW> w = wnear[q0 + l];
        const V2<T> s = sigma[r * ldsig + s0 + l];
        sr += (double)w.x * (double)s.x - (double)w.y * (double)s.y;
        si += (double)w.x * (double)s.y + (double)w.y * (double)s.x;
      }
    }
    pot[r * ldpot + i].x += (T)sr;
    pot[r * ldpot + i].y += (T)si;
  }
}

// Far-sum reduction fused with the CSR near correction and, with SUB (FP64 add/subtract
// form), the near subtraction, for all right-hand sides (uniform patch size p): one
// wavefront per target row, lanes over the row's contiguous wnear segment; every wnear
// element is loaded once per group of RB right-hand sides.  One launch instead of three for
// a small problem (1920 points: the whole apply 83 -> 37 us, with the far sum's 53 us cut by
// its finer source splits).
//   pot[r][i] = (sum over source splits of part[r][i]) / (4 pi) + sum_e wnear_e sigma_r(src_e)
// PC > 0: the patch size as a compile-time constant (the orders 1..10), else p_rt.
template <typename T, typename TW, int RB, int PC, bool SUB>
__global__ void k_reduce_csr(int64_t ntarg, int nrhs, int nsplit, const V2<T>* __restrict__ part, int64_t ldpart,
                             const int64_t* __restrict__ row_ptr, const int* __restrict__ csr_src,
                             const int64_t* __restrict__ iquad, int p_rt,
                             const V2<TW>* __restrict__ wnear, const V2<T>* __restrict__ sigma, int64_t ldsig,
                             V2<T>* __restrict__ pot, int64_t ldpot, SubArgs S) {
  const int p = PC > 0 ? PC : p_rt;
  const int64_t i = blockIdx.x * (int64_t)(blockDim.x / 64) + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (i >= ntarg) return;
  const int64_t j0 = row_ptr[i] - 1, j1 = row_ptr[i + 1] - 1;
  const int64_t q0 = j0 < j1 ? iquad[j0] - 1 : 0;
  const int64_t ne = (j1 - j0) * (int64_t)p;
  for (int rb = 0; rb < nrhs; rb += RB) {
    double ar[RB], ai[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) { ar[r] = 0.0; ai[r] = 0.0; }
    for (int e = lane; e < (int)ne; e += 64) {
      const int k = e / p;  // patch entry of the row (compile-time divisor for the orders 1..10)
      const int64_t src = csr_src[j0 + k] + (e - k * p);
      const V2<TW> w = wnear[q0 + e];
#pragma unroll
      for (int r = 0; r < RB; r++) {
        if (rb + r < nrhs) {
          const V2<T> sg = sigma[(rb + r) * ldsig + src];
          ar[r] += (double)w.x * (double)sg.x - (double)w.y * (double)sg.y;
          ai[r] += (double)w.x * (double)sg.y + (double)w.y * (double)sg.x;
        }
      }
    }
    if constexpr (SUB) near_sub<RB>(S, i, j0, j1, rb, nrhs, ar, ai);
    // the source splits: with one right-hand side the lanes share them
    T fr = 0, fi = 0;
    if constexpr (RB == 1) {
      for (int sp = lane; sp < nsplit; sp += 64) {
        const V2<T> v = part[(int64_t)sp * ldpart + rb * ntarg + i];
        fr += v.x;
        fi += v.y;
      }
      fr = wave_sum(fr);
      fi = wave_sum(fi);
    }
    double mr = 0.0, mi = 0.0;
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const double sr = wave_sum(ar[r]), si = wave_sum(ai[r]);
      if (lane == r) { mr = sr; mi = si; }
    }
    const int r = rb + lane;
    if (lane < RB && r < nrhs) {
      if constexpr (RB > 1) {
        for (int sp = 0; sp < nsplit; sp++) {
          const V2<T> v = part[(int64_t)sp * ldpart + r * ntarg + i];
          fr += v.x;
          fi += v.y;
        }
      }
      pot[r * ldpot + i] = {(T)(fr * (T)OVER4PI + (T)mr), (T)(fi * (T)OVER4PI + (T)mi)};
    }
  }
}

// Sum of the far-sum partials over the source splits, in place into split 0: a workgroup
// of 256 threads takes 64 targets, thread (t, g) adds splits g, g + 4, ... of target t
// (loads coalesced over t) and the four groups meet in LDS.
template <typename T>
__global__ void __launch_bounds__(256) k_split_sum(int64_t ntarg, int nsplit, V2<T>* __restrict__ part,
                                                   int64_t ldpart) {
  __shared__ V2<T> sh[4][64];
  const int t = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t i = blockIdx.x * (int64_t)64 + t;
  const int64_t r = blockIdx.y;
  T sr = 0, si = 0;
  if (i < ntarg) {
    const V2<T>* pp = part + r * ntarg + i;
#pragma unroll 4
    for (int sp = g; sp < nsplit; sp += 4) {
      const V2<T> v = pp[(int64_t)sp * ldpart];
      sr += v.x;
      si += v.y;
    }
  }
  sh[g][t] = {sr, si};
  __syncthreads();
  if (g == 0 && i < ntarg) {
    const V2<T> a = sh[1][t], b = sh[2][t], c = sh[3][t];
    part[r * ntarg + i] = {(sr + a.x) + (b.x + c.x), (si + a.y) + (b.y + c.y)};
  }
}

// constant fill (tuning densities)
template <typename T>
__global__ void k_fill(int64_t n, T* __restrict__ a, T v) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// Source geometry records (normals scaled by ns; FP32 coordinates by unit32 and normals by its
// square) from rows x y z du dv n of 12 doubles
__global__ void k_geo(int64_t n, const double* __restrict__ s12, double ns, double unit32,
                      double* __restrict__ g64, float* __restrict__ g32) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* s = s12 + 12 * i;
  const double v[6] = {s[0], s[1], s[2], ns * s[9], ns * s[10], ns * s[11]};
  for (int m = 0; m < 6; m++) {
    g64[GEO<double> * i + m] = v[m];
    g32[GEO<float> * i + m] = (float)(unit32 * (m < 3 ? v[m] : unit32 * v[m]));
  }
  g32[GEO<float> * i + 6] = g32[GEO<float> * i + 7] = 0.0f;
}

struct Targets {
  double* t64[3];
  float* t32[3];
};
__global__ void k_split_targ(int64_t n, const double* __restrict__ t, int64_t stride, double unit32, Targets T) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int m = 0; m < 3; m++) {
    const double v = t[stride * i + m];
    T.t64[m][i] = v;
    T.t32[m][i] = (float)(unit32 * v);
  }
}

template <typename A, typename B>
__global__ void k_convert(int64_t n, const A* __restrict__ a, B* __restrict__ b) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = (B)a[i];
}

__global__ void k_real_to_cplx(int64_t n, const double* __restrict__ a, V2<double>* __restrict__ b) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = {a[i], 0.0};
}

__global__ void k_cplx_to_real(int64_t n, const V2<double>* __restrict__ a, double* __restrict__ b) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i].x;
}

template <typename T>
T* dal(size_t n) {
  void* p = nullptr;
  if (hipMalloc(&p, (n ? n : 1) * sizeof(T)) != hipSuccess) return nullptr;
  return (T*)p;
}

// Workgroups of one wavefront that fill the chip twice (256 CUs x 4 SIMDs x 8 wavefronts)
constexpr int64_t FAR_FILL = 16384;
// Far-sum partials (splits x targets) up to which the CSR kernel sums them itself
constexpr int64_t SPLIT_INLINE = (int64_t)1 << 19;

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

#define ACHK(x)                                                                    \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) {                                                        \
      fprintf(stderr, "fmm3dbie_amd: %s failed: %s\n", #x, hipGetErrorString(e_)); \
      return -1;                                                                   \
    }                                                                              \
  } while (0)

ApplyPlan::~ApplyPlan() {
  apply_plan_free_ws(this);
  for (void* p : owned)
    if (p) (void)hipFree(p);
}

template <typename T>
static T* own(ApplyPlan* P, size_t n) {
  T* p = dal<T>(n);
  P->owned.push_back((void*)p);
  return p;
}

// The far sum's kernel: alpha + beta t (1 - ikr) = (phase mu) (a + ns t (1 - ikr)) with mu the
// power of two above |alpha| and |beta|, phase = beta / |beta| (1 without a double layer),
// a = alpha / (phase mu) and ns = |beta| / mu: |a|, ns <= 1 in any units of alpha and beta,
// and for beta = 1 (the usual double layer) no factor is rounded.
static void apply_plan_scale(ApplyPlan* P) {
  const double ar = P->alpha[0], ai = P->helm ? P->alpha[1] : 0.0;
  const double br = P->beta[0], bi = P->helm ? P->beta[1] : 0.0;
  const double bm = std::hypot(br, bi), m = std::max(std::hypot(ar, ai), bm);
  int e = 0;
  (void)std::frexp(m, &e);
  const double mu = std::ldexp(1.0, e);
  const double pr = bm > 0.0 ? br / bm : 1.0, pi = bm > 0.0 ? bi / bm : 0.0;
  P->far_phase[0] = m > 0.0 ? pr * mu : 0.0;
  P->far_phase[1] = m > 0.0 ? pi * mu : 0.0;
  P->far_a[0] = (ar * pr + ai * pi) / mu;
  P->far_a[1] = (ai * pr - ar * pi) / mu;
  P->far_ns = bm / mu;
}

int apply_plan_build(ApplyPlan* P, const ApplyPlanInput& in, hipStream_t s) {
  P->npatches = in.npatches;
  P->npts = in.npts;
  P->nptso = in.nptso;
  P->ntarg = in.targs ? in.ntarg : in.npts;
  P->nnz = in.nnz;
  P->helm = in.helm;
  P->zk[0] = in.zk[0]; P->zk[1] = in.zk[1];
  P->alpha[0] = in.alpha[0]; P->alpha[1] = in.alpha[1];
  P->beta[0] = in.beta[0]; P->beta[1] = in.beta[1];
  apply_plan_scale(P);
  const int64_t npat = in.npatches, N = P->ntarg, NO = in.nptso;
  const double* tsrc = in.targs ? in.targs : in.srcvals;  // target coordinates
  const int64_t tstride = in.targs ? in.ndtarg : 12;
  // the far sum counts nodes and targets, rounded up to a tile, in 32 bits (more do not fit the
  // card: 96 bytes of geometry records and strengths per node and 12 KB of partial sums per target)
  if (NO > INT32_MAX - 4096 || N > INT32_MAX - 4096) {
    fprintf(stderr, "fmm3dbie_amd: %lld oversampled nodes and %lld targets: at most 2^31 - 4097 of each\n",
            (long long)NO, (long long)N);
    return -2;
  }
  // host-side tables: interpolation matrices per (norder, nover), patch of each
  // oversampled point, sorted near lists, uniform-p check
  std::vector<int64_t> ioff(npat);
  std::vector<int> np_of(npat), opatch(NO);
  std::vector<double> imat_all;
  std::vector<std::pair<int, int>> keys;
  std::vector<int64_t> koff;
  P->uniform_p = 0;
  int p0 = -1;
  bool uni = true;
  for (int64_t i = 0; i < npat; i++) {
    const int no = (int)in.norders[i], nv = (int)in.novers[i];
    int64_t off = -1;
    for (size_t k = 0; k < keys.size(); k++)
      if (keys[k].first == no && keys[k].second == nv) off = koff[k];
    if (off < 0) {
      std::vector<double> im;
      fmmhost::interp_matrix(no, nv, im);
      off = (int64_t)imat_all.size();
      imat_all.insert(imat_all.end(), im.begin(), im.end());
      keys.push_back({no, nv});
      koff.push_back(off);
    }
    ioff[i] = off;
    np_of[i] = (int)(in.ixyzs[i + 1] - in.ixyzs[i]);
    if (p0 < 0) p0 = np_of[i];
    if (np_of[i] != p0) uni = false;
    for (int64_t j = in.ixyzso[i] - 1; j < in.ixyzso[i + 1] - 1; j++) opatch[j] = (int)i;
  }
  P->uniform_p = uni ? p0 : 0;
  std::vector<int> nsorted(in.nnz);
  for (int64_t t = 0; t < N; t++) {
    const int64_t a = in.row_ptr[t] - 1, b = in.row_ptr[t + 1] - 1;
    for (int64_t j = a; j < b; j++) nsorted[j] = (int)(in.col_ind[j] - 1);
    std::sort(nsorted.begin() + a, nsorted.begin() + b);
  }
  // threshold: 2^-51 * max bounding-box edge of sources and targets
  double mn[3], mx[3];
  for (int m = 0; m < 3; m++) mn[m] = mx[m] = in.srcover[m];
  for (int64_t i = 0; i < NO; i++)
    for (int m = 0; m < 3; m++) {
      const double v = in.srcover[12 * i + m];
      mn[m] = v < mn[m] ? v : mn[m];
      mx[m] = v > mx[m] ? v : mx[m];
    }
  for (int64_t i = 0; i < N; i++)
    for (int m = 0; m < 3; m++) {
      const double v = tsrc[tstride * i + m];
      mn[m] = v < mn[m] ? v : mn[m];
      mx[m] = v > mx[m] ? v : mx[m];
    }
  double bs = mx[0] - mn[0];
  if (mx[1] - mn[1] > bs) bs = mx[1] - mn[1];
  if (mx[2] - mn[2] > bs) bs = mx[2] - mn[2];
  P->thresh = std::ldexp(1.0, -51) * bs;
  // largest FP32 phase |k| r / (2 pi) over the box diagonal: the hardware sine takes up to
  // 256 revolutions; beyond 200 the FP32 far sum reduces the phase first
  const double diag = std::sqrt((mx[0] - mn[0]) * (mx[0] - mn[0]) + (mx[1] - mn[1]) * (mx[1] - mn[1]) +
                                (mx[2] - mn[2]) * (mx[2] - mn[2]));
  P->phase_small = !in.helm || std::fabs(in.zk[0]) * diag * 0.15915494309189533577 < 200.0;
  // FP32 coordinates in wavelengths where the phase is r itself (KIND 1); units so long or so
  // short, or surfaces so small against the wavelength, that FP32 powers of r could leave its
  // range keep the caller's (KIND 2)
  const double rev = in.zk[0] * 0.15915494309189533577;
  P->wave32 = in.helm && in.zk[1] == 0.0 && P->phase_small && rev > 1e-6 && rev < 1e6 && rev * diag > 1e-6;
  P->unit32 = P->wave32 ? rev : 1.0;
  // the FP64 kernel evaluations take sin/cos of k r for |k r| <= SINCOS_RED_MAX
  if (in.helm && std::fabs(in.zk[0]) * diag > SINCOS_RED_MAX) {
    fprintf(stderr, "fmm3dbie_amd: |Re k| x surface diameter = %g exceeds %g\n", std::fabs(in.zk[0]) * diag,
            SINCOS_RED_MAX);
    return -6;
  }

  P->ixyzs = own<int64_t>(P, npat + 1);
  P->ixyzso = own<int64_t>(P, npat + 1);
  P->row_ptr = own<int64_t>(P, N + 1);
  P->col_ind = own<int64_t>(P, in.nnz);
  P->iquad = own<int64_t>(P, in.nnz + 1);
  P->ioff = own<int64_t>(P, npat);
  P->np_of = own<int>(P, npat);
  P->opatch = own<int>(P, NO);
  P->near_sorted = own<int>(P, in.nnz);
  P->csr_src = own<int>(P, in.nnz);
  std::vector<int> csr_src(in.nnz);
  for (int64_t j = 0; j < in.nnz; j++) csr_src[j] = (int)(in.ixyzs[in.col_ind[j] - 1] - 1);
  P->imat = own<double>(P, imat_all.size());
  P->wover = own<double>(P, NO);
  P->wover32 = own<float>(P, NO);
  P->geo64 = own<double>(P, GEO<double> * NO);
  P->geo32 = own<float>(P, GEO<float> * NO);
  for (int c = 0; c < 3; c++) {
    P->trg64[c] = own<double>(P, N);
    P->trg32[c] = own<float>(P, N);
  }
  const int64_t nq = in.nquad;
  P->nquad = nq;
  P->wnear64 = own<double>(P, 2 * nq);
  P->wnear32 = own<float>(P, 2 * nq);
  double* d_srcover = dal<double>(12 * NO);
  double* d_srcvals = dal<double>(tstride * N);
  if (!d_srcover || !d_srcvals || !P->wnear32 || !P->wnear64) return -2;
  ACHK(hipMemcpyAsync(P->ixyzs, in.ixyzs, 8 * (npat + 1), hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->ixyzso, in.ixyzso, 8 * (npat + 1), hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->row_ptr, in.row_ptr, 8 * (N + 1), hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->col_ind, in.col_ind, 8 * in.nnz, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->iquad, in.iquad, 8 * (in.nnz + 1), hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->ioff, ioff.data(), 8 * npat, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->np_of, np_of.data(), 4 * npat, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->opatch, opatch.data(), 4 * NO, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->near_sorted, nsorted.data(), 4 * in.nnz, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->csr_src, csr_src.data(), 4 * in.nnz, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->imat, imat_all.data(), 8 * imat_all.size(), hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(P->wover, in.whtsover, 8 * NO, hipMemcpyHostToDevice, s));
  ACHK(hipMemcpyAsync(d_srcover, in.srcover, 8 * 12 * NO, hipMemcpyHostToDevice, s));
  if (N > 0) ACHK(hipMemcpyAsync(d_srcvals, tsrc, 8 * tstride * N, hipMemcpyHostToDevice, s));
  if (nq == 0) {
    // no near pairs: nothing to copy
  } else if (in.wnear_is_device) {
    if (in.helm) {
      ACHK(hipMemcpyAsync(P->wnear64, in.wnear, 16 * nq, hipMemcpyDeviceToDevice, s));
    } else {
      k_real_to_cplx<<<nblk(nq, 256), 256, 0, s>>>(nq, in.wnear, (V2<double>*)P->wnear64);
    }
  } else if (in.helm) {
    ACHK(hipMemcpyAsync(P->wnear64, in.wnear, 16 * nq, hipMemcpyHostToDevice, s));
  } else {
    double* tmp = dal<double>(nq);
    if (!tmp) return -2;
    ACHK(hipMemcpyAsync(tmp, in.wnear, 8 * nq, hipMemcpyHostToDevice, s));
    k_real_to_cplx<<<nblk(nq, 256), 256, 0, s>>>(nq, tmp, (V2<double>*)P->wnear64);
    ACHK(hipStreamSynchronize(s));
    (void)hipFree(tmp);
  }
  if (nq > 0) k_convert<double, float><<<nblk(2 * nq, 256), 256, 0, s>>>(2 * nq, P->wnear64, P->wnear32);
  if (NO > 0) k_geo<<<nblk(NO, 256), 256, 0, s>>>(NO, d_srcover, P->far_ns, P->unit32, P->geo64, P->geo32);
  if (N > 0)
    k_split_targ<<<nblk(N, 256), 256, 0, s>>>(N, d_srcvals, tstride, P->unit32,
                                              Targets{{P->trg64[0], P->trg64[1], P->trg64[2]},
                                                      {P->trg32[0], P->trg32[1], P->trg32[2]}});
  if (NO > 0) k_convert<double, float><<<nblk(NO, 256), 256, 0, s>>>(NO, P->wover, P->wover32);
  ACHK(hipGetLastError());
  ACHK(hipStreamSynchronize(s));
  (void)hipFree(d_srcover);
  (void)hipFree(d_srcvals);
  P->ws_cap = 0;
  return 0;
}

// Right-hand sides in whole groups of grp
static int padded_rhs(int nrhs, int grp) { return (nrhs + grp - 1) / grp * grp; }
// ... and the most that a block of nrhs takes with any group
static int padded_rhs(int nrhs) { return nrhs == 1 ? 1 : padded_rhs(nrhs, MG); }

static int ensure_ws(ApplyPlan* P, int nrhs) {
  if (P->ws_cap >= nrhs) return 0;
  apply_plan_free_ws(P);
  const size_t ns = (size_t)P->nptso * padded_rhs(nrhs);
  P->str64 = dal<double>(2 * ns);
  P->str32 = dal<float>(2 * ns + bmax_values(P->nptso, padded_rhs(nrhs)));
  P->sig64c = dal<double>(2 * (size_t)P->npts);
  P->pot64c = dal<double>(2 * (size_t)P->ntarg);
  // partial far sums: nsplit x nrhs x npts with nsplit x nrhs <= far_split_cap x 64
  const size_t npart = (size_t)P->far_split_cap * 64 * P->ntarg;
  P->part64 = dal<double>(2 * npart);
  P->part32 = dal<float>(2 * npart);
  if (!P->str64 || !P->str32 || !P->sig64c || !P->pot64c || !P->part64 || !P->part32) return -2;
  P->ws_cap = nrhs;
  return 0;
}

void apply_plan_free_ws(ApplyPlan* P) {
  void* ps[] = {P->str64, P->sig64c, P->pot64c, P->part64, P->str32, P->part32};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  P->str64 = P->sig64c = P->pot64c = P->part64 = nullptr;
  P->str32 = P->part32 = nullptr;
  P->ws_cap = 0;
}

template <typename T>
static FarPar<T> far_par(const ApplyPlan* P) {
  const double zr = P->helm ? P->zk[0] : 0.0, zi = P->helm ? P->zk[1] : 0.0;
  FarPar<T> F;
  F.ar = (T)P->far_a[0];
  F.ai = (T)P->far_a[1];
  F.kr = (T)zr;
  F.ki = (T)zi;
  if constexpr (sizeof(T) == 8) {
    double hi, lo;
    half_turns(zr, hi, lo);
    F.khi = hi;
    F.klo = lo;
  } else {
    F.khi = (T)(zr * 0.15915494309189533577);  // k / (2 pi)
    F.klo = (T)0;
    // in wavelengths 1 / r is over the unit, so that a + t (1 - ikr) takes it (k_geo: t's part)
    F.ar = (T)(P->far_a[0] * P->unit32);
    F.ai = (T)(P->far_a[1] * P->unit32);
    if (P->wave32) F.kr = (T)6.283185307179586;
  }
  return F;
}

// Kernel form (FarPar's KIND) of a plan in precision T
template <typename T>
static int far_kind(const ApplyPlan* P) {
  if (!P->helm) return 0;
  return P->zk[1] != 0.0 || (sizeof(T) == 4 && !P->wave32) ? 2 : 1;
}

template <typename T>
static const T* const* targets_of(const ApplyPlan* P) {
  if constexpr (sizeof(T) == 8) return (const T* const*)P->trg64;
  else return (const T* const*)P->trg32;
}
template <typename T>
static const T* sources_of(const ApplyPlan* P) {
  if constexpr (sizeof(T) == 8) return P->geo64;
  else return P->geo32;
}

// Source splits and sources per split (a multiple of tile) of a far sum whose launch has g
// workgroups per split: up to wg_target workgroups, within the partial buffer, and no
// split below 256 sources (its partial sums would cost more than the balance gains)
// unless the launch would leave slots empty (fewer than `fill` workgroups).
static int64_t split_sources(int64_t nsrc, int tile, int64_t g, int64_t wg_target, int64_t fill, int64_t cap,
                             int64_t* chunk) {
  const int64_t ntiles = (nsrc + tile - 1) / tile;
  int64_t nsplit = (wg_target + g - 1) / g;
  const int64_t need = (fill + g - 1) / g;
  nsplit = std::min(nsplit, std::max((nsrc + 255) / 256, need));
  nsplit = std::max<int64_t>(1, std::min({nsplit, cap, ntiles, (int64_t)65535}));  // (grid y)
  *chunk = ((ntiles + nsplit - 1) / nsplit) * tile;
  return (nsrc + *chunk - 1) / *chunk;
}

// Far sum of nrhs right-hand sides in groups of NRHS (grid z).
template <typename T, int NRHS>
static int launch_far(ApplyPlan* P, bool mask, int64_t wg_target, const V2<T>* str, int nrhs, V2<T>* part,
                      int64_t part_cap, int64_t* nsplit_out, hipStream_t s) {
  const T* const* trg = targets_of<T>(P);
  const unsigned g = nblk(P->ntarg, 64);
  const int ngrp = (nrhs + NRHS - 1) / NRHS;
  int64_t chunk;
  const int64_t nsplit = split_sources(P->nptso, STILE, (int64_t)g * ngrp, 4 * wg_target, FAR_FILL,
                                       part_cap / ((int64_t)nrhs * P->ntarg), &chunk);
  const dim3 grid(g, (unsigned)nsplit, (unsigned)ngrp);
  const T th2 = (T)(P->thresh * P->thresh);
#define FMM_FAR(MK, ...)                                                                                    \
  k_farsum<T, MK, __VA_ARGS__><<<grid, 64, 0, s>>>((int)P->ntarg, trg[0], trg[1], trg[2], (int)P->nptso,    \
                                                   sources_of<T>(P), P->ixyzso, str, P->row_ptr, P->near_sorted, \
                                                   far_par<T>(P), th2, (int)chunk, nrhs, part,              \
                                                   (int64_t)nrhs * P->ntarg)
  const int kind = far_kind<T>(P);
  const bool value = NRHS == 1 && sizeof(T) == 4 && (P->unit32 < 1.0 / UNIT32_MILD || P->unit32 > UNIT32_MILD);
  if (mask || sizeof(T) == 4) {
    if (kind == 0) FMM_FAR(true, 0, NRHS);
    else if (kind == 2) FMM_FAR(true, 2, NRHS);
    else if (!value) FMM_FAR(true, 1, NRHS);
    else if constexpr (NRHS == 1 && sizeof(T) == 4) FMM_FAR(true, 1, 1, true);
  } else if constexpr (sizeof(T) == 8) {
    if (kind == 0) FMM_FAR(false, 0, NRHS);
    else if (kind == 1) FMM_FAR(false, 1, NRHS);
    else FMM_FAR(false, 2, NRHS);
  }
#undef FMM_FAR
  *nsplit_out = nsplit;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The matrix-core far sums: groups of 16 right-hand sides, the last one padded with zeros.
// FP64: a group per workgroup (grid z).
static int launch_far_mfma(ApplyPlan* P, bool mask, int64_t wg_target, const V2<double>* str, int nrhs,
                           V2<double>* part, int64_t part_cap, int64_t* nsplit_out, hipStream_t s) {
  const double* const* trg = targets_of<double>(P);
  const unsigned g = nblk(P->ntarg, 16 * FW * MT);
  const int ngrp = (nrhs + MG - 1) / MG;
  int64_t chunk;
  const int64_t nsplit = split_sources(P->nptso, FT, (int64_t)g * ngrp, wg_target, FAR_FILL / FW,
                                       part_cap / ((int64_t)nrhs * P->ntarg), &chunk);
  const dim3 grid(g, (unsigned)nsplit, (unsigned)ngrp);
  const int kind = far_kind<double>(P);
#define FMM_FARM(MK, KD)                                                                                         \
  k_farsum_mfma<MK, KD><<<grid, 64 * FW, 0, s>>>((int)P->ntarg, trg[0], trg[1], trg[2], (int)P->nptso, P->geo64, \
                                                 P->ixyzso, str, P->row_ptr, P->near_sorted, far_par<double>(P), \
                                                 P->thresh * P->thresh, (int)chunk, nrhs, part,                  \
                                                 (int64_t)nrhs * P->ntarg)
  if (mask) {
    if (kind == 0) FMM_FARM(true, 0);
    else if (kind == 1) FMM_FARM(true, 1);
    else FMM_FARM(true, 2);
  } else {
    if (kind == 0) FMM_FARM(false, 0);
    else if (kind == 1) FMM_FARM(false, 1);
    else FMM_FARM(false, 2);
  }
#undef FMM_FARM
  *nsplit_out = nsplit;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// FP32: all groups (at most four) in each workgroup.
static int launch_far_split(ApplyPlan* P, int64_t wg_target, const V2<float>* str, int nrhs, V2<float>* part,
                            int64_t part_cap, int64_t* nsplit_out, hipStream_t s) {
  const float* const* trg = targets_of<float>(P);
  const unsigned g = nblk(P->ntarg, 16 * FW * MT);
  const int ng = (nrhs + MG - 1) / MG;
  int64_t chunk;
  const int64_t nsplit = split_sources(P->nptso, FT, g, wg_target, FAR_FILL / FW,
                                       part_cap / ((int64_t)nrhs * P->ntarg), &chunk);
  const dim3 grid(g, (unsigned)nsplit);
  const int kind = far_kind<float>(P);
  const float* bmax = (const float*)(str + P->nptso * padded_rhs(nrhs, MG));  // as in oversample
#define FMM_FARS(KD, NG)                                                                                          \
  k_farsum_split<KD, NG><<<grid, 64 * FW, 0, s>>>(                                                             \
      (int)P->ntarg, trg[0], trg[1], trg[2], (int)P->nptso, P->geo32, P->ixyzso, str,                          \
      bmax, P->row_ptr, P->near_sorted, far_par<float>(P), (int)chunk, nrhs, part,                              \
      (int64_t)nrhs * P->ntarg)
#define FMM_FARK(NG)                     \
  do {                                   \
    if (kind == 0) FMM_FARS(0, NG);      \
    else if (kind == 1) FMM_FARS(1, NG); \
    else FMM_FARS(2, NG);                \
  } while (0)
  if (ng == 1) FMM_FARK(1);
  else if (ng == 2) FMM_FARK(2);
  else if (ng == 3) FMM_FARK(3);
  else if (ng == 4) FMM_FARK(4);
  else return -6;
#undef FMM_FARK
#undef FMM_FARS
  *nsplit_out = nsplit;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Right-hand sides per far-sum group by default: the smallest of 1, 2, 4, 8 that holds the
// block, and 16 (matrix cores) beyond.
static int default_group(int nrhs) {
  int grp = 1;
  while (grp < nrhs && grp < MG) grp *= 2;
  return grp;
}

// Right-hand sides per far-sum group, tuned or default; a last group is padded with zeros.  Measured
// in cycles of a SIMD per 64 pairs (43008 x 69120 pairs, Helmholtz): FP64 268 / 289 / 325 / 409
// for 1, 2, 4 and 8 densities and 528 for each 16 (a group of 8 is the cheaper one for 5 to 8
// densities, and two of them, 818, the dearer for 9 to 16); FP32 93 / 107 / 140 / 208 and 190 for 16,
// 401 for 64.  Laplace: FP64 117 / 118 / 145 / 203 and 257; FP32 65 / 71 / 82 / 121 and 114, 262.
// str_cap: strengths
// (complex values) that fit the buffer of the call; a padded block that does not falls back
// to a group that divides nrhs.
static int far_group(const ApplyPlan* P, int nrhs, int prec, int64_t str_cap, int64_t* wg) {
  const auto it = P->tuned.find(prec * 1000 + nrhs);
  *wg = it != P->tuned.end() ? it->second.second : P->far_wg_target;
  int grp = it != P->tuned.end() ? it->second.first : default_group(nrhs);
  auto need = [&](int g) {
    const int nr = padded_rhs(nrhs, g);
    return P->nptso * nr + (prec == 32 && g == MG ? (bmax_values(P->nptso, nr) + 1) / 2 : 0);
  };
  while (need(grp) > str_cap) {
    grp /= 2;
    while (nrhs % grp != 0) grp /= 2;
  }
  return grp;
}

template <typename T>
static int dispatch_far(ApplyPlan* P, bool mask, int grp, int64_t wg, const V2<T>* str, int nrhs, V2<T>* part,
                        int64_t part_cap, int64_t* nsplit, hipStream_t s) {
  switch (grp) {
    case 1: return launch_far<T, 1>(P, mask, wg, str, nrhs, part, part_cap, nsplit, s);
    case 2: return launch_far<T, 2>(P, mask, wg, str, nrhs, part, part_cap, nsplit, s);
    case 4: return launch_far<T, 4>(P, mask, wg, str, nrhs, part, part_cap, nsplit, s);
    case 8: return launch_far<T, 8>(P, mask, wg, str, nrhs, part, part_cap, nsplit, s);
    case MG:
      if constexpr (sizeof(T) == 8) return launch_far_mfma(P, mask, wg, str, nrhs, part, part_cap, nsplit, s);
      else return launch_far_split(P, wg, str, nrhs, part, part_cap, nsplit, s);
    default: return -6;
  }
}

// pot = far (+ CSR, and with sub the near subtraction) for all right-hand sides
template <typename T>
static int far_and_csr(ApplyPlan* P, bool mask, bool sub, int grp, int64_t wg, const V2<T>* str, const V2<T>* sg,
                       V2<T>* pt, int nrhs, V2<T>* part, int64_t part_cap, hipStream_t s, hipEvent_t ev_far) {
  const int64_t N = P->ntarg, NO = P->nptso, NS = P->npts;
  const V2<T>* wn = (const V2<T>*)(sizeof(T) == 8 ? (void*)P->wnear64 : (void*)P->wnear32);
  int64_t nsplit = 0;
  if (N == 0) return 0;
  if (NO > 0) {
    const int rc = dispatch_far<T>(P, mask, grp, wg, str, nrhs, part, part_cap, &nsplit, s);
    if (rc) return rc;
  }
  if (ev_far) ACHK(hipEventRecord(ev_far, s));
  SubArgs S = {};
  if constexpr (sizeof(T) == 8)
    S = {P->trg64[0], P->trg64[1], P->trg64[2], P->geo64, str, NO, grp, P->col_ind, P->ixyzso, far_par<double>(P),
         P->thresh * P->thresh};
  // many source splits: one coalesced pass over the partials first; the partials of one
  // right-hand side of a small problem are summed by the lanes of the CSR kernel instead
  // (a launch less; their strided reads stay in L2)
  if (nsplit > 4 && !(nrhs == 1 && P->uniform_p > 0 && nsplit * N <= SPLIT_INLINE)) {
    k_split_sum<T><<<dim3((unsigned)((N + 63) / 64), (unsigned)nrhs), 256, 0, s>>>(N, (int)nsplit, part,
                                                                                  (int64_t)nrhs * N);
    nsplit = 1;
  }
  if (P->uniform_p > 0) {
#define FMM_CSR1(RB, PC, SB)                                                                                    \
  k_reduce_csr<T, T, RB, PC, SB><<<nblk(N, 4), 256, 0, s>>>(N, nrhs, (int)nsplit, part, (int64_t)nrhs * N,       \
                                                            P->row_ptr, P->csr_src, P->iquad, P->uniform_p, wn, \
                                                            sg, NS, pt, N, S)
#define FMM_CSR(PC)                                        \
  do {                                                     \
    if constexpr (sizeof(T) == 8) {                        \
      if (sub) {                                           \
        if (nrhs == 1) FMM_CSR1(1, PC, true);              \
        else FMM_CSR1(8, PC, true);                        \
        break;                                             \
      }                                                    \
    }                                                      \
    if (nrhs == 1) FMM_CSR1(1, PC, false);                 \
    else FMM_CSR1(8, PC, false);                           \
  } while (0)
    switch (P->uniform_p) {
      case 3: FMM_CSR(3); break;
      case 6: FMM_CSR(6); break;
      case 10: FMM_CSR(10); break;
      case 15: FMM_CSR(15); break;
      case 21: FMM_CSR(21); break;
      case 28: FMM_CSR(28); break;
      case 36: FMM_CSR(36); break;
      case 45: FMM_CSR(45); break;
      case 55: FMM_CSR(55); break;
      case 66: FMM_CSR(66); break;
      default: FMM_CSR(0);
    }
#undef FMM_CSR
#undef FMM_CSR1
  } else {
    if (nsplit > 0)
      k_farsum_reduce<T><<<dim3(nblk(N, 256), nrhs), 256, 0, s>>>(N, nrhs, (int)nsplit, part, (int64_t)nrhs * N, pt,
                                                                  N);
    else
      k_fill<T><<<nblk(2 * N * nrhs, 256), 256, 0, s>>>(2 * N * nrhs, (T*)pt, (T)0);
    k_csr_gen<T, T><<<nblk(N, 256), 256, 0, s>>>(N, P->row_ptr, P->col_ind, P->iquad, P->ixyzs, wn, sg, NS, nrhs,
                                                 pt, N);
    if constexpr (sizeof(T) == 8)
      if (sub) k_near_sub<<<nblk(N, 4), 256, 0, s>>>(N, P->row_ptr, S, nrhs, pt, N);
  }
  ACHK(hipGetLastError());
  return 0;
}

// Work buffers of one apply in the precision of the call: strengths at the oversampled nodes
// (str_cap complex values, at least nptso x nrhs) and the far-sum partials (part_cap complex
// values, at least ntarg x nrhs: one source split).
struct ApplyWs {
  void *str, *part;
  int64_t str_cap, part_cap;
};

template <typename T>
static void oversample(ApplyPlan* P, const V2<T>* sigma, int nrhs, int grp, V2<T>* str, hipStream_t s) {
  const int64_t NO = P->nptso;
  const int nr = padded_rhs(nrhs, grp);
  const T* wover;
  if constexpr (sizeof(T) == 8) wover = P->wover;
  else wover = P->wover32;
  float* bmax = nullptr;
  if constexpr (sizeof(T) == 4)
    if (grp == MG) bmax = (float*)(str + NO * nr);  // for k_farsum_split, behind the strengths
#define FMM_OVER(RB)                                                                                             \
  k_oversample<T, RB><<<dim3(nblk(NO, 256), (unsigned)(nr / RB)), 256, 0, s>>>(                                  \
      NO, P->opatch, P->ixyzs, P->ixyzso, P->ioff, P->np_of, P->imat, sigma, nrhs, P->npts, wover,               \
      P->far_phase[0], P->far_phase[1], grp, str, bmax)
  if (grp % 4 == 0) FMM_OVER(4);
  else if (grp == 2) FMM_OVER(2);
  else FMM_OVER(1);
#undef FMM_OVER
}

// sigma/pot: complex (interleaved) device arrays of length npts * nrhs, leading dim npts
template <typename T>
static int apply_run_t(ApplyPlan* P, bool mask, const void* sigma, void* pot, int nrhs, hipStream_t s,
                       const ApplyWs& W, hipEvent_t* ev) {
  int64_t wg;
  const int grp = far_group(P, nrhs, sizeof(T) * 8, W.str_cap, &wg);
  if (P->nptso > 0) oversample<T>(P, (const V2<T>*)sigma, nrhs, grp, (V2<T>*)W.str, s);
  if (ev) ACHK(hipEventRecord(ev[1], s));
  return far_and_csr<T>(P, mask, !mask, grp, wg, (const V2<T>*)W.str, (const V2<T>*)sigma, (V2<T>*)pot, nrhs,
                        (V2<T>*)W.part, W.part_cap, s, ev ? ev[2] : nullptr);
}

static int apply_run_ws(ApplyPlan* P, int prec, int mode, const void* sigma, void* pot, int nrhs, hipStream_t s,
                        ApplyTimes* tm, const ApplyWs& W) {
  hipEvent_t ev[4];
  if (tm)
    for (auto& e : ev) ACHK(hipEventCreate(&e));
  if (tm) ACHK(hipEventRecord(ev[0], s));
  const int rc = prec == 64 ? apply_run_t<double>(P, mode == APPLY_MASKED, sigma, pot, nrhs, s, W, tm ? ev : nullptr)
                            : apply_run_t<float>(P, true, sigma, pot, nrhs, s, W, tm ? ev : nullptr);
  if (tm) ACHK(hipEventRecord(ev[3], s));
  if (rc) return rc;
  ACHK(hipGetLastError());
  if (tm) {
    ACHK(hipEventSynchronize(ev[3]));
    float ms;
    (void)hipEventElapsedTime(&ms, ev[0], ev[1]); tm->ms_over = ms;
    (void)hipEventElapsedTime(&ms, ev[1], ev[2]); tm->ms_far = ms;
    (void)hipEventElapsedTime(&ms, ev[2], ev[3]); tm->ms_csr = ms;
    tm->ms_sub = 0.0;  // within ms_csr: one kernel
    for (auto& e : ev) (void)hipEventDestroy(e);
  }
  return 0;
}

static int check_prec_nrhs(int prec, int nrhs) {
  if (nrhs < 1 || nrhs > 64) return -6;
  if (prec != 32 && prec != 64) {
    fprintf(stderr, "fmm3dbie_amd: apply precision %d (must be 32 or 64)\n", prec);
    return -6;
  }
  return 0;
}

static ApplyWs plan_ws(const ApplyPlan* P, int prec) {
  const int nr = padded_rhs(P->ws_cap);
  const int64_t cap = (int64_t)P->far_split_cap * 64 * P->ntarg, str = P->nptso * nr;
  if (prec == 64) return {P->str64, P->part64, str, cap};
  return {P->str32, P->part32, str + (bmax_values(P->nptso, nr) + 1) / 2, cap};
}

// sigma/pot: complex (interleaved) device arrays of length npts * nrhs, leading dim npts;
// work buffers owned by the plan (allocated on the first call that needs them)
int apply_plan_run(ApplyPlan* P, int prec, int mode, const void* sigma, void* pot, int nrhs, hipStream_t s,
                   ApplyTimes* tm) {
  const int rc = check_prec_nrhs(prec, nrhs);
  if (rc) return rc;
  if (ensure_ws(P, nrhs) != 0) return -2;
  return apply_run_ws(P, prec, mode, sigma, pot, nrhs, s, tm, plan_ws(P, prec));
}

// ------------------------------------------------------------------ allocation-free apply
// The work buffers of apply_plan_run_noalloc live in this file-scope device array, one
// copy per GPU, held until the process ends.  Host code never passes `scratch` itself to
// a kernel (on the host the name is only a stand-in): it uses the device address that
// hipGetSymbolAddress returns, looked up once per device.
constexpr size_t APPLY_SCRATCH_BYTES = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[APPLY_SCRATCH_BYTES];

static std::mutex g_scratch_mutex;
static std::map<int, void*> g_scratch_ptr;  // device -> address of its copy of `scratch`

static void* scratch_address() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  auto it = g_scratch_ptr.find(dev);
  if (it != g_scratch_ptr.end()) return it->second;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    fprintf(stderr, "fmm3dbie_amd: hipGetSymbolAddress(scratch) failed: %s\n", hipGetErrorString(e));
    return nullptr;
  }
  g_scratch_ptr[dev] = ptr;
  return ptr;
}

size_t apply_scratch_bytes() { return APPLY_SCRATCH_BYTES; }

int apply_plan_run_noalloc(ApplyPlan* P, int prec, int mode, const void* sigma, void* pot, int nrhs, hipStream_t s) {
  int rc = check_prec_nrhs(prec, nrhs);
  if (rc) return rc;
  const size_t cs = prec == 64 ? 2 * sizeof(double) : 2 * sizeof(float);  // one complex value
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t strength = up(cs * (size_t)(P->nptso > 0 ? P->nptso : 1) * nrhs);
  const size_t one_split = cs * (size_t)(P->ntarg > 0 ? P->ntarg : 1) * nrhs;
  if (2 * strength + one_split > APPLY_SCRATCH_BYTES) {
    fprintf(stderr,
            "fmm3dbie_amd: allocation-free apply: %zu bytes of work buffers needed (nptso %lld, targets %lld, "
            "nrhs %d, prec %d), the fixed scratch holds %zu\n",
            2 * strength + one_split, (long long)P->nptso, (long long)P->ntarg, nrhs, prec, APPLY_SCRATCH_BYTES);
    return -7;
  }
  unsigned char* base = (unsigned char*)scratch_address();
  if (!base) return -1;
  // strengths in the first two blocks, partials in the rest
  ApplyWs W;
  W.str = base;
  W.str_cap = (int64_t)(2 * strength / cs);
  W.part = base + 2 * strength;
  W.part_cap = (int64_t)((APPLY_SCRATCH_BYTES - 2 * strength) / cs);
  return apply_run_ws(P, prec, mode, sigma, pot, nrhs, s, nullptr, W);
}

// Autotuner of the far-sum launch shape for (prec, nrhs): every right-hand-side group size
// from 1 to the default one, which pads the last group (FP64 blocks of 16 and more leave out
// the group of one, 16 times the kernel values of the matrix cores), and workgroup targets of
// 4096, 8192, 16384, 32768 are timed (one warm-up launch, then one launch each) on unit
// densities; the fastest is kept in the plan and used by every later apply with the same
// (prec, nrhs).
int apply_plan_tune(ApplyPlan* P, int prec, int nrhs, hipStream_t s, double* report, int nreport) {
  if (nrhs < 1 || nrhs > 64 || (prec != 32 && prec != 64)) return -6;
  if (ensure_ws(P, nrhs) != 0) return -2;
  if (P->ntarg == 0 || P->nptso == 0) return 0;
  const int64_t nval = 2 * P->nptso * padded_rhs(nrhs), nmax = bmax_values(P->nptso, padded_rhs(nrhs));
  if (prec == 64) k_fill<double><<<nblk(nval, 256), 256, 0, s>>>(nval, P->str64, 1.0);
  else k_fill<float><<<nblk(nval + nmax, 256), 256, 0, s>>>(nval + nmax, P->str32, 1.0f);
  auto far = [&](int gsz, int64_t wg) {
    int64_t nsplit;
    const int64_t cap = (int64_t)P->far_split_cap * 64 * P->ntarg;
    return prec == 64 ? dispatch_far<double>(P, true, gsz, wg, (const V2<double>*)P->str64, nrhs,
                                             (V2<double>*)P->part64, cap, &nsplit, s)
                      : dispatch_far<float>(P, true, gsz, wg, (const V2<float>*)P->str32, nrhs,
                                            (V2<float>*)P->part32, cap, &nsplit, s);
  };
  hipEvent_t e0, e1;
  ACHK(hipEventCreate(&e0));
  ACHK(hipEventCreate(&e1));
  const int groups[5] = {1, 2, 4, 8, MG};
  const int64_t wgs[4] = {4096, 8192, 16384, 32768};
  float best = 1e30f;
  int bg = 1, nrep = 0;
  int64_t bw = P->far_wg_target;
  // one warm-up launch, then one timed launch per shape
  int rc = far(default_group(nrhs), P->far_wg_target);
  if (rc) return rc;
  for (int gsz : groups) {
    if (gsz > default_group(nrhs) || (prec == 64 && gsz == 1 && nrhs >= MG)) continue;
    for (int64_t wg : wgs) {
      ACHK(hipEventRecord(e0, s));
      rc = far(gsz, wg);
      if (rc) return rc;
      ACHK(hipEventRecord(e1, s));
      ACHK(hipEventSynchronize(e1));
      float ms;
      (void)hipEventElapsedTime(&ms, e0, e1);
      if (report && nrep + 3 <= nreport) {
        report[nrep++] = gsz;
        report[nrep++] = (double)wg;
        report[nrep++] = ms;
      }
      if (ms < best) {
        best = ms;
        bg = gsz;
        bw = wg;
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  P->tuned[prec * 1000 + nrhs] = {bg, bw};
  return nrep / 3;
}

// real (Laplace) densities: convert to complex, apply, take real part
int apply_plan_run_real(ApplyPlan* P, int mode, const double* sigma, double* pot, hipStream_t s) {
  if (ensure_ws(P, 1) != 0) return -2;
  const int64_t N = P->npts, NT = P->ntarg;
  k_real_to_cplx<<<nblk(N, 256), 256, 0, s>>>(N, sigma, (V2<double>*)P->sig64c);
  int r = apply_plan_run(P, 64, mode, P->sig64c, P->pot64c, 1, s, nullptr);
  if (r) return r;
  if (NT > 0) k_cplx_to_real<<<nblk(NT, 256), 256, 0, s>>>(NT, (const V2<double>*)P->pot64c, pot);
  ACHK(hipGetLastError());
  return 0;
}
