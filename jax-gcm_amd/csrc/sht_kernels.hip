// Dynamics <-> physics transforms for gfx950: spherical-harmonic analysis and
// synthesis on a Gaussian grid, fp32 matrix instructions over l or latitude and
// short FFTs over longitude, with the unit conversions, the modal
// vorticity/divergence <-> wind operators and the hydrostatic geopotential fused
// into them: two launches a conversion.
//
// Reference behaviour: jcm/physics_interface.py:196-303 over dinosaur's
// RealSphericalHarmonics (Grid.T<N>, jcm/utils.py:28-54).
//
// Data flow of one conversion (B stacked fields, modes Mm = 2*n_m-1):
//   to_nodal:  modal [B][Mm][L] --Legendre--> Y [B][n_m][nlat] --Fourier--> nodal [B][nlon][nlat]
//   to_modal:  nodal [B][nlon][nlat] --Fourier--> Y [B][n_m][nlat] --Legendre--> modal [B][Mm][L]
// with Y a float2 of the cosine and the sine mode.  The modal operators run on the
// Legendre kernels' rows; per-field pre/post operations (1/cos(lat), unit scales,
// reference temperature, log/exp of surface pressure) ride in the Fourier kernels'
// loads and stores.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "speedy_sht.h"

struct SpeedyShtPlan {
  int32_t n_m, n_l, nlon, nlat, mm;   // mm = 2*n_m-1 modes
  double radius;
  int device;
  int32_t n1, n2;      // nlon = n1 * n2 (the Fourier stages' two passes)
  int32_t tl_a, tl_s;  // latitudes per workgroup of the Fourier analysis / synthesis
  float* Ps;    // Legendre operand blocks of the synthesis
  float* Pa;    // and of the analysis (LegendreArgs says how they are laid out)
  int32_t* blk; // [n_m] first block of order m
  float* sec;   // [nlat] 1 / cos(lat)
  float* tw;    // [2][nlon]: cos(2 pi j / nlon), -sin(2 pi j / nlon)
};

namespace sht {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

constexpr int kThreads = 256;
constexpr int kMaxSeg = 8;

enum : int32_t { kOpLog = 1, kOpExp = 2, kOpSecLat = 4, kOpSubLevel = 8, kOpAddLevel = 16 };

// A run of stacked fields that share a source (Fourier analysis) or a
// destination (Fourier synthesis) and one operation.
struct Seg {
  const float* src;
  float* dst;
  const float* level;   // per-field constant, index (f - first) % period, or null
  int32_t first, count, period, op;
  float mul;
};
struct SegTable {
  Seg s[kMaxSeg];
  int32_t n;
};

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int find_seg(const SegTable& t, int f) {
  int k = 0;
  for (int i = 1; i < t.n; ++i)
    if (f >= t.s[i].first) k = i;
  return k;
}

// eps(m, l) = sqrt((l^2 - m^2) / (4 l^2 - 1)) for m <= l, l >= 1; else 0:
// x P_l^m = eps(m, l+1) P_{l+1}^m + eps(m, l) P_{l-1}^m (unit-norm functions).
__device__ __forceinline__ float eps_ml(int m, int l) {
  if (l <= 0 || m > l) return 0.0f;
  const float fl = (float)l, fm = (float)m;
  return sqrtf((fl * fl - fm * fm) / (4.0f * fl * fl - 1.0f));
}

// Modal coefficient (mode 0, l 0) of the constant 1: 1 / (F_0 P_0^0) = 2 sqrt(pi).
constexpr float kConstCoef = 3.5449077018110318f;

// ------------------------------------------------------------ Legendre stages
// One workgroup takes one order m and eight fields: 16 rows, the cosine and the sine
// mode of each (row 2 f and 2 f + 1; m = 0 has no sine mode and its rows are zero).
// The modal operators of the conversions couple l with l +- 1 and the cosine with the
// sine mode, both inside the workgroup, so they run on the 16 rows in LDS.
//
// Gaussian latitudes are symmetric and P_l^m(-x) = (-1)^(l+m) P_l^m(x): the l with l+m
// even (parity 0) and odd (parity 1) are separate sums over the southern half of the
// latitudes.  P_l^m is zero for l < m, and those l are not summed: l = m + par + 2 c.
// The operand P is laid out for the matrix instructions: blocks of 16 c x 16 southern
// latitudes j, 1 KiB each, [m][par][c / 16][j / 16], zero outside; lane (g = lane / 16,
// n = lane % 16) reads the 16 bytes it feeds to the four k substeps of a block: q = 0 .. 3
// is c = 4 q + g at j = n (synthesis) or j = 4 g + q at c = n (analysis).  The synthesis
// so sums in ascending l: the terms of a wind's m = 0 cancel from one l to the next at
// the poles, and other orders leave a larger error there.  The Fourier basis's
// 1 / sqrt(2 pi) (m = 0) and 1 / sqrt(pi) are in the analysis's P, with the Gauss weights
// 2 pi w / nlon; the synthesis multiplies its sums by them, and by the 1 / 2 of the
// Fourier stage's Hermitian pairs (in P they made the error at the poles 1.5 times as
// large, by rounding the P of neighbouring l apart).
//
// Bound by the latency of its three dependent steps (modal input, matrix products, Y),
// at T213 too (more or fewer workgroups on a CU, or operand blocks in flight, change
// nothing; the matrix instructions take 5 of 23 us).  Chunks of one order run on one XCD
// (workgroups go round the 8 XCDs), so that P comes into its L2 once.  Before, dense
// batched products per mode and parity over all l >= 0 with the modal operators as a
// kernel of their own: 4.9 + 11.5 us (T85 x 41 fields synthesis) and 7.5 + 3.5 us (T85 x
// 32 fields analysis), now 8.2 and 6.1; T213 x 41 synthesis 14 + 53 us, now 23.
struct LegendreArgs {
  int32_t n_m, nl, nlat, kx;
  int32_t winds, plain, geo;   // levels of winds, other fields, geopotential levels
  int32_t nfield;              // fields of Y: the plain ones past it are zero (analysis)
  int32_t kt;                  // 16-wide tiles of the summed index staged at a time
  const float* P;
  const int32_t* blk;
  float2* y;                   // [field][m][nlat]: cosine and sine mode
  float* z;                    // analysis: [workgroup][16][nl], if not in LDS
  float inv_radius, radius2, gravity;
  const float* vor;            // [kx][mm][nl]
  const float* div;
  float* vor_out;
  float* div_out;
  const float* src[4];         // the plain fields, a run of `count` [mm][nl] each
  float* dst[4];
  int32_t count[4];
  // geopotential: phi_j = g orography + sum_k W[j][k] (T_var_k + reference_k as a constant)
  const float* tvar;
  const float* orography;
  const float* reference;
  float geo_w[SPEEDY_SHT_KX_MAX][SPEEDY_SHT_KX_MAX];
};

enum ChunkKind { kWinds, kPlain, kGeo };
struct Chunk {
  int m, id, kind, f0;   // f0: first level (winds, geo) or field (plain)
};

__host__ __device__ constexpr int chunks(int winds, int plain, int geo) {
  return (winds + 3) / 4 + (plain + 7) / 8 + (geo + 7) / 8;
}

__device__ __forceinline__ Chunk find_chunk(const LegendreArgs& a) {
  const int n = chunks(a.winds, a.plain, a.geo), q = (int)blockIdx.x >> 3;
  Chunk c;
  c.id = q % n;
  c.m = q / n * 8 + ((int)blockIdx.x & 7);
  int k = c.id;
  c.kind = kWinds;
  c.f0 = 4 * k;
  k -= (a.winds + 3) / 4;
  if (k >= 0) {
    c.kind = kPlain;
    c.f0 = 8 * k;
    k -= (a.plain + 7) / 8;
    if (k >= 0) {
      c.kind = kGeo;
      c.f0 = 8 * k;
    }
  }
  return c;
}

// Stacked field of a chunk's slot (0 .. 7), or -1.  The winds of a level are two slots.
__device__ __forceinline__ int slot_field(const LegendreArgs& a, const Chunk& c, int slot) {
  if (c.kind == kWinds) {
    const int k = c.f0 + (slot >> 1);
    return k < a.winds ? (slot & 1) * a.winds + k : -1;
  }
  const int f = c.f0 + slot;
  if (c.kind == kPlain) return f < a.plain ? 2 * a.winds + f : -1;
  return f < a.geo ? 2 * a.winds + a.plain + f : -1;
}

// Run and place in it of plain field f < a.plain.
__device__ __forceinline__ int plain_run(const LegendreArgs& a, int& f) {
  int r = 0;
  for (; r < 3 && f >= a.count[r]; ++r) f -= a.count[r];
  return r;
}

constexpr int lds_row(int kt) { return 16 * kt + 4; }   // 4 mod 64 banks: 16 rows' 16-byte reads cover all banks
// Place of c in its row of the synthesis: the lane group c % 4 reads four in one.
__host__ __device__ constexpr int place(int c) { return (c & ~15) | (c & 3) << 2 | (c >> 2 & 3); }
constexpr int kAhead = 4;                               // operand blocks in flight per parity

__global__ __launch_bounds__(kThreads) void legendre_synthesis_kernel(LegendreArgs a) {
  extern __shared__ __align__(16) float lds[];   // [par][16][ld]
  const Chunk c = find_chunk(a);
  if (c.m >= a.n_m) return;
  const int m = c.m, nl = a.nl, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int h = a.nlat >> 1, jts = (h + 15) >> 4, cts = ((nl - m + 1) / 2 + 15) >> 4;
  const int ld = lds_row(a.kt), par1 = 16 * ld;
  const size_t per = (size_t)(2 * a.n_m - 1) * nl;
  const size_t oc = (size_t)(m == 0 ? 0 : 2 * m - 1) * nl, os = oc + (m == 0 ? 0 : nl);   // cosine, sine rows
  const floatx4* P = reinterpret_cast<const floatx4*>(a.P) + (size_t)a.blk[m] * 64 + lane;
  const float scale = m == 0 ? 0.5f * 0.3989422804014327f : 0.5f * 0.5641895835477563f;

  for (int k0 = 0; k0 < cts; k0 += a.kt) {
    const int k1 = min(k0 + a.kt, cts);
    floatx4 next[2][kAhead];
    auto load = [&](int jt, int ct) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
#pragma unroll
        for (int par = 0; par < 2; ++par)
          next[par][u] = P[(size_t)((par * cts + min(ct + u, k1 - 1)) * jts + jt) * 64];
    };
    if (wave < jts) load(wave, k0);
    if (k0) __syncthreads();
    // the modal rows: coefficient l = m + i at [i & 1][row][place(i / 2)]; loads at clamped l (no
    // condition, so that those of several l are in flight), zero past the last
    if (c.kind == kWinds) {   // (psi, chi) -> (u cos(lat), v cos(lat)), the highest l clipped
      const int k = c.f0 + wave;
      const bool on = k < a.winds;
      const float* z = a.vor + (size_t)(on ? k : 0) * per;
      const float* d = a.div + (size_t)(on ? k : 0) * per;
#pragma unroll 2
      for (int i = 32 * k0 + lane; i < 32 * k1; i += 64) {
        const bool in = on && m + i < nl - 1;
        const int l = min(m + i, nl - 2), lm = max(l - 1, 0);
        auto inv_lap = [&](int ll) { return ll == 0 ? 0.0f : -a.radius2 / ((float)ll * (float)(ll + 1)); };
        const float zc = z[oc + l], zs = z[os + l], dc = d[oc + l], ds = d[os + l];
        const float zcp = z[oc + l + 1], zsp = z[os + l + 1], dcp = d[oc + l + 1], dsp = d[os + l + 1];
        const float zcm = z[oc + lm], zsm = z[os + lm], dcm = d[oc + lm], dsm = d[os + lm];
        // cos(lat) d/dlat at l: (l+2) eps(l+1) x_{l+1} - (l-1) eps(l) x_{l-1}
        const float cp = (float)(l + 2) * eps_ml(m, l + 1) * inv_lap(l + 1);
        const float cm = -(float)(l - 1) * eps_ml(m, l) * inv_lap(lm), il = inv_lap(l), fm = (float)m;
        const float uc = (fm * ds * il - (cp * zcp + cm * zcm)) * a.inv_radius;
        const float vc = (fm * zs * il + (cp * dcp + cm * dcm)) * a.inv_radius;
        const float us = (-fm * dc * il - (cp * zsp + cm * zsm)) * a.inv_radius;
        const float vs = (-fm * zc * il + (cp * dsp + cm * dsm)) * a.inv_radius;
        float* o = lds + (i & 1) * par1 + 4 * wave * ld + place(i >> 1) - 16 * k0;
        o[0] = in ? uc : 0.0f;
        o[ld] = in && m ? us : 0.0f;
        o[2 * ld] = in ? vc : 0.0f;
        o[3 * ld] = in && m ? vs : 0.0f;
      }
    } else if (c.kind == kPlain) {
      const float* x[2];
      bool on[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        int f = c.f0 + 2 * wave + q;
        on[q] = f < a.plain;
        if (!on[q]) f = c.f0;
        const int run = plain_run(a, f);
        x[q] = a.src[run] + (size_t)f * per;
      }
#pragma unroll 4
      for (int i = 32 * k0 + lane; i < 32 * k1; i += 64) {
        const bool in = m + i < nl;
        const int l = min(m + i, nl - 1);
        float* o = lds + (i & 1) * par1 + 4 * wave * ld + place(i >> 1) - 16 * k0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const float xc = x[q][oc + l], xs = x[q][os + l];
          o[2 * q * ld] = in && on[q] ? xc : 0.0f;
          o[(2 * q + 1) * ld] = in && on[q] && m ? xs : 0.0f;
        }
      }
    } else {   // get_geopotential in modal space: waves 0 and 1 take slots 0 .. 3, 2 and 3 the others
      const int sine = wave & 1, s0 = wave & 2 ? 4 : 0;
      for (int i = 32 * k0 + lane; i < 32 * k1; i += 64) {
        const bool in = m + i < nl && (m || !sine);
        const size_t at = (sine ? os : oc) + min(m + i, nl - 1);
        const float g0 = a.gravity * a.orography[at];
        float acc[4] = {g0, g0, g0, g0};
        for (int kb = 0; kb < a.kx; kb += 8) {   // eight levels' loads at a time (past kx: the last, not summed)
          float t[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) t[k] = a.tvar[(size_t)min(kb + k, a.kx - 1) * per + at];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            if (kb + k >= a.kx) break;
            if (at == 0) t[k] += a.reference[kb + k] * kConstCoef;
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += a.geo_w[min(c.f0 + s0 + q, SPEEDY_SHT_KX_MAX - 1)][kb + k] * t[k];
          }
        }
        float* o = lds + (i & 1) * par1 + (2 * s0 + sine) * ld + place(i >> 1) - 16 * k0;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[2 * q * ld] = in ? acc[q] : 0.0f;
      }
    }
    __syncthreads();
    // E|O[row][j] = sum_c X[row][l(par, c)] P[c][j]: a wave takes every fourth latitude tile
    floatx4 acc[2] = {};
    const float* A = lds + r16 * ld + 4 * g - 16 * k0;
    for (int jt = wave, ct = k0; jt < jts;) {
      floatx4 p[2][kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) p[0][u] = next[0][u], p[1][u] = next[1][u];
      const bool last = ct + kAhead >= k1;
      const int jn = last ? jt + 4 : jt, cn = last ? k0 : ct + kAhead;
      if (jn < jts) load(jn, cn);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (ct + u >= k1) break;
#pragma unroll
        for (int par = 0; par < 2; ++par) {
          const floatx4 x = *reinterpret_cast<const floatx4*>(A + par * par1 + 16 * (ct + u));
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[par] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q], p[par][u][q], acc[par], 0, 0, 0);
        }
      }
      if (last) {   // lane holds rows 4 g .. 4 g + 3 (two fields) of latitude 16 jt + r16
        const int j = 16 * jt + r16;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int f = slot_field(a, c, 2 * g + q);
          if (f >= 0 && j < h) {
            float2* y = a.y + ((size_t)f * a.n_m + m) * a.nlat;
            const float ec = acc[0][2 * q], es = acc[0][2 * q + 1], odc = acc[1][2 * q], ods = acc[1][2 * q + 1];
            float2 s = make_float2((ec + odc) * scale, (es + ods) * scale);
            float2 n = make_float2((ec - odc) * scale, (es - ods) * scale);
            if (k0) {
              const float2 s0 = y[j], n0 = y[a.nlat - 1 - j];
              s.x += s0.x; s.y += s0.y;
              n.x += n0.x; n.y += n0.y;
            }
            y[j] = s;
            y[a.nlat - 1 - j] = n;
          }
        }
        acc[0] = acc[1] = floatx4{};
      }
      jt = jn;
      ct = cn;
    }
  }
}

// ZLDS: the 16 modal rows fit in LDS behind the staged ones; else they are in a.z.
template <bool ZLDS>
__global__ __launch_bounds__(kThreads) void legendre_analysis_kernel(LegendreArgs a) {
  extern __shared__ __align__(16) float lds[];   // [par][16][ld], then z[16][nl]
  const Chunk c = find_chunk(a);
  if (c.m >= a.n_m) return;
  const int m = c.m, nl = a.nl, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int h = a.nlat >> 1, jts = (h + 15) >> 4, cts = ((nl - m + 1) / 2 + 15) >> 4;
  const int ld = lds_row(a.kt), par1 = 16 * ld;
  float* z = ZLDS ? lds + 2 * par1 : a.z + ((size_t)c.id * a.n_m + m) * 16 * nl;
  // a wave takes one parity and every second c tile
  const int par = wave & 1;
  const floatx4* P = reinterpret_cast<const floatx4*>(a.P) + ((size_t)a.blk[m] + (size_t)par * cts * jts) * 64 + lane;

  for (int k0 = 0; k0 < jts; k0 += a.kt) {
    const int k1 = min(k0 + a.kt, jts);
    floatx4 next[kAhead];
    auto load = [&](int ct, int jt) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u) next[u] = P[(size_t)(ct * jts + min(jt + u, k1 - 1)) * 64];
    };
    const int ct0 = wave >> 1;
    if (ct0 < cts) load(ct0, k0);
    if (k0) __syncthreads();
    // even and odd halves Y_j +- Y_{nlat-1-j} of both modes
    const float2* y[2];
    bool on[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int f = slot_field(a, c, 2 * wave + q);
      on[q] = f >= 0 && f < a.nfield;
      y[q] = a.y + ((size_t)(on[q] ? f : 0) * a.n_m + m) * a.nlat;
    }
#pragma unroll 2
    for (int j = 16 * k0 + lane; j < 16 * k1; j += 64) {
      const int js = min(j, h - 1), jn = a.nlat - 1 - js;
      float* o = lds + 4 * wave * ld + j - 16 * k0;
#pragma unroll
      for (int q = 0; q < 2; ++q, o += 2 * ld) {
        const float2 s = y[q][js], n = y[q][jn];
        const bool in = on[q] && j < h;
        o[0] = in ? s.x + n.x : 0.0f;
        o[ld] = in ? s.y + n.y : 0.0f;
        o[par1] = in ? s.x - n.x : 0.0f;
        o[par1 + ld] = in ? s.y - n.y : 0.0f;
      }
    }
    __syncthreads();
    floatx4 acc = {};
    const float* A = lds + par * par1 + r16 * ld + 4 * g - 16 * k0;
    for (int ct = ct0, jt = k0; ct < cts;) {
      floatx4 p[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) p[u] = next[u];
      const bool last = jt + kAhead >= k1;
      const int cn = last ? ct + 2 : ct, jn = last ? k0 : jt + kAhead;
      if (cn < cts) load(cn, jn);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (jt + u >= k1) break;
        const floatx4 x = *reinterpret_cast<const floatx4*>(A + 16 * (jt + u));
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q], p[u][q], acc, 0, 0, 0);
      }
      if (last) {   // lane holds rows 4 g .. 4 g + 3 of c = 16 ct + r16
        const int l = m + par + 2 * (16 * ct + r16);
        if (l < nl) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float* o = z + (size_t)(4 * g + q) * nl + l;
            *o = k0 ? *o + acc[q] : acc[q];
          }
        }
        acc = floatx4{};
      }
      ct = cn;
      jt = jn;
    }
  }
  __syncthreads();
  // the coefficients below l = m are zero (not finite where the order's others are not)
  auto at = [&](int row, int l) {
    const float v = z[(size_t)row * nl + max(l, m)];
    return l < m ? v * 0.0f + 0.0f : v;
  };
  const size_t per = (size_t)(2 * a.n_m - 1) * nl;
  const size_t oc = (size_t)(m == 0 ? 0 : 2 * m - 1) * nl, os = oc + nl;
  if (c.kind == kWinds) {
    // (U, V) = (u, v) / cos(lat) -> vorticity and divergence, the highest l clipped:
    // sec(lat) d/dlat cos^2(lat) at l is l eps(l+1) x_{l+1} - (l+1) eps(l) x_{l-1}
    const int k = c.f0 + wave, ru = 4 * wave, rv = ru + 2;
    if (k >= a.winds) return;
    const float fm = (float)m;
    for (int l = lane; l < nl; l += 64) {
      float zc = 0.0f, zs = 0.0f, dc = 0.0f, ds = 0.0f;
      if (l < nl - 1) {
        const int lm = max(l - 1, 0);
        const float cp = (float)l * eps_ml(m, l + 1), cm = -(float)(l + 1) * eps_ml(m, l);
        zc = (fm * at(rv + 1, l) - (cp * at(ru, l + 1) + cm * at(ru, lm))) * a.inv_radius;
        dc = (fm * at(ru + 1, l) + (cp * at(rv, l + 1) + cm * at(rv, lm))) * a.inv_radius;
        zs = (-fm * at(rv, l) - (cp * at(ru + 1, l + 1) + cm * at(ru + 1, lm))) * a.inv_radius;
        ds = (-fm * at(ru, l) + (cp * at(rv + 1, l + 1) + cm * at(rv + 1, lm))) * a.inv_radius;
      }
      a.vor_out[k * per + oc + l] = zc;
      a.div_out[k * per + oc + l] = dc;
      if (m) {
        a.vor_out[k * per + os + l] = zs;
        a.div_out[k * per + os + l] = ds;
      }
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int slot = 2 * wave + q;
    int f = c.f0 + slot;
    if (f >= a.plain) return;
    const int run = plain_run(a, f);
    float* o = a.dst[run] + (size_t)f * per;
    for (int l = lane; l < nl; l += 64) {
      o[oc + l] = at(2 * slot, l);
      if (m) o[os + l] = at(2 * slot + 1, l);
    }
  }
}

// ------------------------------------------------------------ Fourier stages
// The longitude contraction is a real DFT of length N = nlon truncated to the
// n_m lowest wavenumbers, computed in two short passes (Cooley-Tukey with
// N = n1 * n2, longitude i = i1 + n1 * i2, wavenumber k = k2 + n2 * k1):
//   X_k = sum_i1 w^(i1 k) Z[i1][k mod n2],   Z[i1][k2] = sum_i2 x[i1 + n1 i2] w_n2^(i2 k2),
// with w = exp(-2 pi i / N) and w_n2 = w^n1.  Z of a real line is Hermitian in
// k2, so only k2 <= n2 / 2 is formed.  Y holds the cosine and the sine projection of
// order k, Re X_k and -Im X_k; the basis's factors are the Legendre stages'.  Synthesis
// runs the same passes backwards.  A workgroup takes one field and `tl` latitudes
// (latitude fastest, as in memory); the intermediate Z or W and the N roots of unity
// live in LDS, in the generic kernels the line tile too.
struct FourierArgs {
  int32_t nlon, nlat, mm, n_m, n1, n2, tl, nfield;
  const float* twr;     // [nlon] cos(2 pi j / nlon)
  const float* twi;     // [nlon] -sin(2 pi j / nlon)
  const float* sec;     // [nlat]
  float2* y;            // [nfield][n_m][nlat]: cosine and sine mode, without the basis's factors
  SegTable seg;
};

__device__ __forceinline__ void load_roots(const FourierArgs& a, float* twr, float* twi) {
  for (int i = threadIdx.x; i < a.nlon; i += kThreads) {
    twr[i] = a.twr[i];
    twi[i] = a.twi[i];
  }
}

// Y_b[m][lat] = sum_lon (cos, sin)(m lon) prologue(x_b[lon][lat]) for one field b
// (blockIdx.y) and latitudes j0 .. j0 + tl - 1 (blockIdx.x).
__global__ __launch_bounds__(kThreads) void fourier_analysis_generic(FourierArgs a) {
  extern __shared__ float lds[];
  const int N = a.nlon, n1 = a.n1, n2 = a.n2, nh = n2 / 2 + 1, tl = a.tl;
  const int b = blockIdx.y, j0 = blockIdx.x * tl;
  float* twr = lds;
  float* twi = twr + N;
  float* xs = twi + N;            // [N][tl]
  float* zr = xs + N * tl;        // [n1][nh][tl]
  float* zi = zr + n1 * nh * tl;
  const Seg sg = a.seg.s[find_seg(a.seg, b)];
  const float* src = sg.src + (size_t)(b - sg.first) * N * a.nlat;
  const float lvl = sg.level ? sg.level[(b - sg.first) % sg.period] : 0.0f;
  load_roots(a, twr, twi);
  for (int e = threadIdx.x; e < N * tl; e += kThreads) {
    const int lon = e / tl, jj = e - lon * tl, j = j0 + jj;
    float v = 0.0f;
    if (j < a.nlat) {
      v = src[(size_t)lon * a.nlat + j];
      if (sg.op & kOpLog) v = logf(v);
      if (sg.op & kOpSubLevel) v -= lvl;
      v *= sg.mul * ((sg.op & kOpSecLat) ? a.sec[j] : 1.0f);
    }
    xs[e] = v;
  }
  __syncthreads();
  // pass 1: Z[i1][k2] = sum_i2 x[i1 + n1 i2] w^(n1 i2 k2), k2 <= n2 / 2
  for (int e = threadIdx.x; e < n1 * nh * tl; e += kThreads) {
    const int r = e / tl, jj = e - r * tl, k2 = r % nh, i1 = r / nh;
    float re = 0.0f, im = 0.0f;
    int q = 0;   // (i2 * k2) mod n2
    for (int i2 = 0; i2 < n2; ++i2) {
      const float x = xs[(i1 + n1 * i2) * tl + jj];
      re += x * twr[q * n1];
      im += x * twi[q * n1];
      q += k2;
      if (q >= n2) q -= n2;
    }
    zr[e] = re;
    zi[e] = im;
  }
  __syncthreads();
  // pass 2: X_k = sum_i1 w^(i1 k) Z[i1][k mod n2] for k < n_m, then the modes
  float2* Y = a.y + (size_t)b * a.n_m * a.nlat;
  for (int e = threadIdx.x; e < a.n_m * tl; e += kThreads) {
    const int k = e / tl, jj = e - k * tl, j = j0 + jj;
    int k2 = k % n2;
    const bool cj = k2 >= nh;          // Z[i1][k2] = conj(Z[i1][n2 - k2])
    if (cj) k2 = n2 - k2;
    const float sgn = cj ? -1.0f : 1.0f;
    float re = 0.0f, im = 0.0f;
    int q = 0;   // (i1 * k) mod N
    const int kq = k % N;
    for (int i1 = 0; i1 < n1; ++i1) {
      const int z = (i1 * nh + k2) * tl + jj;
      const float a_r = zr[z], a_i = sgn * zi[z];
      const float t_r = twr[q], t_i = twi[q];
      re += a_r * t_r - a_i * t_i;
      im += a_r * t_i + a_i * t_r;
      q += kq;
      if (q >= N) q -= N;
    }
    if (j < a.nlat) Y[(size_t)k * a.nlat + j] = make_float2(re, -im);
  }
}

// out_b[lon][lat] = epilogue(sum_m of both modes times (cos, sin)(m lon)), twice the
// halves that the Legendre synthesis leaves in Y_b.
__global__ __launch_bounds__(kThreads) void fourier_synthesis_generic(FourierArgs a) {
  extern __shared__ float lds[];
  const int N = a.nlon, n1 = a.n1, n2 = a.n2, tl = a.tl, n_m = a.n_m;
  const int b = blockIdx.y, j0 = blockIdx.x * tl;
  float* twr = lds;
  float* twi = twr + N;
  float* yc = twi + N;             // [n_m][tl]
  float* ys = yc + n_m * tl;       // [n_m - 1][tl]: m >= 1
  float* wr = ys + (n_m - 1) * tl; // [n1][n2][tl]
  float* wi = wr + N * tl;
  const Seg sg = a.seg.s[find_seg(a.seg, b)];
  load_roots(a, twr, twi);
  const float2* Y = a.y + (size_t)b * n_m * a.nlat;
  for (int e = threadIdx.x; e < n_m * tl; e += kThreads) {
    const int k = e / tl, jj = e - k * tl, j = j0 + jj;
    float2 v = make_float2(0.0f, 0.0f);
    if (j < a.nlat) v = Y[(size_t)k * a.nlat + j];
    yc[e] = v.x;
    if (k) ys[e - tl] = v.y;
  }
  __syncthreads();
  // pass 1: W[i1][k2] = sum_{k = k2 + n2 k1 < n_m} c_k conj(w^(i1 k)), c_k = cosine - i sine of Y
  for (int e = threadIdx.x; e < N * tl; e += kThreads) {
    const int r = e / tl, jj = e - r * tl, k2 = r % n2, i1 = r / n2;
    float re = 0.0f, im = 0.0f;
    for (int k = k2; k < a.n_m; k += n2) {
      const float c_r = yc[k * tl + jj], c_i = k ? -ys[(k - 1) * tl + jj] : 0.0f;
      const int q = (int)(((long)i1 * k) % N);
      const float t_r = twr[q], t_i = -twi[q];
      re += c_r * t_r - c_i * t_i;
      im += c_r * t_i + c_i * t_r;
    }
    wr[e] = re;
    wi[e] = im;
  }
  __syncthreads();
  // pass 2: x[i1 + n1 i2] = Re sum_k2 W[i1][k2] conj(w^(n1 i2 k2)), then the epilogue
  float* dst = sg.dst + (size_t)(b - sg.first) * N * a.nlat;
  const float lvl = sg.level ? sg.level[(b - sg.first) % sg.period] : 0.0f;
  for (int e = threadIdx.x; e < N * tl; e += kThreads) {
    // latitude fastest, then i2: the lanes of a wave share i1, so their W reads
    // are broadcasts or distinct banks
    const int r = e / tl, jj = e - r * tl, j = j0 + jj;
    const int i2 = r % n2, i1 = r / n2, lon = i1 + n1 * i2;
    float v = 0.0f;
    int q = 0;   // (i2 * k2) mod n2
    for (int k2 = 0; k2 < n2; ++k2) {
      const int z = (i1 * n2 + k2) * tl + jj;
      v += wr[z] * twr[q * n1] + wi[z] * twi[q * n1];
      q += i2;
      if (q >= n2) q -= n2;
    }
    if (j < a.nlat) {
      if (sg.op & kOpSecLat) v *= a.sec[j];
      v = v * (2.0f * sg.mul);
      if (sg.op & kOpAddLevel) v += lvl;
      if (sg.op & kOpExp) v = expf(v);
      dst[(size_t)lon * a.nlat + j] = v;
    }
  }
}

// The same two passes with both factors known at compile time (the nlon of the
// Grid.T<N> table): each pass is a short FFT in registers (fft, rfft, c2r below: radix
// 2, 3, 4 and 5 steps with literal roots), with the line tile read from and written to
// memory directly; only the pass-1 results and the N roots of unity for the twiddles
// w^(i1 k2) go through LDS.
//
// The real side of each stage uses the Hermitian symmetry in k2: half the analysis's
// pass-1 results are formed and exchanged, and the real FFTs do half the work; on the
// wavenumber side n_m <= nlon / 2 leaves half the inputs zero or outputs unused.  Bound
// by latency: of the launch's single wave of workgroups at T85, of the few workgroups
// that a CU holds at T213.  With dense sums for the short DFTs (n1 and n2 terms per
// output) and Y as the even and odd halves of every mode, T85 analysis (32 fields) and
// synthesis (41) took 8.7 and 12.3 us, now 5.8 and 7.2; T213 x 41 synthesis 115 us, now
// 30.  A thread that took a pair of k2 in the synthesis, to exchange half as much, had
// twice the chain: T85 17.4 us a conversion against 16.2, T213 69 against 56.
constexpr double kPiD = 3.14159265358979323846;
constexpr double ct_sin(double x) {   // |x| <= pi, Taylor series to 1e-16
  double term = x, sum = x;
  for (int n = 1; n < 24; ++n) {
    term *= -x * x / ((2.0 * n) * (2.0 * n + 1.0));
    sum += term;
  }
  return sum;
}
constexpr double ct_cos(double x) {
  double term = 1.0, sum = 1.0;
  for (int n = 1; n < 24; ++n) {
    term *= -x * x / ((2.0 * n - 1.0) * (2.0 * n));
    sum += term;
  }
  return sum;
}
// w_n^q = exp(-2 pi i q / n) = c[q] + i s[q]
template <int n>
struct Roots {
  float c[n], s[n];
  constexpr Roots() : c(), s() {
    for (int q = 0; q < n; ++q) {
      double t = 2.0 * kPiD * q / n;
      if (t > kPiD) t -= 2.0 * kPiD;
      c[q] = (float)ct_cos(t);
      s[q] = (float)-ct_sin(t);
    }
  }
};

// First radix of a length: 4 where it divides, else the smallest of 2, 3, 5.
constexpr int radix(int n) { return n % 4 == 0 ? 4 : n % 2 == 0 ? 2 : n % 3 == 0 ? 3 : n % 5 == 0 ? 5 : n; }

// X_k = sum_j x_j w_n^(jk), in place and in natural order.  The inverse (conjugated
// roots) is the same with real and imaginary parts exchanged: fft(im, re).  HALF: x_j is
// zero (and not read) for j >= n / 2, n of 2 or a multiple of 4 or n = 2 b.
template <int n, bool HALF = false>
__device__ __forceinline__ void fft(float (&re)[n], float (&im)[n]) {
  static_assert(n == 1 || radix(n) < n || n <= 5, "lengths of factors 2, 3 and 5");
  if constexpr (n == 2) {
    const float r = re[1], i = im[1];
    re[1] = re[0] - r; im[1] = im[0] - i;
    re[0] += r; im[0] += i;
  } else if constexpr (n == 3) {
    constexpr float s = 0.866025403784438647f;
    const float tr = re[1] + re[2], ti = im[1] + im[2];
    const float ar = re[0] - 0.5f * tr, ai = im[0] - 0.5f * ti;
    const float br = s * (im[1] - im[2]), bi = s * (re[2] - re[1]);
    re[0] += tr; im[0] += ti;
    re[1] = ar + br; im[1] = ai + bi;
    re[2] = ar - br; im[2] = ai - bi;
  } else if constexpr (n == 4) {
    const float ar = re[0] + re[2], ai = im[0] + im[2], br = re[0] - re[2], bi = im[0] - im[2];
    const float cr = re[1] + re[3], ci = im[1] + im[3], dr = re[1] - re[3], di = im[1] - im[3];
    re[0] = ar + cr; im[0] = ai + ci;
    re[2] = ar - cr; im[2] = ai - ci;
    re[1] = br + di; im[1] = bi - dr;
    re[3] = br - di; im[3] = bi + dr;
  } else if constexpr (n == 5) {
    constexpr float c1 = 0.309016994374947424f, c2 = -0.809016994374947424f;
    constexpr float s1 = 0.951056516295153572f, s2 = 0.587785252292473129f;
    const float ar = re[1] + re[4], ai = im[1] + im[4], br = re[2] + re[3], bi = im[2] + im[3];
    const float cr = re[1] - re[4], ci = im[1] - im[4], dr = re[2] - re[3], di = im[2] - im[3];
    const float er = re[0] + c1 * ar + c2 * br, ei = im[0] + c1 * ai + c2 * bi;
    const float fr = re[0] + c2 * ar + c1 * br, fi = im[0] + c2 * ai + c1 * bi;
    const float gr = s1 * ci + s2 * di, gi = s1 * cr + s2 * dr;
    const float hr = s2 * ci - s1 * di, hi = s2 * cr - s1 * dr;
    re[0] += ar + br; im[0] += ai + bi;
    re[1] = er + gr; im[1] = ei - gi;
    re[4] = er - gr; im[4] = ei + gi;
    re[2] = fr + hr; im[2] = fi - hi;
    re[3] = fr - hr; im[3] = fi + hi;
  } else if constexpr (n > 1) {
    // j = j1 + b j2, k = k1 + a k2: a-point transforms over j2, twiddles, b-point over j1
    constexpr int a = radix(n), b = n / a;
    constexpr Roots<n> w{};
    float tr[a][b], ti[a][b];
#pragma unroll
    for (int j = 0; j < b; ++j) {
      float xr[a], xi[a];
#pragma unroll
      for (int i = 0; i < (HALF ? a / 2 : a); ++i) { xr[i] = re[j + b * i]; xi[i] = im[j + b * i]; }
      if constexpr (!HALF) {
        fft<a>(xr, xi);
      } else if constexpr (a == 2) {
        xr[1] = xr[0]; xi[1] = xi[0];
      } else {
        static_assert(a == 4, "half-zero transforms start with a radix of 2 or 4");
        const float r0 = xr[0], i0 = xi[0], r1 = xr[1], i1 = xi[1];
        xr[0] = r0 + r1; xi[0] = i0 + i1;
        xr[1] = r0 + i1; xi[1] = i0 - r1;
        xr[2] = r0 - r1; xi[2] = i0 - i1;
        xr[3] = r0 - i1; xi[3] = i0 + r1;
      }
#pragma unroll
      for (int k = 0; k < a; ++k) {
        const float c = w.c[(j * k) % n], s = w.s[(j * k) % n];
        tr[k][j] = j * k == 0 ? xr[k] : xr[k] * c - xi[k] * s;
        ti[k][j] = j * k == 0 ? xi[k] : xr[k] * s + xi[k] * c;
      }
    }
#pragma unroll
    for (int k = 0; k < a; ++k) {
      fft<b>(tr[k], ti[k]);
#pragma unroll
      for (int q = 0; q < b; ++q) { re[k + a * q] = tr[k][q]; im[k + a * q] = ti[k][q]; }
    }
  }
}

// X_k for k <= n / 2 of a real x (the others are their conjugates).
template <int n>
__device__ __forceinline__ void rfft(const float (&x)[n], float (&re)[n / 2 + 1], float (&im)[n / 2 + 1]) {
  if constexpr (n == 1) {
    re[0] = x[0]; im[0] = 0.0f;
  } else if constexpr (n == 2) {
    re[0] = x[0] + x[1]; im[0] = 0.0f;
    re[1] = x[0] - x[1]; im[1] = 0.0f;
  } else if constexpr (n == 3) {
    const float t = x[1] + x[2];
    re[0] = x[0] + t; im[0] = 0.0f;
    re[1] = x[0] - 0.5f * t; im[1] = 0.866025403784438647f * (x[2] - x[1]);
  } else if constexpr (n == 5) {
    constexpr float c1 = 0.309016994374947424f, c2 = -0.809016994374947424f;
    constexpr float s1 = 0.951056516295153572f, s2 = 0.587785252292473129f;
    const float a = x[1] + x[4], b = x[2] + x[3], c = x[1] - x[4], d = x[2] - x[3];
    re[0] = x[0] + (a + b); im[0] = 0.0f;
    re[1] = x[0] + c1 * a + c2 * b; im[1] = -(s1 * c + s2 * d);
    re[2] = x[0] + c2 * a + c1 * b; im[2] = -(s2 * c - s1 * d);
  } else if constexpr (n % 4 == 2) {
    // n = 2 b, b odd: j = b j1 + 2 j2 mod n takes no twiddles (Good-Thomas)
    constexpr int b = n / 2;
    float p[b], q[b], pr[b / 2 + 1], pi[b / 2 + 1], qr[b / 2 + 1], qi[b / 2 + 1];
#pragma unroll
    for (int j = 0; j < b; ++j) {
      p[j] = x[2 * j] + x[(2 * j + b) % n];
      q[j] = x[2 * j] - x[(2 * j + b) % n];
    }
    rfft<b>(p, pr, pi);
    rfft<b>(q, qr, qi);
#pragma unroll
    for (int k = 0; k <= b; ++k) {   // X_k = P (even k) or Q (odd k) at k mod b
      const int m = k % b, c = m <= b / 2 ? m : b - m;
      const float sg = m <= b / 2 ? 1.0f : -1.0f;
      re[k] = k % 2 == 0 ? pr[c] : qr[c];
      im[k] = sg * (k % 2 == 0 ? pi[c] : qi[c]);
    }
  } else {
    static_assert(n % 4 == 0, "rfft lengths");
    constexpr int b = n / 4;
    constexpr Roots<n> w{};
    float t0[b], t1r[b], t1i[b], t2r[b], t2i[b];
#pragma unroll
    for (int j = 0; j < b; ++j) {   // four-point transforms of real values: X_0 and X_2 real
      const float p = x[j] + x[j + 2 * b], q = x[j + b] + x[j + 3 * b];
      const float r = x[j] - x[j + 2 * b], s = x[j + 3 * b] - x[j + b];
      const float c1 = w.c[j], s1 = w.s[j], c2 = w.c[(2 * j) % n], s2 = w.s[(2 * j) % n];
      t0[j] = p + q;
      t1r[j] = j == 0 ? r : r * c1 - s * s1;
      t1i[j] = j == 0 ? s : r * s1 + s * c1;
      t2r[j] = j == 0 ? p - q : (p - q) * c2;
      t2i[j] = j == 0 ? 0.0f : (p - q) * s2;
    }
    float zr[b / 2 + 1], zi[b / 2 + 1];
    rfft<b>(t0, zr, zi);
    fft<b>(t1r, t1i);
    fft<b>(t2r, t2i);
#pragma unroll
    for (int q = 0; q < b; ++q) {
      if (q <= b / 2) { re[4 * q] = zr[q]; im[4 * q] = zi[q]; }
      const int k = 1 + 4 * q;   // k or its mirror image n - k
      if (k <= n / 2) { re[k] = t1r[q]; im[k] = t1i[q]; }
      else { re[n - k] = t1r[q]; im[n - k] = -t1i[q]; }
      if (2 + 4 * q <= n / 2) { re[2 + 4 * q] = t2r[q]; im[2 + 4 * q] = t2i[q]; }
    }
  }
}

// x_j = sum over the whole spectrum of X_k conj(w_n^(jk)), real, from X_k for k <= n / 2
// (the imaginary parts of X_0 and X_{n/2} are not read).
template <int n>
__device__ __forceinline__ void c2r(const float (&re)[n / 2 + 1], const float (&im)[n / 2 + 1], float (&x)[n]) {
  if constexpr (n == 1) {
    x[0] = re[0];
  } else if constexpr (n == 2) {
    x[0] = re[0] + re[1];
    x[1] = re[0] - re[1];
  } else if constexpr (n == 3) {
    const float a = re[0] - re[1], b = 1.73205080756887729f * im[1];
    x[0] = re[0] + 2.0f * re[1];
    x[1] = a - b;
    x[2] = a + b;
  } else if constexpr (n == 5) {
    constexpr float c1 = 0.618033988749894848f, c2 = -1.618033988749894848f;   // twice the cosines
    constexpr float s1 = 1.902113032590307144f, s2 = 1.175570504584946258f;
    const float e = re[0] + c1 * re[1] + c2 * re[2], f = re[0] + c2 * re[1] + c1 * re[2];
    const float g = s1 * im[1] + s2 * im[2], h = s2 * im[1] - s1 * im[2];
    x[0] = re[0] + 2.0f * (re[1] + re[2]);
    x[1] = e - g;
    x[4] = e + g;
    x[2] = f - h;
    x[3] = f + h;
  } else if constexpr (n % 4 == 2) {
    constexpr int b = n / 2;
    float p[b], q[b], pr[b / 2 + 1], pi[b / 2 + 1], qr[b / 2 + 1], qi[b / 2 + 1];
#pragma unroll
    for (int k = 0; k <= b; ++k) {
      const int m = k % b, c = m <= b / 2 ? m : b - m;
      const float sg = m <= b / 2 ? 1.0f : -1.0f;
      if (k % 2 == 0) { pr[c] = re[k]; pi[c] = sg * im[k]; }
      else { qr[c] = re[k]; qi[c] = sg * im[k]; }
    }
    c2r<b>(pr, pi, p);
    c2r<b>(qr, qi, q);
#pragma unroll
    for (int j = 0; j < b; ++j) {
      x[2 * j] = p[j] + q[j];
      x[(2 * j + b) % n] = p[j] - q[j];
    }
  } else {
    static_assert(n % 4 == 0, "c2r lengths");
    constexpr int b = n / 4;
    constexpr Roots<n> w{};
    float zr[b / 2 + 1], zi[b / 2 + 1], t0[b], t1r[b], t1i[b], t2r[b], t2i[b];
#pragma unroll
    for (int q = 0; q < b; ++q) {
      if (q <= b / 2) { zr[q] = re[4 * q]; zi[q] = im[4 * q]; }
      const int k = 1 + 4 * q, m = 2 + 4 * q;
      t1r[q] = k <= n / 2 ? re[k] : re[n - k];
      t1i[q] = k <= n / 2 ? im[k] : -im[n - k];
      t2r[q] = m <= n / 2 ? re[m] : re[n - m];
      t2i[q] = m == n / 2 ? 0.0f : m < n / 2 ? im[m] : -im[n - m];
    }
    c2r<b>(zr, zi, t0);
    fft<b>(t1i, t1r);   // inverse
    fft<b>(t2i, t2r);
#pragma unroll
    for (int j = 0; j < b; ++j) {
      const float c1 = w.c[j], s1 = -w.s[j], c2 = w.c[(2 * j) % n], s2 = -w.s[(2 * j) % n];
      const float ar = j == 0 ? t1r[j] : t1r[j] * c1 - t1i[j] * s1;
      const float ai = j == 0 ? t1i[j] : t1r[j] * s1 + t1i[j] * c1;
      const float d = j == 0 ? t2r[j] : t2r[j] * c2 - t2i[j] * s2;   // real: its own mirror image
      const float p = t0[j] + d, q = t0[j] - d;
      x[j] = p + 2.0f * ar;
      x[j + 2 * b] = p - 2.0f * ar;
      x[j + b] = q - 2.0f * ai;
      x[j + 3 * b] = q + 2.0f * ai;
    }
  }
}

// Threads of a compiled Fourier kernel with tl latitudes: one per (i1, latitude) on the
// longitude side and one per (k2, latitude) on the wavenumber side (n1 <= n2).
constexpr int fourier_threads(int n2, int tl) { return (n2 * tl + 63) / 64 * 64; }

// 32-bit byte offset from a uniform base (a field is below 2^31 / 16 bytes).
template <typename T>
__device__ __forceinline__ T* at(T* base, uint32_t bytes) {
  return (T*)((char*)base + bytes);
}

template <int N1, int N2, int TL>
__global__ __launch_bounds__(fourier_threads(N2, TL)) void fourier_analysis_kernel(FourierArgs a) {
  constexpr int N = N1 * N2, NH = N2 / 2 + 1, T = fourier_threads(N2, TL);
  __shared__ float2 tw[N], z[NH * N1 * TL];   // z: [k2][i1][lat]
  const int b = blockIdx.y, j0 = blockIdx.x * TL;
  const Seg sg = a.seg.s[find_seg(a.seg, b)];
  const float* src = sg.src + (size_t)(b - sg.first) * N * a.nlat;
  const float lvl = sg.op & kOpSubLevel ? sg.level[(b - sg.first) % sg.period] : 0.0f;
  const int row = threadIdx.x / TL, jj = threadIdx.x % TL, j = j0 + jj;
  const bool in = j < a.nlat;
  const int jc = in ? j : 0;
  float x[N2];
  if (row < N1) {
#pragma unroll
    for (int i2 = 0; i2 < N2; ++i2) x[i2] = *at(src, ((row + N1 * i2) * a.nlat + jc) * 4u);
  }
  for (int i = threadIdx.x; i < N; i += T) tw[i] = make_float2(a.twr[i], a.twi[i]);
  // pass 1: thread (i1, lat): Z[i1][k2] = sum_i2 x[i1 + N1 i2] w_N2^(i2 k2), k2 <= N2 / 2
  if (row < N1) {
    const float cs = sg.mul * ((sg.op & kOpSecLat) ? a.sec[jc] : 1.0f);
#pragma unroll
    for (int i2 = 0; i2 < N2; ++i2)
      if (sg.op & kOpLog) x[i2] = logf(x[i2]);
#pragma unroll
    for (int i2 = 0; i2 < N2; ++i2) x[i2] = (x[i2] - lvl) * cs;
    float re[NH], im[NH];
    rfft<N2>(x, re, im);
#pragma unroll
    for (int k2 = 0; k2 < NH; ++k2) z[(k2 * N1 + row) * TL + jj] = make_float2(re[k2], im[k2]);
  }
  __syncthreads();
  // pass 2: thread (k2, lat): X_{k2 + N2 k1} = sum_i1 (Z[i1][k2] w^(i1 k2)) w_N1^(i1 k1), with
  // Z[N2 - k2] = conj(Z[k2])
  const int k2 = row, kz = k2 <= N2 / 2 ? k2 : N2 - k2;
  if (k2 >= N2) return;
  const float cj = k2 <= N2 / 2 ? 1.0f : -1.0f;
  float2* Y = a.y + (size_t)b * a.n_m * a.nlat;
  float re[N1], im[N1];
#pragma unroll
  for (int i1 = 0; i1 < N1; ++i1) {
    const float2 v = z[(kz * N1 + i1) * TL + jj], t = tw[i1 * k2];
    const float vi = cj * v.y;
    re[i1] = v.x * t.x - vi * t.y;
    im[i1] = v.x * t.y + vi * t.x;
  }
  fft<N1>(re, im);
#pragma unroll
  for (int k1 = 0; k1 < N1 / 2; ++k1) {   // 2 n_m - 1 <= N: no wavenumber above N / 2
    if (N2 * k1 >= a.n_m) break;          // uniform; k < n_m is masked per lane below
    const int k = k2 + N2 * k1;
    if (in && k < a.n_m) *at(Y, (k * a.nlat + j) * 8u) = make_float2(re[k1], -im[k1]);
  }
}

// Y_k of one latitude (byte offset `at` in the field): zero for k >= n_m, past the
// buffer's end.
__device__ __forceinline__ float2 load_y(__amdgpu_buffer_rsrc_t y, int at) {
  typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
  const uintx2 v = __builtin_amdgcn_raw_buffer_load_b64(y, at, 0, 0);
  return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}

template <int N1, int N2, int TL>
__global__ __launch_bounds__(fourier_threads(N2, TL)) void fourier_synthesis_kernel(FourierArgs a) {
  constexpr int N = N1 * N2, NH = N2 / 2 + 1, T = fourier_threads(N2, TL);
  __shared__ float2 tw[N], w[N * TL];   // w: [i1][k2][lat]
  const int b = blockIdx.y, j0 = blockIdx.x * TL;
  const int row = threadIdx.x / TL, jj = threadIdx.x % TL, j = j0 + jj;
  const bool in = j < a.nlat;
  const __amdgpu_buffer_rsrc_t Y = __builtin_amdgcn_make_buffer_rsrc(
      a.y + (size_t)b * a.n_m * a.nlat, 0, a.n_m * a.nlat * 8, 0x00020000);
  // pass 1: thread (k2, lat): W[i1][k2] = conj(w^(i1 k2)) sum_k1 c_{k2 + N2 k1} conj(w_N1^(i1 k1)),
  // c = cosine - i sine of Y, zero from k1 = N1 / 2 on
  const int k2 = row;
  float re[N1], im[N1];
  if (k2 < N2) {
    int at = (k2 * a.nlat + (in ? j : 0)) * 8;
#pragma unroll
    for (int k1 = 0; k1 < N1 / 2; ++k1) {
      re[k1] = im[k1] = 0.0f;
      if (N2 * k1 >= a.n_m) continue;   // uniform
      const float2 y = load_y(Y, at);
      re[k1] = y.x;
      im[k1] = -y.y;
      at += N2 * a.nlat * 8;
    }
  }
  for (int i = threadIdx.x; i < N; i += T) tw[i] = make_float2(a.twr[i], a.twi[i]);
  __syncthreads();
  if (k2 < N2) {
    if (k2 == 0) im[0] = 0.0f;   // m = 0 has no sine mode
    fft<N1, true>(im, re);       // inverse
#pragma unroll
    for (int i1 = 0; i1 < N1; ++i1) {
      const float2 t = tw[i1 * k2];   // conjugated
      w[(i1 * N2 + k2) * TL + jj] = make_float2(re[i1] * t.x + im[i1] * t.y, im[i1] * t.x - re[i1] * t.y);
    }
  }
  const Seg sg = a.seg.s[find_seg(a.seg, b)];
  __syncthreads();
  // pass 2: thread (i1, lat): the line is the real part of W's transform over k2, that is
  // the transform of its Hermitian part H[k2] = W[k2] + conj(W[N2 - k2]) (the half is in Y):
  // x[i1 + N1 i2] = sum_k2 H[i1][k2] conj(w_N2^(i2 k2)), then the epilogue
  if (row >= N1 || !in) return;
  float* dst = sg.dst + (size_t)(b - sg.first) * N * a.nlat;
  const float lvl = sg.op & kOpAddLevel ? sg.level[(b - sg.first) % sg.period] : 0.0f;
  const float sc = sg.mul * ((sg.op & kOpSecLat) ? a.sec[j] : 1.0f);
  float hr[NH], hi[NH], x[N2];
#pragma unroll
  for (int k2 = 0; k2 < NH; ++k2) {
    const float2 v = w[(row * N2 + k2) * TL + jj], u = w[(row * N2 + (k2 ? N2 - k2 : 0)) * TL + jj];
    hr[k2] = v.x + u.x;
    hi[k2] = v.y - u.y;
  }
  c2r<N2>(hr, hi, x);
#pragma unroll
  for (int i2 = 0; i2 < N2; ++i2) x[i2] = x[i2] * sc + lvl;
  if (sg.op & kOpExp) {
#pragma unroll
    for (int i2 = 0; i2 < N2; ++i2) x[i2] = expf(x[i2]);
  }
#pragma unroll
  for (int i2 = 0; i2 < N2; ++i2) *at(dst, ((row + N1 * i2) * a.nlat + j) * 4u) = x[i2];
}

// ------------------------------------------------------------------ host side
double legendre_p(int n, double x, double* dp) {
  double p0 = 1.0, p1 = x;
  for (int k = 2; k <= n; ++k) {
    const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
    p0 = p1;
    p1 = p2;
  }
  if (n == 0) {
    *dp = 0.0;
    return 1.0;
  }
  *dp = n * (x * p1 - p0) / (x * x - 1.0);
  return p1;
}

void gauss_nodes(int n, double* x, double* w) {
  for (int i = 0; i < n; ++i) {
    // i-th root from the north (cos guess), stored south to north
    double z = std::cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 0.0;
    for (int it = 0; it < 100; ++it) {
      const double p = legendre_p(n, z, &dp);
      const double dz = p / dp;
      z -= dz;
      if (std::fabs(dz) < 1e-16) break;
    }
    legendre_p(n, z, &dp);
    x[n - 1 - i] = z;
    w[n - 1 - i] = 2.0 / ((1.0 - z * z) * dp * dp);
  }
}

int check_grid(int32_t n_m, int32_t n_l, int32_t nlon, int32_t nlat) {
  if (n_m < 1 || n_l < 2 || nlon < 1 || nlat < 2 || (nlat & 1) || n_m > n_l || 2 * n_m - 1 > nlon || n_l > nlat ||
      (int64_t)n_m * nlat * n_l >= ((int64_t)1 << 31) || (int64_t)nlon * nlat * 64 >= ((int64_t)1 << 31))
    return fail(SPEEDY_ERR_ARG, "speedy_sht: bad grid (need 1 <= n_m <= n_l <= nlat, n_l >= 2, 2*n_m-1 <= nlon, "
                                "nlat even)");
  return SPEEDY_OK;
}

// The normalized P_l^m(x_j), l = 0 .. n_l - 1, of latitudes j < count: each(j, m, column).
template <typename F>
void legendre_columns(int32_t n_m, int32_t n_l, int32_t count, const double* x, F each) {
  std::vector<double> col(n_l);
  for (int j = 0; j < count; ++j) {
    const double xj = x[j], yj = std::sqrt(1.0 - xj * xj);
    double diag = 1.0 / std::sqrt(2.0);
    for (int m = 0; m < n_m; ++m) {
      if (m > 0) diag = -std::sqrt(1.0 + 1.0 / (2.0 * m)) * yj * diag;
      std::fill(col.begin(), col.end(), 0.0);
      col[m] = diag;
      if (m + 1 < n_l) col[m + 1] = std::sqrt(2.0 * m + 3.0) * xj * diag;
      for (int l = m + 2; l < n_l; ++l) {
        const double a = std::sqrt((4.0 * l * l - 1.0) / ((double)l * l - (double)m * m));
        const double b = std::sqrt(((l - 1.0) * (l - 1.0) - (double)m * m) / (4.0 * (l - 1.0) * (l - 1.0) - 1.0));
        col[l] = a * (xj * col[l - 1] - b * col[l - 2]);
      }
      each(j, m, col.data());
    }
  }
}

void fill_basis(int32_t n_m, int32_t n_l, int32_t nlon, int32_t nlat, const double* x, float* fourier,
                float* legendre) {
  const int mm = 2 * n_m - 1;
  if (fourier) {
    for (int i = 0; i < nlon; ++i) {
      const double lon = 2.0 * M_PI * i / nlon;
      fourier[(size_t)i * mm] = (float)(1.0 / std::sqrt(2.0 * M_PI));
      for (int m = 1; m < n_m; ++m) {
        fourier[(size_t)i * mm + 2 * m - 1] = (float)(std::cos(m * lon) / std::sqrt(M_PI));
        fourier[(size_t)i * mm + 2 * m] = (float)(std::sin(m * lon) / std::sqrt(M_PI));
      }
    }
  }
  if (legendre) {
    legendre_columns(n_m, n_l, nlat, x, [&](int j, int m, const double* col) {
      float* dst = legendre + ((size_t)m * nlat + j) * n_l;
      for (int l = 0; l < n_l; ++l) dst[l] = (float)col[l];
    });
  }
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

size_t y_bytes(const SpeedyShtPlan* p, int32_t nfield) {
  return align256((size_t)nfield * p->n_m * p->nlat * sizeof(float2));
}

// LDS of the Legendre kernels: two parities of 16 staged rows, and the analysis's 16
// modal rows where both fit kLegendreLds (two workgroups a CU; T425 takes 69 KiB).
constexpr size_t kLegendreLds = 80 * 1024;
constexpr int kMaxTiles = 30;   // staged at a time: 62 KiB
size_t staged_lds(int kt) { return 2 * 16 * (size_t)lds_row(kt) * sizeof(float); }
int tiles16(int n) { return (n + 15) / 16; }
int analysis_kt(const SpeedyShtPlan* p) { return std::min(tiles16(p->nlat / 2), kMaxTiles); }
int synthesis_kt(const SpeedyShtPlan* p) { return std::min(tiles16((p->n_l + 1) / 2), kMaxTiles); }
size_t z_lds(const SpeedyShtPlan* p) { return 16 * (size_t)p->n_l * sizeof(float); }
bool z_in_lds(const SpeedyShtPlan* p) { return staged_lds(analysis_kt(p)) + z_lds(p) <= kLegendreLds; }

// The Y of a call; where the analysis's modal rows do not fit in LDS, also those of
// every workgroup: with its zero rows a call has at most 5 / 4 nfield fields, in chunks
// of four levels or eight fields.
size_t ws_bytes(const SpeedyShtPlan* p, int32_t nfield) {
  const size_t z = z_in_lds(p) ? 0 : (((size_t)nfield + nfield / 4) / 8 + 2) * p->n_m * z_lds(p);
  return y_bytes(p, nfield) + align256(z);
}

LegendreArgs legendre_args(const SpeedyShtPlan* p, int32_t nfield, void* ws) {
  LegendreArgs a{};
  a.n_m = p->n_m; a.nl = p->n_l; a.nlat = p->nlat; a.nfield = nfield;
  a.blk = p->blk;
  a.y = static_cast<float2*>(ws);
  a.z = reinterpret_cast<float*>(static_cast<char*>(ws) + y_bytes(p, nfield));
  a.inv_radius = (float)(1.0 / p->radius);
  a.radius2 = (float)(p->radius * p->radius);
  return a;
}

FourierArgs fourier_args(const SpeedyShtPlan* p, int32_t nfield, int32_t tl, const SegTable& seg) {
  FourierArgs f{};
  f.nlon = p->nlon; f.nlat = p->nlat; f.mm = p->mm; f.n_m = p->n_m; f.n1 = p->n1; f.n2 = p->n2; f.tl = tl;
  f.nfield = nfield;
  f.twr = p->tw; f.twi = p->tw + p->nlon; f.sec = p->sec;
  f.seg = seg;
  return f;
}

// The Fourier kernels of one factor pair nlon = n1 * n2, compiled for the nlon of the
// Grid.T<N> table, each with the latitudes a workgroup takes in the analysis and the
// synthesis: 16 (64-byte rows), or 8 where a CU would hold too few (T213 conversions 56.3
// us with 8 in the synthesis, 57.6 with 16; tendencies 41.2 with 16 in the analysis, 44.4
// with 8; T425 272 and 229 us with 8, 302 and 261 with 4).  Other nlon take the generic
// LDS kernels.
typedef void (*FourierKernel)(FourierArgs);
struct FourierPair {
  int n1, n2, tl_a, tl_s;
  FourierKernel analysis, synthesis;
};
#define SHT_PAIR(a, b, ta, ts) {a, b, ta, ts, fourier_analysis_kernel<a, b, ta>, fourier_synthesis_kernel<a, b, ts>}
const FourierPair kPairs[] = {SHT_PAIR(8, 8, 16, 16),   SHT_PAIR(8, 12, 16, 16),  SHT_PAIR(8, 16, 16, 16),
                              SHT_PAIR(16, 16, 16, 16), SHT_PAIR(16, 20, 16, 16), SHT_PAIR(18, 20, 16, 16),
                              SHT_PAIR(16, 32, 16, 16), SHT_PAIR(20, 32, 16, 8),  SHT_PAIR(32, 32, 8, 8),
                              SHT_PAIR(32, 40, 8, 8)};
#undef SHT_PAIR

const FourierPair* find_pair(int n1, int n2) {
  for (const FourierPair& f : kPairs)
    if (f.n1 == n1 && f.n2 == n2) return &f;
  return nullptr;
}

// LDS bytes of the generic Fourier kernels (roots, line tile, pass-1 result)
constexpr size_t kFourierLds = 64 * 1024;
size_t analysis_lds(int N, int n1, int n2, int tl) {
  return 4 * (2 * (size_t)N + 2 * (size_t)n1 * (n2 / 2 + 1) * tl + (size_t)N * tl);
}
size_t synthesis_lds(int N, int mm, int tl) { return 4 * (2 * (size_t)N + 2 * (size_t)N * tl + (size_t)mm * tl); }

hipError_t run_fourier(const SpeedyShtPlan* p, int32_t nfield, const SegTable& seg, float2* y, bool analysis,
                       hipStream_t s) {
  const int tl = analysis ? p->tl_a : p->tl_s;
  FourierArgs f = fourier_args(p, nfield, tl, seg);
  f.y = y;
  const dim3 grid((p->nlat + tl - 1) / tl, nfield);
  if (const FourierPair* fp = find_pair(p->n1, p->n2))
    hipLaunchKernelGGL(analysis ? fp->analysis : fp->synthesis, grid, dim3(fourier_threads(fp->n2, tl)),
                       0, s, f);
  else
    hipLaunchKernelGGL(analysis ? fourier_analysis_generic : fourier_synthesis_generic, grid, dim3(kThreads),
                       analysis ? analysis_lds(p->nlon, p->n1, p->n2, tl) : synthesis_lds(p->nlon, p->mm, tl), s, f);
  return hipGetLastError();
}

dim3 legendre_grid(const LegendreArgs& a) { return dim3((a.n_m + 7) / 8 * 8 * chunks(a.winds, a.plain, a.geo)); }

hipError_t run_analysis(const SpeedyShtPlan* p, int32_t nfield, const SegTable& seg, LegendreArgs a, hipStream_t s) {
  const hipError_t e = run_fourier(p, nfield, seg, a.y, true, s);
  if (e != hipSuccess) return e;
  a.P = p->Pa;
  a.kt = analysis_kt(p);
  const bool zlds = z_in_lds(p);
  hipLaunchKernelGGL(zlds ? legendre_analysis_kernel<true> : legendre_analysis_kernel<false>, legendre_grid(a),
                     dim3(kThreads), staged_lds(a.kt) + (zlds ? z_lds(p) : 0), s, a);
  return hipGetLastError();
}

hipError_t run_synthesis(const SpeedyShtPlan* p, int32_t nfield, const SegTable& seg, LegendreArgs a, hipStream_t s) {
  a.P = p->Ps;
  a.kt = synthesis_kt(p);
  hipLaunchKernelGGL(legendre_synthesis_kernel, legendre_grid(a), dim3(kThreads), staged_lds(a.kt), s, a);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess ? e : run_fourier(p, nfield, seg, a.y, false, s);
}

void add_seg(SegTable& t, const float* src, float* dst, int32_t count, int32_t op, float mul,
             const float* level = nullptr, int32_t period = 1) {
  Seg& s = t.s[t.n];
  s.src = src; s.dst = dst; s.level = level; s.period = period; s.op = op; s.mul = mul; s.count = count;
  s.first = t.n == 0 ? 0 : t.s[t.n - 1].first + t.s[t.n - 1].count;
  ++t.n;
}

int check_call(const SpeedyShtPlan* p, int32_t nfield, void* ws, size_t wsb) {
  if (!p) return fail(SPEEDY_ERR_ARG, "speedy_sht: null plan");
  if (nfield < 1 || nfield > 65535) return fail(SPEEDY_ERR_ARG, "speedy_sht: nfield must be in 1..65535");
  if (!ws || wsb < ws_bytes(p, nfield))
    return fail(SPEEDY_ERR_WORKSPACE, "speedy_sht: workspace missing or smaller than speedy_sht_workspace_bytes");
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev != p->device)
    return fail(SPEEDY_ERR_ARG, "speedy_sht: the plan belongs to another device than the current one");
  return SPEEDY_OK;
}

int check_spec(const SpeedyDynamicsSpec* sp) {
  if (!sp || sp->kx < 1 || sp->kx > SPEEDY_SHT_KX_MAX || !sp->reference_temperature)
    return fail(SPEEDY_ERR_ARG, "speedy_sht: bad dynamics spec (kx 1..16, reference temperature)");
  return SPEEDY_OK;
}

int hip_result(hipError_t e) {
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_sht: launch failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

}  // namespace sht

using namespace sht;

extern "C" {

int speedy_sht_host_basis(int32_t n_m, int32_t n_l, int32_t nlon, int32_t nlat, double* sin_lat, double* weights,
                          float* fourier, float* legendre) {
  if (int rc = check_grid(n_m, n_l, nlon, nlat)) return rc;
  if (!sin_lat || !weights) return fail(SPEEDY_ERR_ARG, "speedy_sht_host_basis: null nodes or weights");
  gauss_nodes(nlat, sin_lat, weights);
  fill_basis(n_m, n_l, nlon, nlat, sin_lat, fourier, legendre);
  return SPEEDY_OK;
}

int speedy_sht_create(int32_t n_m, int32_t n_l, int32_t nlon, int32_t nlat, double radius, SpeedyShtPlan** out) {
  if (!out) return fail(SPEEDY_ERR_ARG, "speedy_sht_create: null output");
  *out = nullptr;
  if (int rc = check_grid(n_m, n_l, nlon, nlat)) return rc;
  if (!(radius > 0.0)) return fail(SPEEDY_ERR_ARG, "speedy_sht_create: radius must be positive");
  const int mm = 2 * n_m - 1;
  // nlon = n1 * n2 with n1 the largest divisor <= sqrt(nlon); the latitude tile of the
  // compiled pair, or for the generic kernels the widest (16, 15, .., 1) whose LDS fits
  int n1 = 1;
  for (int d = 1; (int64_t)d * d <= nlon; ++d)
    if (nlon % d == 0) n1 = d;
  const int n2 = nlon / n1;
  const FourierPair* fp = find_pair(n1, n2);
  int tl_a = fp ? fp->tl_a : 16, tl_s = fp ? fp->tl_s : 16;
  if (!fp) {
    while (tl_a > 1 && analysis_lds(nlon, n1, n2, tl_a) > kFourierLds) --tl_a;
    while (tl_s > 1 && synthesis_lds(nlon, mm, tl_s) > kFourierLds) --tl_s;
    if (analysis_lds(nlon, n1, n2, tl_a) > kFourierLds || synthesis_lds(nlon, mm, tl_s) > kFourierLds)
      return fail(SPEEDY_ERR_ARG, "speedy_sht_create: nlon too large for the Fourier stages' 64 KiB of LDS");
  }
  std::vector<double> x(nlat), w(nlat);
  gauss_nodes(nlat, x.data(), w.data());
  // operand blocks of the Legendre stages
  const int h = nlat / 2, jts = tiles16(h);
  std::vector<int32_t> blk(n_m);
  int64_t nblk = 0;
  for (int m = 0; m < n_m; ++m) {
    blk[m] = (int32_t)nblk;
    nblk += (int64_t)2 * tiles16((n_l - m + 1) / 2) * jts;
  }
  std::vector<float> Ps((size_t)nblk * 256, 0.0f), Pa((size_t)nblk * 256, 0.0f), sec(nlat), tw(2 * (size_t)nlon);
  legendre_columns(n_m, n_l, h, x.data(), [&](int j, int m, const double* col) {
    const double f = 1.0 / std::sqrt(m == 0 ? 2.0 * M_PI : M_PI), wj = w[j] * 2.0 * M_PI / nlon;
    const int cts = tiles16((n_l - m + 1) / 2);
    for (int l = m; l < n_l; ++l) {
      const int par = (l - m) & 1, c = (l - m) >> 1, ci = c & 15, ji = j & 15;
      const size_t at = ((size_t)blk[m] + (size_t)(par * cts + c / 16) * jts + j / 16) * 256;
      Ps[at + ((ci & 3) * 16 + ji) * 4 + (ci >> 2)] = (float)col[l];
      Pa[at + ((ji >> 2) * 16 + ci) * 4 + (ji & 3)] = (float)(f * wj * col[l]);
    }
  });
  for (int j = 0; j < nlat; ++j) sec[j] = (float)(1.0 / std::sqrt(1.0 - x[j] * x[j]));
  for (int j = 0; j < nlon; ++j) {
    tw[j] = (float)std::cos(2.0 * M_PI * j / nlon);
    tw[nlon + j] = (float)-std::sin(2.0 * M_PI * j / nlon);
  }
  SpeedyShtPlan* p = new SpeedyShtPlan{n_m, n_l, nlon, nlat, mm, radius, 0, n1, n2, tl_a, tl_s,
                                       nullptr, nullptr, nullptr, nullptr, nullptr};
  hipError_t e = hipGetDevice(&p->device);
  auto up = [&](auto** dst, const auto& v) {
    if (e != hipSuccess) return;
    e = hipMalloc(reinterpret_cast<void**>(dst), v.size() * sizeof(v[0]));
    if (e == hipSuccess) e = hipMemcpy(*dst, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice);
  };
  up(&p->Ps, Ps);
  up(&p->Pa, Pa);
  up(&p->blk, blk);
  up(&p->sec, sec);
  up(&p->tw, tw);
  if (e != hipSuccess) {
    speedy_sht_destroy(p);
    return fail(SPEEDY_ERR_HIP, std::string("speedy_sht_create: ") + hipGetErrorString(e));
  }
  *out = p;
  return SPEEDY_OK;
}

int speedy_sht_destroy(SpeedyShtPlan* p) {
  if (!p) return SPEEDY_OK;
  for (float* q : {p->Ps, p->Pa, p->sec, p->tw})
    if (q) (void)hipFree(q);
  if (p->blk) (void)hipFree(p->blk);
  delete p;
  return SPEEDY_OK;
}

size_t speedy_sht_workspace_bytes(const SpeedyShtPlan* p, int32_t nfield) {
  return p && nfield > 0 ? ws_bytes(p, nfield) : 0;
}

int speedy_sht_to_modal(const SpeedyShtPlan* p, const float* nodal, float* modal, int32_t nfield, void* ws,
                        size_t wsb, void* stream) {
  if (int rc = check_call(p, nfield, ws, wsb)) return rc;
  if (!nodal || !modal) return fail(SPEEDY_ERR_ARG, "speedy_sht_to_modal: null field");
  SegTable seg{};
  add_seg(seg, nodal, nullptr, nfield, 0, 1.0f);
  LegendreArgs a = legendre_args(p, nfield, ws);
  a.plain = a.count[0] = nfield;
  a.dst[0] = modal;
  return hip_result(run_analysis(p, nfield, seg, a, static_cast<hipStream_t>(stream)));
}

int speedy_sht_to_nodal(const SpeedyShtPlan* p, const float* modal, float* nodal, int32_t nfield, void* ws,
                        size_t wsb, void* stream) {
  if (int rc = check_call(p, nfield, ws, wsb)) return rc;
  if (!nodal || !modal) return fail(SPEEDY_ERR_ARG, "speedy_sht_to_nodal: null field");
  SegTable seg{};
  add_seg(seg, nullptr, nodal, nfield, 0, 1.0f);
  LegendreArgs a = legendre_args(p, nfield, ws);
  a.plain = a.count[0] = nfield;
  a.src[0] = modal;
  return hip_result(run_synthesis(p, nfield, seg, a, static_cast<hipStream_t>(stream)));
}

int speedy_dynamics_to_physics(const SpeedyShtPlan* p, const SpeedyDynamicsSpec* spec, const SpeedySpectralState* in,
                               const SpeedyNodalState* out, void* ws, size_t wsb, void* stream) {
  if (int rc = check_spec(spec)) return rc;
  if (!in || !out || !in->vorticity || !in->divergence || !in->temperature_variation || !in->specific_humidity ||
      !in->log_surface_pressure || !spec->orography || !spec->sigma_boundaries || !out->u_wind || !out->v_wind ||
      !out->temperature || !out->specific_humidity || !out->geopotential || !out->normalized_surface_pressure)
    return fail(SPEEDY_ERR_ARG, "speedy_dynamics_to_physics: null field");
  const int kx = spec->kx, nsp = in->nsp;
  if (nsp < 1 || nsp > kx || out->nsp != nsp)
    return fail(SPEEDY_ERR_ARG, "speedy_dynamics_to_physics: nsp must be in 1..kx and equal on both sides");
  const int nfield = 5 * kx + nsp;
  if (int rc = check_call(p, nfield, ws, wsb)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // 1. modal (u cos, v cos), the other modal inputs and the modal geopotential:
  //    fields [u kx][v kx][T_var kx][q kx][log ps nsp][phi kx]
  LegendreArgs m = legendre_args(p, nfield, ws);
  m.kx = m.winds = m.geo = kx;
  m.plain = 2 * kx + nsp;
  m.vor = in->vorticity; m.div = in->divergence;
  m.src[0] = in->temperature_variation; m.count[0] = kx;
  m.src[1] = in->specific_humidity; m.count[1] = kx;
  m.src[2] = in->log_surface_pressure; m.count[2] = nsp;
  m.tvar = in->temperature_variation;
  m.orography = spec->orography;
  m.reference = spec->reference_temperature;
  m.gravity = (float)spec->gravity;
  // hydrostatic trapezoid on log(sigma): alpha_k = (ln s_k+1 - ln s_k)/2,
  // alpha_K-1 = -ln s_K-1; W[j][j] = alpha_j, W[j][k>j] = alpha_k + alpha_k-1
  std::vector<double> ls(kx), alpha(kx);
  for (int k = 0; k < kx; ++k) ls[k] = std::log(0.5 * (spec->sigma_boundaries[k] + spec->sigma_boundaries[k + 1]));
  for (int k = 0; k + 1 < kx; ++k) alpha[k] = 0.5 * (ls[k + 1] - ls[k]);
  alpha[kx - 1] = -ls[kx - 1];
  for (int j = 0; j < kx; ++j)
    for (int k = 0; k < kx; ++k)
      m.geo_w[j][k] = (float)(spec->gas_constant * (k < j ? 0.0 : k == j ? alpha[j] : alpha[k] + alpha[k - 1]));
  // 2. synthesis with the nodal post-operations
  SegTable seg{};
  add_seg(seg, nullptr, out->u_wind, kx, kOpSecLat, 1.0f);
  add_seg(seg, nullptr, out->v_wind, kx, kOpSecLat, 1.0f);
  add_seg(seg, nullptr, out->temperature, kx, kOpAddLevel, 1.0f, spec->reference_temperature, kx);
  add_seg(seg, nullptr, out->specific_humidity, kx, 0, 1000.0f);
  add_seg(seg, nullptr, out->normalized_surface_pressure, nsp, kOpExp, 1.0f);
  add_seg(seg, nullptr, out->geopotential, kx, 0, 1.0f);
  return hip_result(run_synthesis(p, nfield, seg, m, s));
}

namespace {
int nodal_to_spectral(const SpeedyShtPlan* p, const SpeedyDynamicsSpec* spec, const SpeedyNodalState* in,
                      const SpeedySpectralState* out, void* ws, size_t wsb, void* stream, bool tendency) {
  const char* who = tendency ? "speedy_physics_tendency_to_dynamics" : "speedy_physics_to_dynamics";
  if (int rc = check_spec(spec)) return rc;
  if (!in || !out || !in->u_wind || !in->v_wind || !in->temperature || !in->specific_humidity ||
      (!tendency && !in->normalized_surface_pressure) || !out->vorticity || !out->divergence ||
      !out->temperature_variation || !out->specific_humidity || !out->log_surface_pressure)
    return fail(SPEEDY_ERR_ARG, std::string(who) + ": null field");
  const int kx = spec->kx, nsp = out->nsp;
  if (nsp < 1 || nsp > kx || (!tendency && in->nsp != nsp))
    return fail(SPEEDY_ERR_ARG, std::string(who) + ": nsp must be in 1..kx and equal on both sides");
  const int nsp_in = tendency ? 0 : nsp;
  const int nfield = 4 * kx + nsp_in;
  if (int rc = check_call(p, nfield, ws, wsb)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SegTable seg{};
  add_seg(seg, in->u_wind, nullptr, kx, kOpSecLat, 1.0f);
  add_seg(seg, in->v_wind, nullptr, kx, kOpSecLat, 1.0f);
  if (tendency)
    add_seg(seg, in->temperature, nullptr, kx, 0, 1.0f);
  else
    add_seg(seg, in->temperature, nullptr, kx, kOpSubLevel, 1.0f, spec->reference_temperature, kx);
  add_seg(seg, in->specific_humidity, nullptr, kx, 0, 1e-3f);
  if (!tendency) add_seg(seg, in->normalized_surface_pressure, nullptr, nsp, kOpLog, 1.0f);
  LegendreArgs m = legendre_args(p, nfield, ws);
  m.kx = m.winds = kx;
  m.plain = 2 * kx + nsp;
  m.vor_out = out->vorticity; m.div_out = out->divergence;
  m.dst[0] = out->temperature_variation; m.count[0] = kx;
  m.dst[1] = out->specific_humidity; m.count[1] = kx;
  m.dst[2] = out->log_surface_pressure; m.count[2] = nsp;   // zeros for a tendency
  return hip_result(run_analysis(p, nfield, seg, m, s));
}
}  // namespace

int speedy_physics_to_dynamics(const SpeedyShtPlan* p, const SpeedyDynamicsSpec* spec, const SpeedyNodalState* in,
                               const SpeedySpectralState* out, void* ws, size_t wsb, void* stream) {
  return nodal_to_spectral(p, spec, in, out, ws, wsb, stream, false);
}

int speedy_physics_tendency_to_dynamics(const SpeedyShtPlan* p, const SpeedyDynamicsSpec* spec,
                                        const SpeedyNodalState* in, const SpeedySpectralState* out, void* ws,
                                        size_t wsb, void* stream) {
  return nodal_to_spectral(p, spec, in, out, ws, wsb, stream, true);
}

const char* speedy_sht_last_error(void) { return g_err.c_str(); }

}  // extern "C"
